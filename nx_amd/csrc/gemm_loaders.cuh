// The loaders of the contraction kernels: where each lane's 16-byte pieces of a slab lie, in the operand and in LDS.  Everything here
// is addresses; what reads and moves the bytes (load_piece, lds_dma16, lds_dma16_at) and makes a pointer scalar (wave_uniform) is defined by
// whoever includes it: gemm_mfma.cuh, or a host program that walks every lane over ragged sizes and sees what is read (tests/test_dot_loads.py).
#pragma once
#include <cstdint>

#include "gemm_choice.h"

namespace hipnx {

// Swizzle of the [row][k] LDS layout: 16-byte chunk index XOR a 3-bit function of the row.  Its
// part in the low four row bits (bit0 = r0^r2, bit1 = r1^r2, bit2 = r2^r3) is one of the maps a
// sweep over all linear maps of those bits measured as conflict-free for the fragment read
// (16 consecutive rows x 4 chunks per ds_read_b128: 4 clocks per instruction instead of 8); row
// bits 4..6 are constant within a fragment and are mixed in for the transposed writes of the
// register-staged operands, whose lanes hold rows 4, 8 or 16 apart.
__device__ __forceinline__ int lds_slot(int row, int chunk) {
  const int low = ((row ^ (row >> 2)) & 1) | ((((row >> 1) ^ (row >> 2)) & 1) << 1) | ((((row >> 2) ^ (row >> 3)) & 1) << 2);
  return chunk ^ low ^ ((row >> 4) & 7);
}

// The last `rem` (1 .. 15) of the 16 bytes that end at `end`, moved to the front, zeros behind them: the end of a row that is not
// whole pieces.  One load that lies inside the row, whatever is behind it (the row has sixteen bytes, the host sees to it).
__device__ __forceinline__ v4i row_end_piece(const unsigned char *end, int rem) {
  typedef unsigned long long v2ul __attribute__((ext_vector_type(2)));
  const v2ul w = __builtin_bit_cast(v2ul, load_piece(end - 16));
  const int shift = (16 - rem) * 8;
  v2ul out;
  if (shift >= 64) {
    out[0] = w[1] >> (shift - 64);
    out[1] = 0;
  } else {
    out[0] = (w[0] >> shift) | (w[1] << (64 - shift));
    out[1] = w[1] >> shift;
  }
  return __builtin_bit_cast(v4i, out);
}

// K-inner slab loader: ROWS x 128 B, direct to LDS.  The per-lane source pointers (row clamp,
// row * stride, swizzled chunk) are computed once; per slab only the K offset moves.
// Rows past `rows_valid` are clamped (loaded from the last valid row; their results are never
// stored).
template <int ROWS, int NWAVES>
struct KInnerLoader {
  static constexpr int INSTR = ROWS / 8;  // wave instructions per slab (1 KiB of LDS each)
  static constexpr int PER = INSTR / NWAVES;
  static_assert(INSTR % NWAVES == 0, "slab rows must split evenly over the waves");
  const unsigned char *src[PER];
  int lds_off[PER];

  __device__ __forceinline__ void init(const unsigned char *__restrict__ g, int64_t ld, int64_t row0, int64_t rows_valid,
                                       int wave, int lane) {
#pragma unroll
    for (int i = 0; i < PER; i++) {
      const int t = wave + NWAVES * i;
      const int r = t * 8 + (lane >> 3);
      const int chunk = lds_slot(r, lane & 7);  // the XOR map is an involution: slot -> chunk
      int64_t gr = row0 + r;
      gr = gr < rows_valid ? gr : rows_valid - 1;
      src[i] = g + gr * ld + chunk * 16;
      lds_off[i] = t * 1024;
    }
  }
  __device__ __forceinline__ void issue(int64_t kbyte0, unsigned char *lds) const {
#pragma unroll
    for (int i = 0; i < PER; i++)
      lds_dma16(src[i] + kbyte0, lds + lds_off[i]);
  }
  // a slab of which only the first `valid` bytes of each row exist; a row's last piece, where it is not whole, is zero until
  // finish_partial writes it, behind the wave's wait for these requests
  __device__ __forceinline__ void issue_partial(int64_t kbyte0, int valid, unsigned char *lds, int wave, int lane) const {
#pragma unroll
    for (int i = 0; i < PER; i++) {
      const int r = (wave + NWAVES * i) * 8 + (lane >> 3);
      lds_dma16(lds_slot(r, lane & 7) * 16 + 16 <= valid ? src[i] + kbyte0 : (const unsigned char *)g_zero16, lds + lds_off[i]);
    }
  }
  __device__ __forceinline__ void finish_partial(int64_t kbyte0, int valid, unsigned char *lds, int wave, int lane) const {
    if ((valid & 15) == 0) return;
    v4i v[PER];
#pragma unroll
    for (int i = 0; i < PER; i++)
      if (lds_slot((wave + NWAVES * i) * 8 + (lane >> 3), lane & 7) == valid >> 4) v[i] = row_end_piece(src[i] + kbyte0 + (valid & 15), valid & 15);
#pragma unroll
    for (int i = 0; i < PER; i++)
      if (lds_slot((wave + NWAVES * i) * 8 + (lane >> 3), lane & 7) == valid >> 4) *reinterpret_cast<v4i *>(lds + lds_off[i] + lane * 16) = v[i];
  }
  // instruction i of the slab goes out at step i * spread / PER + phase (+ skew, which may be a
  // run-time value); with t, spread and phase known after unrolling the tests fold away
  __device__ __forceinline__ void issue_at(int t, int spread, int phase, int skew, int64_t kbyte0, unsigned char *lds) const {
#pragma unroll
    for (int i = 0; i < PER; i++)
      if (t == i * spread / PER + phase + skew) lds_dma16(src[i] + kbyte0, lds + lds_off[i]);
  }
};

// ---- K-outer operands: g is [K, rows] (rows contiguous).  A lane loads a small block of
// 16-byte row runs at consecutive k, transposes it in registers and writes K-runs into the same
// [row][k] LDS layout the K-inner loader produces.  Block shape per element size ES:
//   ES = 2:  8 k x  8 rows -> eight 16-byte K-runs (v_perm_b32 pairs halves)
//   ES = 4:  4 k x  4 rows -> four 16-byte K-runs (pure register renaming)
//   ES = 1:  4 k x 16 rows -> sixteen 4-byte K-runs (4 x 4 byte transposes with v_perm_b32)
// A k-row that is not whole pieces (rows_valid no multiple of RB): its last piece runs into the next k-row, which only rows of
// the tile past the edge see; the very last k-row has nothing behind it, so its piece is read so as to end with the row
// (fetch_partial: the host makes the last slab a partial one).  Of a partial slab the k past the end of K are zero.
template <int ES> struct KOuterShape;
template <> struct KOuterShape<2> { static constexpr int KB = 8, RB = 8; };
template <> struct KOuterShape<4> { static constexpr int KB = 4, RB = 4; };
template <> struct KOuterShape<1> { static constexpr int KB = 4, RB = 16; };
template <> struct KOuterShape<8> { static constexpr int KB = 2, RB = 2; };

template <int ES, int ROWS, int NTHREADS>
struct KOuterStage {
  static constexpr int KB = KOuterShape<ES>::KB, RB = KOuterShape<ES>::RB;
  static constexpr int KSLAB = SLAB / ES;                       // k values per slab
  static constexpr int BLOCKS = (ROWS / RB) * (KSLAB / KB);
  static constexpr int PER = (BLOCKS + NTHREADS - 1) / NTHREADS;
  static constexpr int LOADS = PER * KB;                        // vector-memory ops per slab per lane
  v4i v[PER][KB];

  __device__ __forceinline__ void fetch(const unsigned char *__restrict__ g, int64_t ld, int64_t row0, int64_t rows_valid,
                                        int64_t k0, int tid) {
#pragma unroll
    for (int p = 0; p < PER; p++) {
      const int blk = tid + p * NTHREADS;
      if (blk >= BLOCKS) break;
      const int rb = blk % (ROWS / RB), kb = blk / (ROWS / RB);
      int64_t col = row0 + rb * RB;
      col = col < rows_valid ? col : (rows_valid - 1) / RB * RB;  // tile rows past the edge: any piece
#pragma unroll
      for (int j = 0; j < KB; j++)
        v[p][j] = load_piece(g + (k0 + kb * KB + j) * ld + col * ES);
    }
  }

  // a slab of which only the first `valid` k exist
  __device__ __forceinline__ void fetch_partial(const unsigned char *__restrict__ g, int64_t ld, int64_t row0, int64_t rows_valid,
                                                int64_t k0, int valid, int tid) {
#pragma unroll
    for (int p = 0; p < PER; p++) {
      const int blk = tid + p * NTHREADS;
      if (blk >= BLOCKS) break;
      const int rb = blk % (ROWS / RB), kb = blk / (ROWS / RB);
      int64_t col = row0 + rb * RB;
      col = col < rows_valid ? col : (rows_valid - 1) / RB * RB;
      const bool runs_over = col + RB > rows_valid;
#pragma unroll
      for (int j = 0; j < KB; j++) {
        const int k = kb * KB + j;
        const unsigned char *q = g + (k0 + k) * ld;
        if (k >= valid) v[p][j] = v4i{0, 0, 0, 0};
        else if (runs_over && k == valid - 1) v[p][j] = row_end_piece(q + rows_valid * ES, (int)(rows_valid - col) * ES);
        else v[p][j] = load_piece(q + col * ES);
      }
    }
  }

  __device__ __forceinline__ void store(unsigned char *lds, int tid) const {
#pragma unroll
    for (int p = 0; p < PER; p++) {
      const int blk = tid + p * NTHREADS;
      if (blk >= BLOCKS) break;
      const int rb = blk % (ROWS / RB), kb = blk / (ROWS / RB);
      if constexpr (ES == 2) {
#pragma unroll
        for (int i = 0; i < 8; i++) {  // row i: dword j = { k = 2j , k = 2j+1 }
          v4i t;
#pragma unroll
          for (int j = 0; j < 4; j++) {
            const unsigned lo = (unsigned)v[p][2 * j][i >> 1], hi = (unsigned)v[p][2 * j + 1][i >> 1];
            t[j] = (int)__builtin_amdgcn_perm(hi, lo, (i & 1) ? 0x07060302u : 0x05040100u);
          }
          const int r = rb * 8 + i;
          *reinterpret_cast<v4i *>(lds + r * SLAB + lds_slot(r, kb) * 16) = t;
        }
      } else if constexpr (ES == 4) {
#pragma unroll
        for (int i = 0; i < 4; i++) {
          const v4i t = {v[p][0][i], v[p][1][i], v[p][2][i], v[p][3][i]};
          const int r = rb * 4 + i;
          *reinterpret_cast<v4i *>(lds + r * SLAB + lds_slot(r, kb) * 16) = t;
        }
      } else if constexpr (ES == 8) {
#pragma unroll
        for (int i = 0; i < 2; i++) {  // row i: its two k of this block, 8 bytes each
          const v4i t = {v[p][0][2 * i], v[p][0][2 * i + 1], v[p][1][2 * i], v[p][1][2 * i + 1]};
          const int r = rb * 2 + i;
          *reinterpret_cast<v4i *>(lds + r * SLAB + lds_slot(r, kb) * 16) = t;
        }
      } else {
#pragma unroll
        for (int c = 0; c < 4; c++) {  // dword column c holds rows 4c .. 4c+3 of the four k
          const unsigned w0 = (unsigned)v[p][0][c], w1 = (unsigned)v[p][1][c], w2 = (unsigned)v[p][2][c], w3 = (unsigned)v[p][3][c];
          const unsigned a01 = __builtin_amdgcn_perm(w1, w0, 0x05010400u), b01 = __builtin_amdgcn_perm(w1, w0, 0x07030602u);
          const unsigned a23 = __builtin_amdgcn_perm(w3, w2, 0x05010400u), b23 = __builtin_amdgcn_perm(w3, w2, 0x07030602u);
          const unsigned o[4] = {__builtin_amdgcn_perm(a23, a01, 0x05040100u), __builtin_amdgcn_perm(a23, a01, 0x07060302u),
                                 __builtin_amdgcn_perm(b23, b01, 0x05040100u), __builtin_amdgcn_perm(b23, b01, 0x07060302u)};
#pragma unroll
          for (int i = 0; i < 4; i++) {  // row 4c+i: its four k bytes are dword (kb % 4) of chunk (kb / 4)
            const int r = rb * 16 + 4 * c + i;
            *reinterpret_cast<unsigned *>(lds + r * SLAB + lds_slot(r, kb >> 2) * 16 + (kb & 3) * 4) = o[i];
          }
        }
      }
    }
  }
};

// ---- K-outer 1- and 2-byte operands of the big tiles: no register staging at all.  The slab is
// copied as it lies in memory -- [k][ROWS], ROWS*ES bytes per k -- straight into LDS, and the MFMA
// fragments are fetched with the transposing LDS reads of gfx950 (semantics measured on the part).
// Within each group of 16 lanes every lane supplies the address of an 8-byte run, and
//   ds_read_b64_tr_b16: lane j receives element j%4 of the runs of lanes j/4 + {0, 4, 8, 12};
//     with lane i pointing at (k0 + i/4, n0 + 4*(i%4)) lane j receives [k0..k0+3][n0 + j];
//   ds_read_b64_tr_b8:  lane j receives byte j%8 of the runs of lanes j/8 + {0, 2, .., 14};
//     with lane i pointing at (k0 + i/2, n0 + 8*(i%2)) lane j receives [k0..k0+7][n0 + j]
// -- in both cases half an MFMA operand (8 bytes of consecutive k of one row).
// LDS layout: k-major, the 16-byte chunk index of a k-row XOR-ed with a function of k chosen so
// that the 32 lanes served per clock (lanes 0..31, then 32..63) cover all 64 banks
// (SQ_LDS_BANK_CONFLICT = 0): per clock the 16-bit form touches 8 k-rows x 32 bytes
// (k = 8g + 4h + 0..3 for lane groups g and g+1), the 8-bit form 16 k-rows x 16 bytes
// (k = 16g + 8h + 0..7).  A k-row must span all banks, i.e. at least 256 bytes.
template <int ES>
__device__ __forceinline__ int tr_slot(int k, int chunk) {
  if constexpr (ES == 2) return chunk ^ ((k & 3) << 2) ^ (((k >> 3) & 1) << 1);
  else return chunk ^ (k & 7) ^ (((k >> 4) & 1) << 3);
}

// the same for k-rows narrower than the 256 bytes that span all LDS banks (int8 tiles of 64 or 128 columns): the
// chunk index XOR as many low bits of k as the row has chunk bits
template <int ES, int RBYTES>
__device__ __forceinline__ int tr_slot_w(int k, int chunk) {
  if constexpr (RBYTES >= 256) return tr_slot<ES>(k, chunk);
  else {
    static_assert(ES == 1 && (RBYTES == 128 || RBYTES == 64), "narrow k-rows: int8 tiles of 64 or 128 columns");
    return chunk ^ (k & (RBYTES / 16 - 1));
  }
}

template <int ES, int ROWS, int NWAVES>
struct KOuterDmaLoader {
  static constexpr int RBYTES = ROWS * ES;     // bytes per k-row of the slab
  static constexpr int INSTR = ROWS / 8;       // (128 / ES) k-rows * RBYTES / 1 KiB
  static constexpr int PER = INSTR / NWAVES;
  static_assert(RBYTES >= 256 && INSTR % NWAVES == 0, "needs at least 16 chunks per k-row");
  const unsigned char *src[PER];
  int lds_off[PER];
  int rem[PER];  // bytes of this lane's piece that lie inside its k-row, 0: all of them
  bool whole_pieces;  // (of a k-row, the same for all lanes: what nobody needs is jumped over, not looked at by each)

  // g: [K, cols] with `ld` bytes per k; the tile covers columns col0 .. col0+ROWS-1, of which cols_valid exist: chunks past the
  // edge re-read the last one, which runs into the next k-row where k-rows are not whole pieces (see KOuterStage)
  __device__ __forceinline__ void init(const unsigned char *__restrict__ g, int64_t ld, int64_t col0, int64_t cols_valid,
                                       int wave, int lane) {
    whole_pieces = (int)(cols_valid * ES) % 16 == 0;
#pragma unroll
    for (int i = 0; i < PER; i++) {
      const int t = wave + NWAVES * i;
      const int o = t * 1024 + lane * 16;
      const int k = o / RBYTES, slot = (o % RBYTES) / 16;
      int64_t byte = col0 * ES + tr_slot<ES>(k, slot) * 16;
      const int64_t last = (cols_valid * ES - 1) & ~(int64_t)15;
      byte = byte <= last ? byte : last;
      rem[i] = byte == last ? (int)(cols_valid * ES) & 15 : 0;
      src[i] = g + (int64_t)k * ld + byte;
      lds_off[i] = t * 1024;
    }
  }
  __device__ __forceinline__ void issue(int64_t k0, int64_t ld, unsigned char *lds) const {
#pragma unroll
    for (int i = 0; i < PER; i++)
      lds_dma16(src[i] + k0 * ld, lds + lds_off[i]);
  }
  // a slab of which only the first `valid` k-rows exist; the last one's piece that is not whole is zero until finish_partial
  __device__ __forceinline__ void issue_partial(int64_t k0, int64_t ld, int valid, unsigned char *lds, int wave, int lane) const {
#pragma unroll
    for (int i = 0; i < PER; i++) {
      const int k = ((wave + NWAVES * i) * 1024 + lane * 16) / RBYTES;
      lds_dma16(k < valid - (rem[i] != 0) ? src[i] + k0 * ld : (const unsigned char *)g_zero16, lds + lds_off[i]);
    }
  }
  __device__ __forceinline__ void finish_partial(int64_t k0, int64_t ld, int valid, unsigned char *lds, int wave, int lane) const {
    if (whole_pieces) return;
#pragma unroll
    for (int i = 0; i < PER; i++)
      if (rem[i] != 0 && ((wave + NWAVES * i) * 1024 + lane * 16) / RBYTES == valid - 1)
        *reinterpret_cast<v4i *>(lds + lds_off[i] + lane * 16) = row_end_piece(src[i] + k0 * ld + rem[i], rem[i]);
  }
  __device__ __forceinline__ void issue_at(int t, int spread, int phase, int skew, int64_t k0, int64_t ld, unsigned char *lds) const {
#pragma unroll
    for (int i = 0; i < PER; i++)
      if (t == i * spread / PER + phase + skew) lds_dma16(src[i] + k0 * ld, lds + lds_off[i]);
  }
};

// Swizzle of the [row][k] LDS layout of this kernel: the 16-byte chunk index XOR the part of
// lds_slot() that depends on the low four row bits only (the part that makes a fragment read of 16
// consecutive rows conflict-free).  A fragment's address is then one per-lane base per K step plus
// a compile-time multiple of 16 rows, which the LDS instruction carries as its immediate offset:
// two address registers per operand instead of one per fragment.
__device__ __forceinline__ int lds_slot16(int row, int chunk) {
  return chunk ^ (((row ^ (row >> 2)) & 1) | ((((row >> 1) ^ (row >> 2)) & 1) << 1) | ((((row >> 2) ^ (row >> 3)) & 1) << 2));
}

// K-inner rows [row0, row0 + ROWS) of an operand, ROWS x 128 B per slab, shared by NWAVES waves:
// PER instructions per wave, each filling 1 KiB of LDS (8 rows x 8 chunks).  Offsets are relative
// to the operand's first tile row (clamped into the matrix), so they fit 32 bits whenever
// 2 * ROWS * ld does (the host checks).
template <int ROWS, int NWAVES>
struct PPKInnerLoader {
  static constexpr int PER = ROWS / 8 / NWAVES;
  const unsigned char *base;
  unsigned off[PER];
  __device__ __forceinline__ void init(const unsigned char *g, int64_t ld, int64_t row0, int64_t rows_valid, int wave, int lane) {
    const int64_t first = row0 < rows_valid ? row0 : rows_valid - 1;
    base = wave_uniform(g + first * ld);
#pragma unroll
    for (int i = 0; i < PER; i++) {
      const int r = (wave + NWAVES * i) * 8 + (lane >> 3);
      int64_t gr = row0 + r;
      gr = gr < rows_valid ? gr : rows_valid - 1;
      off[i] = (unsigned)((gr - first) * ld) + lds_slot16(r, lane & 7) * 16;
    }
  }
  __device__ __forceinline__ void issue(int64_t kbyte0, unsigned char *lds, int wave) const {
    const unsigned char *b = base + kbyte0;
#pragma unroll
    for (int i = 0; i < PER; i++) lds_dma16_at(b, off[i], lds + (wave + NWAVES * i) * 1024);
  }
  // a slab of which only the first `valid` bytes of each row exist; a row's last piece, where it is not whole, is zero until
  // finish_partial writes it, behind the wave's wait for these requests
  __device__ __forceinline__ void issue_partial(int64_t kbyte0, int valid, unsigned char *lds, int wave, int lane) const {
    const unsigned char *b = base + kbyte0;
#pragma unroll
    for (int i = 0; i < PER; i++) {
      const int r = (wave + NWAVES * i) * 8 + (lane >> 3);
      lds_dma16(lds_slot16(r, lane & 7) * 16 + 16 <= valid ? b + off[i] : (const unsigned char *)g_zero16, lds + (wave + NWAVES * i) * 1024);
    }
  }
  __device__ __forceinline__ void finish_partial(int64_t kbyte0, int valid, unsigned char *lds, int wave, int lane) const {
    if ((valid & 15) == 0) return;
    const unsigned char *b = base + kbyte0 + (valid & 15);
    v4i v[PER];
#pragma unroll
    for (int i = 0; i < PER; i++)
      if (lds_slot16((wave + NWAVES * i) * 8 + (lane >> 3), lane & 7) == valid >> 4) v[i] = row_end_piece(b + off[i], valid & 15);
#pragma unroll
    for (int i = 0; i < PER; i++)
      if (lds_slot16((wave + NWAVES * i) * 8 + (lane >> 3), lane & 7) == valid >> 4)
        *reinterpret_cast<v4i *>(lds + (wave + NWAVES * i) * 1024 + lane * 16) = v[i];
  }
};

// K-outer columns [col0, col0 + ROWS) of an operand copied k-major ([k][ROWS * ES bytes]) for the
// transposing fragment reads (tr_slot layout of gemm_mfma.cuh), with 32-bit offsets from the tile's
// first column (clamped).
template <int ES, int ROWS, int NWAVES>
struct PPKOuterLoader {
  static constexpr int RBYTES = ROWS * ES;
  static constexpr int PER = ROWS / 8 / NWAVES;
  static_assert(RBYTES >= 256 || ES == 1, "a 2-byte k-row must span all LDS banks");
  const unsigned char *base;
  unsigned off[PER];
  int rem[PER];  // bytes of this lane's piece that lie inside its k-row, 0: all of them (KOuterDmaLoader)
  bool whole_pieces;
  __device__ __forceinline__ void init(const unsigned char *g, int64_t ld, int64_t col0, int64_t cols_valid, int wave, int lane) {
    whole_pieces = (int)(cols_valid * ES) % 16 == 0;
    const int64_t last = (cols_valid * ES - 1) & ~(int64_t)15;
    const int64_t first = col0 * ES <= last ? col0 * ES : last;
    base = wave_uniform(g + first);
#pragma unroll
    for (int i = 0; i < PER; i++) {
      const int o = (wave + NWAVES * i) * 1024 + lane * 16;
      const int k = o / RBYTES, slot = (o % RBYTES) / 16;
      int64_t byte = col0 * ES + tr_slot_w<ES, RBYTES>(k, slot) * 16;
      byte = byte <= last ? byte : last;
      rem[i] = byte == last ? (int)(cols_valid * ES) & 15 : 0;
      off[i] = (unsigned)((int64_t)k * ld + (byte - first));
    }
  }
  __device__ __forceinline__ void issue(int64_t k0, int64_t ld, unsigned char *lds, int wave) const {
    const unsigned char *b = base + k0 * ld;
#pragma unroll
    for (int i = 0; i < PER; i++) lds_dma16_at(b, off[i], lds + (wave + NWAVES * i) * 1024);
  }
  // a slab of which only the first `valid` k-rows exist; the last one's piece that is not whole is zero until finish_partial
  __device__ __forceinline__ void issue_partial(int64_t k0, int64_t ld, int valid, unsigned char *lds, int wave, int lane) const {
    const unsigned char *b = base + k0 * ld;
#pragma unroll
    for (int i = 0; i < PER; i++) {
      const int k = ((wave + NWAVES * i) * 1024 + lane * 16) / RBYTES;
      lds_dma16(k < valid - (rem[i] != 0) ? b + off[i] : (const unsigned char *)g_zero16, lds + (wave + NWAVES * i) * 1024);
    }
  }
  __device__ __forceinline__ void finish_partial(int64_t k0, int64_t ld, int valid, unsigned char *lds, int wave, int lane) const {
    if (whole_pieces) return;
    const unsigned char *b = base + k0 * ld;
#pragma unroll
    for (int i = 0; i < PER; i++)
      if (rem[i] != 0 && ((wave + NWAVES * i) * 1024 + lane * 16) / RBYTES == valid - 1)
        *reinterpret_cast<v4i *>(lds + (wave + NWAVES * i) * 1024 + lane * 16) = row_end_piece(b + off[i] + rem[i], rem[i]);
  }
};

}  // namespace hipnx
