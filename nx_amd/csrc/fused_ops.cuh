// The device side of the fused element-wise groups, shared by the interpreting kernels of
// fused.hip and by the kernels compiled at run time for one program (fused_rtc.cpp): the lane's
// vectors, the loads with their conversions, the rounding after every instruction, the kernel
// bodies, and the program as compile-time constants.  Both forms call the same functions in the
// same order on the same values, which is what makes their results bit-identical.
// This header is also given to the run-time compiler, which has no host headers: keep it to
// device code.
#pragma once
#include "elementwise_ops.cuh"
#include "reduce_ops.cuh"
#include "threefry.cuh"

namespace hipnx {


constexpr int FBLOCK = 256;
constexpr int FE = 8;  // elements per vector: two 16-byte accesses of f32, one of a 2-byte type
constexpr int FV = 1;  // vectors per lane and trip (more were measured: the registers they take cost more in
                       // waves per SIMD than the shared decoding saves: 276 / 303 / 402 us for 1 / 2 / 4)

static_assert(sizeof(hipnx_fused_instr) == 16, "an instruction is one 16-byte scalar load");

struct FusedArgs {
  int n_instr, n_inputs;
  int64_t pad_to_16;
  hipnx_fused_instr ins[HIPNX_FUSED_MAX_INSTR];
  const void *in[HIPNX_FUSED_MAX_INPUTS];
  int in_dt[HIPNX_FUSED_MAX_INPUTS];
  int64_t in_rs[HIPNX_FUSED_MAX_INPUTS];  // element stride between rows (0 = the same row for all)
  int in_cs[HIPNX_FUSED_MAX_INPUTS];      // element stride along a row: 1, or 0 = one value per row
  void *out;
  int out_dt;
  int words;  // the input that is not in memory: in[words] holds a key, and the input is the cipher's words (-1: there is none)
  int64_t rows, cols, vecs_per_row, nvec;
  // a reduction of the result along rows that are cut into segments (nseg > 1): segment `seg` of a row covers the
  // columns [seg * seg_len, min(cols, (seg + 1) * seg_len)) and leaves its raw accumulator in partial[row * nseg + seg]
  int64_t seg_len;
  void *partial;
  int nseg;
  // the input that is the result of a contraction and not in memory (-1: there is none): rows of l against rows of r, K contiguous
  // elements each, `scores_rows` rows of l per batch item; strides in elements along the batch's two axes and from row to row
  int scores, scores_inner;
  int64_t scores_rows;
  const void *l, *r;
  int64_t l_outer, l_inner, l_ld, r_outer, r_inner, r_ld;
  int key_parts, key_index;  // the key is number key_index of the key_parts that in[words] splits into (0 parts: in[words] itself)
  int beside_index;          // which of the key's parts goes to `beside` (FusedWordsArgs), where that is not null
};
// What only the kernels over random words take, behind the block that every kernel does (with it in that block
// the attention probabilities of 4 x 8 x 512 x 512 took 19.6 us a pass, 19.4 without).  It lies in the last of the block's 64-byte lines:
// in one more, 63711 normal samples took 6.56 us, 6.39 so.
struct FusedWordsArgs : FusedArgs {
  uint32_t *beside;
};
static_assert(sizeof(FusedArgs) / 64 == (sizeof(FusedWordsArgs) - 1) / 64, "no line of its own");

// The argument block is read where the launch put it (the kernel-argument segment, constant address
// space) with wave-uniform indices: indexing the by-value copy would move it to per-lane scratch.
typedef const __attribute__((address_space(4))) FusedArgs *KernArgs;
typedef const __attribute__((address_space(4))) FusedWordsArgs *WordsKernArgs;
typedef float Vecs[FV][FE];

// what a store to `dt` followed by a load would give back
__device__ __forceinline__ float round_to(float x, int dt) {
  switch (dt) {
    case HIPNX_BF16: return bf16_bits_to_f32(f32_to_bf16_bits_trunc(x));
    case HIPNX_F16: return (float)bits_f16(f32_to_f16_bits(x));
    default: return x;  // f32, and u8 truth values (0 / 1)
  }
}

// one uniform dispatch per instruction, the loops over the vectors inside each case
template <int OP>
__device__ __forceinline__ void unary_vecs(Vecs &x) {
#pragma unroll
  for (int u = 0; u < FV; u++)
#pragma unroll
    for (int e = 0; e < FE; e++) x[u][e] = unary_apply<OP, float>(x[u][e], 32);
}

template <int OP>
__device__ __forceinline__ void binary_vecs(Vecs &x, const Vecs &y, bool swap) {
#pragma unroll
  for (int u = 0; u < FV; u++)
#pragma unroll
    for (int e = 0; e < FE; e++)
      x[u][e] = swap ? binary_apply<OP, float, false>(y[u][e], x[u][e]) : binary_apply<OP, float, false>(x[u][e], y[u][e]);
}

__device__ __forceinline__ float element_to_f32(uint32_t bits, int dt) {
  switch (dt) {
    case HIPNX_U8: case HIPNX_U16: case HIPNX_U32: return (float)bits;
    case HIPNX_S8: return (float)(int32_t)(int8_t)bits;
    case HIPNX_S16: return (float)(int32_t)(int16_t)bits;
    case HIPNX_S32: return (float)(int32_t)bits;
    case HIPNX_F16: return (float)bits_f16((uint16_t)bits);
    case HIPNX_BF16: return bf16_bits_to_f32((uint16_t)bits);
    default: return __uint_as_float(bits);
  }
}

// input k (element type dt, column stride cs) for the lane's FV vectors: all loads are requested,
// then converted.  UNAL: the vectors begin at any element (rows that are not whole vectors): the loads claim no alignment.
template <bool UNAL = false>
__device__ __forceinline__ void load_input_as(KernArgs a, int k, int dt, int cs, const int64_t (&row)[FV],
                                              const int64_t (&col)[FV], Vecs &dst) {
  const int esz = (dt == HIPNX_U8 || dt == HIPNX_S8) ? 1 : (dt == HIPNX_U32 || dt == HIPNX_S32 || dt == HIPNX_F32) ? 4 : 2;
  const char *base = (const char *)a->in[k];
  const int64_t rs = a->in_rs[k];
  uint32_t w[FV][FE];  // raw words: 8 for 4-byte elements, 4 for 2-byte ones, 2 for bytes, 1 for a broadcast value
#pragma unroll
  for (int u = 0; u < FV; u++) {
    const char *p = base + (row[u] * rs + col[u] * cs) * esz;
    if (cs == 0) {
      w[u][0] = esz == 4 ? *reinterpret_cast<const uint32_t *>(p)
                : esz == 2 ? (uint32_t)*reinterpret_cast<const uint16_t *>(p)
                           : (uint32_t)*reinterpret_cast<const uint8_t *>(p);
    } else if constexpr (UNAL) {
      if (esz == 4) __builtin_memcpy(w[u], p, FE * 4);
      else if (esz == 2) __builtin_memcpy(w[u], p, FE * 2);
      else __builtin_memcpy(w[u], p, FE);
    } else if (esz == 4) {
      const uint4 lo = *reinterpret_cast<const uint4 *>(p), hi = *reinterpret_cast<const uint4 *>(p + 16);
      w[u][0] = lo.x; w[u][1] = lo.y; w[u][2] = lo.z; w[u][3] = lo.w;
      w[u][4] = hi.x; w[u][5] = hi.y; w[u][6] = hi.z; w[u][7] = hi.w;
    } else if (esz == 2) {
      const uint4 lo = *reinterpret_cast<const uint4 *>(p);
      w[u][0] = lo.x; w[u][1] = lo.y; w[u][2] = lo.z; w[u][3] = lo.w;
    } else {
      const uint2 lo = *reinterpret_cast<const uint2 *>(p);
      w[u][0] = lo.x; w[u][1] = lo.y;
    }
  }
#pragma unroll
  for (int u = 0; u < FV; u++) {
    if (cs == 0) {
      const float v = element_to_f32(w[u][0], dt);
#pragma unroll
      for (int e = 0; e < FE; e++) dst[u][e] = v;
    } else if (esz == 4) {
      if (dt == HIPNX_F32) {
#pragma unroll
        for (int e = 0; e < FE; e++) dst[u][e] = __uint_as_float(w[u][e]);
      } else {
#pragma unroll
        for (int e = 0; e < FE; e++) dst[u][e] = element_to_f32(w[u][e], dt);
      }
    } else if (esz == 2) {
#pragma unroll
      for (int e = 0; e < FE; e++) dst[u][e] = element_to_f32((w[u][e / 2] >> (16 * (e & 1))) & 0xFFFFu, dt);
    } else {
#pragma unroll
      for (int e = 0; e < FE; e++) dst[u][e] = element_to_f32((w[u][e / 4] >> (8 * (e & 3))) & 0xFFu, dt);
    }
  }
}

// the last, partial vector of a flat index space: only its first `valid` elements exist in memory
__device__ __forceinline__ void load_input_tail(KernArgs a, int k, int dt, int cs, const int64_t (&row)[FV],
                                                const int64_t (&col)[FV], int valid, Vecs &dst) {
  if (cs == 0) {
    load_input_as(a, k, dt, cs, row, col, dst);
    return;
  }
  const int esz = (dt == HIPNX_U8 || dt == HIPNX_S8) ? 1 : (dt == HIPNX_U32 || dt == HIPNX_S32 || dt == HIPNX_F32) ? 4 : 2;
  const char *p = (const char *)a->in[k] + (row[0] * a->in_rs[k] + col[0]) * esz;
#pragma unroll
  for (int e = 0; e < FE; e++) {
    uint32_t w = 0;
    if (e < valid)
      w = esz == 4 ? *reinterpret_cast<const uint32_t *>(p + 4 * e)
          : esz == 2 ? (uint32_t)*reinterpret_cast<const uint16_t *>(p + 2 * e)
                     : (uint32_t)*reinterpret_cast<const uint8_t *>(p + e);
    dst[0][e] = element_to_f32(w, dt);
  }
}

__device__ __forceinline__ void copy_vecs(Vecs &dst, const Vecs &src) {
#pragma unroll
  for (int u = 0; u < FV; u++)
#pragma unroll
    for (int e = 0; e < FE; e++) dst[u][e] = src[u][e];
}

struct Saved {
  Vecs s[HIPNX_FUSED_SAVED];
};


// ---- the program as compile-time constants ------------------------------------------------------
// P holds the program one field per array (kind[], op[], src[], arg[], src2[], arg2[], flags[],
// dt[], imm[] and imm2[] as f32 bit patterns), the inputs' element types and column strides, and
// the result type.  Every branch the interpreter takes on an instruction field is taken by the
// compiler here.
typedef float RowStats[HIPNX_FUSED_STATS];  // results of the row reductions of earlier stages (fused_row_stages_body)

// what a lane keeps of one vector of its row between stages (fused_row_stages_body)
struct RowVector {
  float carry[FE];  // the value the previous stage reduced
  float held[FE];   // input P::held
};

// How the lanes of a row share it (P::form).  In every form a lane meets its elements in the order in which the separate
// reduction of rows of that length folds them (reduce_rows_kernel and its short-row forms) -- but for the rows of contracted
// scores, which may have fewer lanes (share_row, fused_rtc.hip): a sum along them is added in an order of its own.
//   ROW_WHOLE: rows of whole vectors; lane l takes the vectors l, l + tpr, ...
//   ROW_LANE: rows of at most 16 elements; a lane takes a row (tpr = 1): its vectors, then the P::tail elements behind them.
//   ROW_GROUP: rows of 17 to 256 elements that are not whole vectors; 8, 16 or 32 lanes, so that each has one vector at most;
//     the elements behind the last vector one per lane.
//   ROW_RAGGED: longer rows that are not whole vectors; the elements up to a vector boundary of the BUFFER one per lane, whole
//     aligned vectors as ROW_WHOLE, the elements behind them one per lane.
// Rows off the vector grid went node by node before, every intermediate through memory: f32 layer norm of 26248 x 185
// 106 us, bf16 softmax of 247650 x 178 160 us.
enum { ROW_WHOLE, ROW_LANE, ROW_GROUP, ROW_RAGGED };

// ---- a contraction's result as an input (fused_scores_body) ----
constexpr int SCORE_ROWS = 16;
// the block's rows of it in LDS: row i's column c at element c + score_shift of row i, so that the vectors of a ROW_RAGGED row are
// aligned; a pitch that sets the sixteen rows four banks apart
template <typename P>
__device__ __forceinline__ uint16_t *score_row(int i) {
  __shared__ __attribute__((aligned(16))) uint16_t sm[SCORE_ROWS * (P::scores_cols + 8)];
  return sm + i * (P::scores_cols + 8);
}
__device__ __forceinline__ int score_shift(int64_t r, int64_t cols, bool ragged) { return ragged ? (int)(r * cols & 7) : 0; }
template <typename P>
__device__ __forceinline__ void load_scores(KernArgs a, int64_t r, int64_t k, int valid, Vecs &dst) {
  const int i = (int)((uint32_t)r % (uint32_t)a->scores_rows) % SCORE_ROWS;
  const uint16_t *p = score_row<P>(i) + k + score_shift(r, a->cols, P::form == ROW_RAGGED);
  uint32_t w[FE];
  if (valid == FE) {
    const uint4 v = *reinterpret_cast<const uint4 *>(p);
    w[0] = v.x & 0xFFFFu, w[1] = v.x >> 16, w[2] = v.y & 0xFFFFu, w[3] = v.y >> 16, w[4] = v.z & 0xFFFFu, w[5] = v.z >> 16, w[6] = v.w & 0xFFFFu, w[7] = v.w >> 16;
  } else {
#pragma unroll
    for (int e = 0; e < FE; e++) w[e] = e < valid ? p[e] : 0u;
  }
#pragma unroll
  for (int e = 0; e < FE; e++) dst[0][e] = element_to_f32(w[e], P::in_dt[P::scores < 0 ? 0 : P::scores]);
}

template <typename P, int SRC, int ARG, unsigned IMM, bool RAW>
__device__ __forceinline__ void fetch_static(KernArgs a, const Saved &S, const RowStats &stats, const int64_t (&row)[FV],
                                             const int64_t (&col)[FV], int valid, const RowVector *kept, Vecs &dst) {
  if constexpr (SRC == HIPNX_FUSED_SRC_CARRY) {
#pragma unroll
    for (int e = 0; e < FE; e++) dst[0][e] = kept->carry[e];
  } else if constexpr (SRC == HIPNX_FUSED_SRC_INPUT && ARG == P::words) {
#pragma unroll
    for (int e = 0; e < FE; e++) dst[0][e] = RAW ? kept->held[e] : element_to_f32(__float_as_uint(kept->held[e]), HIPNX_U32);
  } else if constexpr (SRC == HIPNX_FUSED_SRC_INPUT && ARG == P::held && !RAW) {
#pragma unroll
    for (int e = 0; e < FE; e++) dst[0][e] = kept->held[e];
  } else if constexpr (SRC == HIPNX_FUSED_SRC_ROWSTAT) {
#pragma unroll
    for (int u = 0; u < FV; u++)
#pragma unroll
      for (int e = 0; e < FE; e++) dst[u][e] = stats[ARG];
  } else if constexpr (SRC == HIPNX_FUSED_SRC_INPUT) {
    if constexpr (ARG == P::scores) {
      load_scores<P>(a, row[0], col[0], valid, dst);
      return;
    }
    // RAW: the words of a 4-byte input as they are (what the f32 path does with its bits)
    if (valid == FE) load_input_as<P::unal>(a, ARG, RAW ? (int)HIPNX_F32 : P::in_dt[ARG], P::in_cs[ARG], row, col, dst);
    else load_input_tail(a, ARG, RAW ? (int)HIPNX_F32 : P::in_dt[ARG], P::in_cs[ARG], row, col, valid, dst);
  } else if constexpr (SRC == HIPNX_FUSED_SRC_SAVED) {
    copy_vecs(dst, S.s[ARG]);
  } else {
#pragma unroll
    for (int u = 0; u < FV; u++)
#pragma unroll
      for (int e = 0; e < FE; e++) dst[u][e] = __uint_as_float(IMM);
  }
}

// Exponentials over one value of their row (a softmax's last stage) in programs of a few vectors a lane, which vector instructions
// bound: x / y by Markstein's corrected quotient: the correctly rounded reciprocal r of y, q = x r, q + r (x - q y), the last two fused.
// The correction is at most 1.5 units of q and wrong by 2^-24 of itself, its residual by a unit of the product's last place: the result can
// miss the correctly rounded quotient only where x / y lies within 5 / (2 y) units (y as a 24-bit integer) of a midpoint between
// two numbers.  All 4.6 10^7 pairs of 24-bit significands within 8 / (2 y) were tried: each gives division's bits.  (While nothing
// leaves the normal numbers: the ranges tested below.)  Three instructions an element and two for the test instead of seventeen slots.  (With more
// vectors a lane the branch costs the overlap of their trips: f32 8192 x 32000, sixteen vectors, 385 -> 539 us.)
template <typename P, int PC>
constexpr bool divides_exponentials() {
  constexpr auto is_exp = [](int i) { return P::kind[i] == HIPNX_FUSED_UNARY && P::op[i] == HIPNX_EXP; };
  if (PC < 1 || P::nv > (P::scores >= 0 ? 4 : 2) || (P::nv == 0 && P::form != ROW_LANE)) return false;
  if (is_exp(PC - 1)) return true;
  if (P::kind[PC - 1] != HIPNX_FUSED_SET || P::src[PC - 1] != HIPNX_FUSED_SRC_CARRY) return false;
  for (int i = PC - 1; i > 0; i--)  // what the stage before left: the value its reduction was taken over
    if (P::kind[i] == HIPNX_FUSED_ROW_REDUCE) return is_exp(i - 1);
  return false;
}
__device__ __forceinline__ void divide_exponentials(Vecs &x, float y) {
  uint32_t least = 0xFFFFFFFFu, most = 0;
#pragma unroll
  for (int e = 0; e < FE; e++) {
    const uint32_t b = __float_as_uint(x[0][e]);
    least = b - 1 < least ? b - 1 : least;  // (zero counts as large)
    most = b > most ? b : most;
  }
  if (least >= (37u << 23) - 1 && most < (227u << 23) && y >= 0x1p-20f && y <= 0x1p29f) {  // x: 0, or 2^-90 to 2^100
    const float r = 1.0f / y;
#pragma unroll
    for (int e = 0; e < FE; e++) {
      const float q = x[0][e] * r;
      x[0][e] = __builtin_fmaf(__builtin_fmaf(-q, y, x[0][e]), r, q);
    }
  } else {
#pragma unroll
    for (int e = 0; e < FE; e++) x[0][e] = binary_apply<HIPNX_DIVIDE, float, false>(x[0][e], y);
  }
}

// What an arithmetic instruction computes is never a NaN whose set bits all lie in the half that truncation to bf16 drops
// (a computed NaN is a quiet one): the bits can be cut without looking.  (A value that only passes through can be.)
constexpr bool computes_quiet_nan(int kind, int op) {
  return (kind == HIPNX_FUSED_UNARY && (op == HIPNX_EXP || op == HIPNX_LOG || op == HIPNX_SQRT || op == HIPNX_RSQRT || op == HIPNX_TANH)) ||
         (kind == HIPNX_FUSED_BINARY && (op == HIPNX_ADD || op == HIPNX_SUBTRACT || op == HIPNX_MULTIPLY || op == HIPNX_DIVIDE));
}

// 32-bit integers travel through the lane's vectors as raw bits; an operation on them widens to
// the 64-bit integer class of the separate kernels and keeps the low word, as their stores do
template <int OP, bool UNS>
__device__ __forceinline__ float int_binary(float x, float y, bool swap) {
  const uint32_t a = __float_as_uint(swap ? y : x), b = __float_as_uint(swap ? x : y);
  const int64_t wa = UNS ? (int64_t)a : (int64_t)(int32_t)a, wb = UNS ? (int64_t)b : (int64_t)(int32_t)b;
  return __uint_as_float((uint32_t)binary_apply<OP, int64_t, UNS>(wa, wb));
}

template <int OP, bool UNS>
__device__ __forceinline__ float int_unary(float x) {
  const uint32_t a = __float_as_uint(x);
  return __uint_as_float((uint32_t)unary_apply<OP, int64_t>(UNS ? (int64_t)a : (int64_t)(int32_t)a, 32));
}

// A program that relabels bits or computes on integers can look at the bits of a float it made.  The separate kernels
// store every NaN they compute as the one quiet NaN (0x7FC00000), so such a program does the same after each float
// instruction that one of those follows (the last store writes the one quiet NaN itself); bits that only pass through (an
// input, a BITCAST) stay as they are, there as here.
template <typename P>
constexpr bool bits_are_observed_after(int pc) {
  for (int i = pc + 1; i < P::n_instr; i++)
    if (P::kind[i] == HIPNX_FUSED_BITCAST || (P::flags[i] & HIPNX_FUSED_FLAG_INT) != 0) return true;
  return false;
}
// the result is the bits of the last instruction when that is a BITCAST to f32 (any NaN pattern leaves as it came)
template <typename P>
constexpr bool result_is_relabelled_bits() {
  return P::out_dt == HIPNX_U32 || P::out_dt == HIPNX_S32 || (P::out_dt == HIPNX_F32 && P::kind[P::n_instr - 1] == HIPNX_FUSED_BITCAST);
}

// Where integer bits become a float (a BITCAST, a conversion of a computed integer) the compiler is made to forget how
// the bits were computed.  Knowing it, this compiler (a) takes an integer with few significant bits for exactly
// convertible to f16 whatever its size and drops the rounding to f16 -- (x << 24) as f16 then stays finite -- and (b) turns
// an arithmetic shift by 24 whose result a float instruction reads into that instruction's byte select, which cannot
// sign-extend: the bits of -3 relabelled as f32 (a NaN) minus 1.0 came out as -1.0.
__device__ __forceinline__ void forget_provenance(float &x) { asm volatile("" : "+v"(x)); }

// instructions PC .. END-1
template <typename P, int PC, int END>
__device__ __forceinline__ void static_steps(KernArgs a, const int64_t (&row)[FV], const int64_t (&col)[FV], Vecs &acc, Saved &S,
                                             const RowStats &stats, int valid = FE, const RowVector *kept = nullptr) {
  if constexpr (PC < END) {
    constexpr int kind = P::kind[PC], op = P::op[PC], src = P::src[PC], arg = P::arg[PC];
    constexpr int src2 = P::src2[PC], arg2 = P::arg2[PC], flags = P::flags[PC], dt = P::dt[PC];
    constexpr unsigned imm = P::imm[PC], imm2 = P::imm2[PC];
    constexpr bool ints = (flags & HIPNX_FUSED_FLAG_INT) != 0, uns = dt == HIPNX_U32;
    if constexpr (kind == HIPNX_FUSED_SET) {
      fetch_static<P, src, arg, imm, ints>(a, S, stats, row, col, valid, kept, acc);
    } else if constexpr (kind == HIPNX_FUSED_UNARY) {
      if constexpr (ints) {
#pragma unroll
        for (int u = 0; u < FV; u++)
#pragma unroll
          for (int e = 0; e < FE; e++) acc[u][e] = int_unary<op, uns>(acc[u][e]);
      } else {
        unary_vecs<op>(acc);
      }
    } else if constexpr (kind == HIPNX_FUSED_BINARY && op == HIPNX_DIVIDE && src == HIPNX_FUSED_SRC_ROWSTAT && !ints && !(flags & 1) && divides_exponentials<P, PC>()) {
      if (valid == FE) divide_exponentials(acc, stats[arg]);
      else {
#pragma unroll
        for (int e = 0; e < FE; e++) acc[0][e] = binary_apply<HIPNX_DIVIDE, float, false>(acc[0][e], stats[arg]);
      }
    } else if constexpr (kind == HIPNX_FUSED_BINARY) {
      Vecs y;
      fetch_static<P, src, arg, imm, ints>(a, S, stats, row, col, valid, kept, y);
      if constexpr (ints) {
#pragma unroll
        for (int u = 0; u < FV; u++)
#pragma unroll
          for (int e = 0; e < FE; e++) acc[u][e] = int_binary<op, uns>(acc[u][e], y[u][e], (flags & 1) != 0);
      } else {
        binary_vecs<op>(acc, y, (flags & 1) != 0);
      }
    } else if constexpr (kind == HIPNX_FUSED_SELECT) {
      Vecs y, z;
      fetch_static<P, src, arg, imm, false>(a, S, stats, row, col, valid, kept, y);
      fetch_static<P, src2, arg2, imm2, false>(a, S, stats, row, col, valid, kept, z);
#pragma unroll
      for (int u = 0; u < FV; u++)
#pragma unroll
        for (int e = 0; e < FE; e++) acc[u][e] = acc[u][e] != 0.0f ? y[u][e] : z[u][e];  // NaN is true
    } else if constexpr (kind == HIPNX_FUSED_AS_TYPE && ints) {  // the integer of type `op`, held as bits, to a float
#pragma unroll
      for (int u = 0; u < FV; u++)
#pragma unroll
        for (int e = 0; e < FE; e++) {
          forget_provenance(acc[u][e]);
          acc[u][e] = element_to_f32(__float_as_uint(acc[u][e]), op);
        }
    } else if constexpr (kind == HIPNX_FUSED_BITCAST) {  // changes nothing in the registers
#pragma unroll
      for (int u = 0; u < FV; u++)
#pragma unroll
        for (int e = 0; e < FE; e++) forget_provenance(acc[u][e]);
    }  // a float AS_TYPE is the rounding below
    constexpr bool computed = kind == HIPNX_FUSED_UNARY || kind == HIPNX_FUSED_BINARY || kind == HIPNX_FUSED_SELECT || kind == HIPNX_FUSED_AS_TYPE ||
                              (kind == HIPNX_FUSED_SET && (src == HIPNX_FUSED_SRC_ROWSTAT || src == HIPNX_FUSED_SRC_CARRY));
    if constexpr (dt == HIPNX_F32 && computed && bits_are_observed_after<P>(PC)) {
#pragma unroll
      for (int u = 0; u < FV; u++)
#pragma unroll
        for (int e = 0; e < FE; e++) {  // (tested on the bits: a float comparison that selects between floats is folded away)
          const uint32_t b = __float_as_uint(acc[u][e]);
          acc[u][e] = __uint_as_float((b & 0x7FFFFFFFu) > 0x7F800000u ? 0x7FC00000u : b);
        }
    }
    if constexpr (dt == HIPNX_BF16 && !ints && computes_quiet_nan(kind, op) && !bits_are_observed_after<P>(PC)) {
#pragma unroll
      for (int u = 0; u < FV; u++)
#pragma unroll
        for (int e = 0; e < FE; e++) acc[u][e] = __uint_as_float(__float_as_uint(acc[u][e]) & 0xFFFF0000u);
    } else if constexpr (dt == HIPNX_BF16 || dt == HIPNX_F16) {
#pragma unroll
      for (int u = 0; u < FV; u++)
#pragma unroll
        for (int e = 0; e < FE; e++) acc[u][e] = round_to(acc[u][e], dt);
    }
    if constexpr ((flags >> 4) != 0) copy_vecs(S.s[(flags >> 4) - 1], acc);
    static_steps<P, PC + 1, END>(a, row, col, acc, S, stats, valid, kept);
  }
}

template <typename P>
struct RunStatic {
  static __device__ __forceinline__ void run(KernArgs a, const int64_t (&row)[FV], const int64_t (&col)[FV], Vecs &acc, int valid = FE) {
    Saved S;
    const RowStats none = {};
    static_steps<P, 0, P::n_instr>(a, row, col, acc, S, none, valid);
  }
  // a u32 / s32 result leaves as the bits it is held as
  static __device__ __forceinline__ int out_dt(KernArgs) { return P::out_dt; }
  static constexpr bool raw_out = result_is_relabelled_bits<P>();
};

// ---- kernel bodies: RUN is RunStatic<P> or the interpreter of fused.hip ---------------------------
template <typename RUN>
__device__ __forceinline__ void fused_elementwise_body() {
  KernArgs a = (KernArgs)__builtin_amdgcn_kernarg_segment_ptr();
  const int64_t nvec = a->nvec, vecs_per_row = a->vecs_per_row, cols = a->cols;
  const int64_t stride = (int64_t)gridDim.x * FBLOCK;
  for (int64_t v0 = (int64_t)blockIdx.x * FBLOCK + threadIdx.x; v0 < nvec; v0 += stride * FV) {
    int64_t row[FV], col[FV];
    bool live[FV];
#pragma unroll
    for (int u = 0; u < FV; u++) {
      int64_t v = v0 + u * stride;
      live[u] = v < nvec;
      if (!live[u]) v = v0;  // a vector past the end repeats the lane's first one and is not stored
      row[u] = 0;
      col[u] = v * FE;
      if (vecs_per_row != nvec) {  // more than one row
        row[u] = nvec <= 0xFFFFFFFFll ? (int64_t)((uint32_t)v / (uint32_t)vecs_per_row) : v / vecs_per_row;
        col[u] = (v - row[u] * vecs_per_row) * FE;
      }
    }
    static_assert(FV == 1, "the partial last vector is written for one vector per lane");
    // a flat index space need not be a whole number of vectors: the last one is partial
    const int64_t left = a->rows * cols - (row[0] * cols + col[0]);
    const int valid = left < FE ? (int)left : FE;
    Vecs acc;
    if (valid == FE) RUN::run(a, row, col, acc);
    else RUN::run(a, row, col, acc, valid);
    void *out = (void *)a->out;
    const int odt = RUN::out_dt(a);
#pragma unroll
    for (int u = 0; u < FV; u++) {
      if (!live[u]) continue;
      const int64_t at = row[u] * cols + col[u];
      if (valid < FE) {
        for (int e = 0; e < valid; e++) {
          if constexpr (RUN::raw_out) ((uint32_t *)out)[at + e] = __float_as_uint(acc[u][e]);
          else store_one<float>(out, odt, at + e, acc[u][e]);
        }
      } else if constexpr (RUN::raw_out) {
        uint4 *p = reinterpret_cast<uint4 *>((uint32_t *)out + at);
        p[0] = make_uint4(__float_as_uint(acc[u][0]), __float_as_uint(acc[u][1]), __float_as_uint(acc[u][2]), __float_as_uint(acc[u][3]));
        p[1] = make_uint4(__float_as_uint(acc[u][4]), __float_as_uint(acc[u][5]), __float_as_uint(acc[u][6]), __float_as_uint(acc[u][7]));
      } else {
        store_vec<float, FE>(out, odt, at, acc[u]);
      }
    }
  }
}

// A group over random words that exist only here: a lane enciphers eight counter pairs and takes the program over the two vectors
// of words they give, elements i .. i + 7 and half + i .. half + i + 7 (the order of threefry2x32_kernel, nx/lib/nx/random.ex:214-229).
// Bound by vector instructions, the cipher's (35 an element) and the program's (66 for normal samples); the words' way
// through memory and the launches in front of it are gone: 2^26 normal samples 227 -> 183 us a pass, 664464 of them 27.7 -> 10.8.
template <typename P>
__device__ __forceinline__ void fused_words_body() {
  WordsKernArgs a = (WordsKernArgs)__builtin_amdgcn_kernarg_segment_ptr();
  const uint32_t *key = (const uint32_t *)a->in[P::words];
  uint32_t key1 = __builtin_amdgcn_readfirstlane(key[0]), key2 = __builtin_amdgcn_readfirstlane(key[1]);
  if (a->beside && blockIdx.x == 0) {  // (uniform: a launch of its own cost 1.6 us on the device and 2.4 on the host)
    uint32_t b1 = key1, b2 = key2;
    threefry_sub_key(b1, b2, a->key_parts, a->beside_index);
    if (threadIdx.x == 0) ((uint32_t *)a->beside)[0] = b1, ((uint32_t *)a->beside)[1] = b2;
  }
  if (a->key_parts > 0) threefry_sub_key(key1, key2, a->key_parts, a->key_index);
  const int64_t n = a->cols, half = (n + 1) / 2, groups = (half + FE - 1) / FE;
  for (int64_t g = (int64_t)blockIdx.x * FBLOCK + threadIdx.x; g < groups; g += (int64_t)gridDim.x * FBLOCK) {
    uint32_t w[2][FE];
#pragma unroll
    for (int e = 0; e < FE; e++) {
      w[0][e] = (uint32_t)(g * FE + e);
      w[1][e] = half + g * FE + e < n ? (uint32_t)(half + g * FE + e) : 0u;
      threefry_pair(w[0][e], w[1][e], key1, key2);
    }
#pragma unroll 1
    for (int side = 0; side < 2; side++) {
      const int64_t at = side * half + g * FE, left = (side ? n : half) - at;
      const int valid = left < FE ? (int)left : FE;
      if (valid <= 0) break;
      RowVector words;
#pragma unroll
      for (int e = 0; e < FE; e++) words.held[e] = __uint_as_float(side ? w[1][e] : w[0][e]);
      const int64_t row[FV] = {0}, col[FV] = {at};
      Vecs x;
      Saved S;
      const RowStats none = {};
      static_steps<P, 0, P::n_instr>(a, row, col, x, S, none, valid, &words);
      void *out = (void *)a->out;
      constexpr bool raw = result_is_relabelled_bits<P>();
      constexpr int bytes = FE * (raw || P::out_dt == HIPNX_F32 ? 4 : P::out_dt == HIPNX_U8 ? 1 : 2);
      raw_vec<bytes> v;
      if constexpr (raw) {
        uint32_t bits[FE];
#pragma unroll
        for (int e = 0; e < FE; e++) bits[e] = __float_as_uint(x[0][e]);
        __builtin_memcpy(&v, bits, bytes);
      } else store_vec<float, FE>(&v, P::out_dt, 0, x[0]);
      if (valid == FE) __builtin_memcpy((char *)out + at * (bytes / FE), &v, bytes);
      else {
#pragma unroll
        for (int e = 0; e < FE - 1; e++)
          if (e < valid) {
            if constexpr (raw) ((uint32_t *)out)[at + e] = __float_as_uint(x[0][e]);
            else store_one<float>(out, P::out_dt, at + e, x[0][e]);
          }
      }
    }
  }
}

// The group's result reduced along its rows without ever being stored: TPR lanes per row walk it
// in the order of reduce_rows_kernel (lane l takes the vectors l, l + TPR, ... and folds their
// elements in turn, then lanes combine by wave shuffles and the block's waves through LDS) with the
// same reducer policy, so the value equals what the element-wise group followed by the separate
// reduction kernel gives, bit for bit.  A few very long rows are cut into segments exactly as that
// kernel cuts them (plan_row_segments), a work-group each, and the same second kernel folds them.
template <typename RUN, typename R, typename CT, int TPR>
__device__ __forceinline__ void fused_reduce_rows_body() {
  static_assert(FV == 1, "one vector per lane and step");
  KernArgs a = (KernArgs)__builtin_amdgcn_kernarg_segment_ptr();
  constexpr int RPB = FBLOCK / TPR;
  const int sub = threadIdx.x / TPR, lane = threadIdx.x % TPR;
  const int64_t rows = a->rows, red = a->cols;
  const int nseg = a->nseg;
  const int64_t unit = (int64_t)blockIdx.x * RPB + sub;  // (row, segment): whole rows unless nseg > 1
  const int64_t r = nseg > 1 ? unit / nseg : unit;
  const int seg = nseg > 1 ? (int)(unit - r * nseg) : 0;
  const int64_t k0 = nseg > 1 ? (int64_t)seg * a->seg_len : 0;
  const int64_t k1 = nseg > 1 && k0 + a->seg_len < red ? k0 + a->seg_len : red;
  typename R::acc_t acc = R::init();
  if (r < rows) {
    const int64_t step = (int64_t)TPR * FE;
    for (int64_t k = k0 + (int64_t)lane * FE; k < k1; k += step) {
      const int64_t row[FV] = {r}, col[FV] = {k};
      Vecs x;
      RUN::run(a, row, col, x);
#pragma unroll
      for (int e = 0; e < FE; e++) acc = R::accumulate(acc, (CT)x[0][e], k + e);
    }
  }
  acc = wave_reduce<R>(acc);
  if constexpr (TPR > WAVE) {
    __shared__ typename R::acc_t sm[FBLOCK / WAVE];
    if (threadIdx.x % WAVE == 0) sm[threadIdx.x / WAVE] = acc;
    __syncthreads();
    if (threadIdx.x == 0) {
#pragma unroll
      for (int w = 1; w < FBLOCK / WAVE; w++) acc = R::combine(acc, sm[w]);
    }
  }
  if (lane == 0 && r < rows) {
    if (nseg > 1) ((typename R::acc_t *)a->partial)[r * nseg + seg] = acc;
    else finalize((void *)a->out, a->out_dt, r, acc);
  }
}

// ---- several stages over the same rows in one kernel ------------------------------------------------
// A program with HIPNX_FUSED_ROW_REDUCE markers is a sequence of stages: each stage but the last
// ends in a reduction of its value along the row, and later stages read that row statistic as an
// operand (softmax: the row maximum, then the sum of the exponentials, then the division).  A group of
// lanes takes a row through all stages; a stage walks the row exactly as the separate reduction does
// (same lanes, same order, same reducer), and a statistic is carried on as the value a
// store to its type and a load would give -- so the result equals the separate kernels', bit for bit.
// A row that a lane's registers hold (P::held: an input that more than one stage reads, at most 16 vectors a lane) is read
// from memory once; a longer one, and one of a program walked in a loop, is read again by every stage.  Bound by memory: f32 softmax of
// 8192 x 32000 in 381 us (5.5 TB/s; 600 with a read per stage), f32 layer norm of 16384 x 1024 in 25 us (5.4 TB/s).
template <typename CT>
__device__ __forceinline__ float as_stored(CT v, int dt) {
  switch (dt) {
    case HIPNX_BF16: return bf16_bits_to_f32(conv<CT>::to_bf16(v));
    case HIPNX_F16: return (float)bits_f16(conv<CT>::to_f16(v));
    default: return __uint_as_float(conv<CT>::to_f32(v));
  }
}

template <int N>
struct Elements {
  static constexpr int n = N;
};

struct RowWalk {
  int64_t begin, end;  // the vectors of the row, all its lanes': columns [begin, end)
  int64_t cols;
};
template <typename P>
__device__ __forceinline__ RowWalk row_walk(int64_t r, int64_t cols) {
  if constexpr (P::form == ROW_RAGGED) {
    const int64_t head = (FE - r * cols % FE) % FE;
    return {head, head + (cols - head) / FE * FE, cols};
  } else if constexpr (P::form == ROW_GROUP) return {0, cols / FE * FE, cols};
  else return {0, cols, cols};
}

// A lane's part of a row: body(first column, what is kept of these elements, Elements<how many>).  Whole vectors are the
// vectors l, l + P::tpr, ... -- P::nv of them, the last one if it lies in the row, when the program keeps vectors from one
// stage to the next (P::nv > 0), any number otherwise.  Where it pays (fused_rtc.hip)
// the trips are written out by recursion: what is kept is indexed by the trip and has to stay in registers.  (As a loop with an
// unroll pragma the compiler leaves 16 light trips rolled and turns the index into chains of selects, 16 of them per element.)
template <typename P, int IT, typename F>
__device__ __forceinline__ void trips_from(int lane, const RowWalk &w, RowVector *kept, F &&body) {
  if constexpr (IT < P::nv) {
    const int64_t k = w.begin + ((int64_t)lane + (int64_t)IT * P::tpr) * FE;
    if constexpr (IT + 1 < P::nv || P::form == ROW_LANE) body(k, kept[IT], Elements<FE>{});
    else if (k < w.end) body(k, kept[IT], Elements<FE>{});
    trips_from<P, IT + 1>(lane, w, kept, body);
  }
}
// `kept`: of the vectors, then of the element in front of them, then of those behind them
template <typename P, typename F>
__device__ __forceinline__ void for_each_vector(int lane, const RowWalk &w, RowVector *kept, F &&body) {
  constexpr int own = P::nv > 0 ? P::nv : 1;
  if constexpr (P::form == ROW_RAGGED)
    if (lane < w.begin) body((int64_t)lane, kept[own], Elements<1>{});
  if constexpr (P::nv > 0 && (P::written_out || P::form == ROW_LANE)) trips_from<P, 0>(lane, w, kept, body);
  else if constexpr (P::nv > 0) {
#pragma unroll
    for (int it = 0; it < P::nv; it++) {
      const int64_t k = w.begin + ((int64_t)lane + (int64_t)it * P::tpr) * FE;
      if (k < w.end) body(k, kept[it], Elements<FE>{});
    }
  } else if constexpr (P::form != ROW_LANE)
    for (int64_t k = w.begin + (int64_t)lane * FE; k < w.end; k += (int64_t)P::tpr * FE) body(k, kept[0], Elements<FE>{});
  if constexpr (P::form == ROW_LANE && P::tail > 0) body((int64_t)P::nv * FE, kept[own + 1], Elements<P::tail>{});
  if constexpr (P::form == ROW_GROUP || P::form == ROW_RAGGED)
    if (w.end + lane < w.cols) body(w.end + lane, kept[own + 1], Elements<1>{});
}

// the reduction of a stage over the P::tpr lanes of a row, left in every lane: within a wave by the
// butterfly, across the waves of a block through LDS in the order of fused_reduce_rows_body
template <typename P, typename R>
__device__ __forceinline__ typename R::acc_t row_reduce(typename R::acc_t acc) {
  acc = wave_reduce<R, (P::tpr < WAVE ? P::tpr : WAVE)>(acc);
  if constexpr (P::tpr > WAVE) {
    __shared__ typename R::acc_t sm[FBLOCK / WAVE];
    __syncthreads();  // the previous stage's readers are done with sm
    if (threadIdx.x % WAVE == 0) sm[threadIdx.x / WAVE] = acc;
    __syncthreads();
    acc = sm[0];
#pragma unroll
    for (int w = 1; w < FBLOCK / WAVE; w++) acc = R::combine(acc, sm[w]);
  }
  return acc;
}

template <typename P, int SEG>
__device__ __forceinline__ void row_stage(KernArgs a, int64_t r, int lane, const RowWalk &walk, RowStats &stats, RowVector *kept) {
  // stage SEG: instructions [begin, red) on the row's elements, the reduction at `red`, instructions
  // (red, save) on the statistic, which is kept at `save`; the last stage is [begin, n_instr)
  constexpr int begin = SEG == 0 ? 0 : P::seg_save[SEG - 1] + 1;
  constexpr int red = P::seg_red[SEG], save = P::seg_save[SEG];
  if constexpr (SEG == P::held_stage) {  // the first stage that reads the held input: all of the lane's part is requested at once
    for_each_vector<P>(lane, walk, kept, [&](int64_t k, RowVector &mine, auto count) __attribute__((always_inline)) {
      constexpr int n = decltype(count)::n;
      const int64_t row[FV] = {r}, col[FV] = {k};
      Vecs x;
      if constexpr (P::held == P::scores) load_scores<P>(a, r, k, n, x);
      else if constexpr (n == FE) load_input_as<P::unal>(a, P::held, P::in_dt[P::held], 1, row, col, x);
      else load_input_tail(a, P::held, P::in_dt[P::held], 1, row, col, n, x);
#pragma unroll
      for (int e = 0; e < n; e++) mine.held[e] = x[0][e];
    });
  }
  if constexpr (red < 0) {  // the last stage: its value is the result
    void *out = (void *)a->out;
    for_each_vector<P>(lane, walk, kept, [&](int64_t k, RowVector &mine, auto count) __attribute__((always_inline)) {
      constexpr int n = decltype(count)::n;
      const int64_t row[FV] = {r}, col[FV] = {k}, at = r * walk.cols + k;
      Vecs x;
      Saved S;
      static_steps<P, begin, P::n_instr>(a, row, col, x, S, stats, n, &mine);
      if constexpr (n < FE) {
#pragma unroll
        for (int e = 0; e < n; e++) {
          if constexpr (result_is_relabelled_bits<P>()) ((uint32_t *)out)[at + e] = __float_as_uint(x[0][e]);
          else store_one<float>(out, P::out_dt, at + e, x[0][e]);
        }
      } else if constexpr (result_is_relabelled_bits<P>()) {
        uint32_t bits[FE];
#pragma unroll
        for (int e = 0; e < FE; e++) bits[e] = __float_as_uint(x[0][e]);
        __builtin_memcpy((uint32_t *)out + at, bits, sizeof(bits));
      } else if constexpr (P::unal) {
        constexpr int bytes = FE * (P::out_dt == HIPNX_F32 ? 4 : P::out_dt == HIPNX_U8 ? 1 : 2);
        raw_vec<bytes> v;
        store_vec<float, FE>(&v, P::out_dt, 0, x[0]);
        __builtin_memcpy((char *)out + at * (bytes / FE), &v, bytes);
      } else {
        store_vec<float, FE>(out, P::out_dt, at, x[0]);
      }
    });
  } else {
    constexpr int op = P::op[red];
    typedef typename std::conditional<op == HIPNX_RED_SUM, double, float>::type CT;
    typedef PlainReducer<CT, op, false> R;
    typename R::acc_t acc = R::init();
    for_each_vector<P>(lane, walk, kept, [&](int64_t k, RowVector &mine, auto count) __attribute__((always_inline)) {
      constexpr int n = decltype(count)::n;
      const int64_t row[FV] = {r}, col[FV] = {k};
      Vecs x;
      Saved S;
      static_steps<P, begin, red>(a, row, col, x, S, stats, n, &mine);
#pragma unroll
      for (int e = 0; e < n; e++) acc = R::accumulate(acc, (CT)x[0][e], k + e);
      if constexpr (P::nv > 0 || P::form == ROW_LANE) {  // kept for the next stage (after this stage's own reads of the previous one's)
#pragma unroll
        for (int e = 0; e < n; e++) mine.carry[e] = x[0][e];
      }
    });
    acc = row_reduce<P, R>(acc);  // the same value in every lane of the row
    // the work on the statistic: the same instructions on a vector that holds it eight times
    const int64_t row[FV] = {r}, col[FV] = {0};
    Vecs x;
    Saved S;
#pragma unroll
    for (int e = 0; e < FE; e++) x[0][e] = as_stored<CT>(acc, P::dt[red]);
    static_steps<P, red + 1, save>(a, row, col, x, S, stats);
    if constexpr ((P::flags[save] & HIPNX_FUSED_FLAG_RESULT) != 0) {  // this one value per row is the result
      if (lane == 0) store_one<float>((void *)a->out, P::out_dt, r, x[0][0]);  // lane 0 of the row
    } else {
      stats[P::arg[save]] = x[0][0];
      row_stage<P, SEG + 1>(a, r, lane, walk, stats, kept);
    }
  }
}

template <typename P>
__device__ __forceinline__ void fused_row_stages_body() {
  static_assert(FV == 1, "one vector per lane and step");
  KernArgs a = (KernArgs)__builtin_amdgcn_kernarg_segment_ptr();
  // P::tpr lanes per row: a part of a wave, a wave (rows of at most 4096 elements) or the whole block, as the separate reduction has it
  const int64_t r = (int64_t)blockIdx.x * (FBLOCK / P::tpr) + threadIdx.x / P::tpr;
  if (r >= a->rows) return;  // (all lanes of a row, or with a block per row nobody: no barrier is left waiting)
  RowStats stats = {};
  RowVector kept[(P::nv > 0 ? P::nv : 1) + 2];  // (indexed by compile-time trip numbers only: registers)
  row_stage<P, 0>(a, r, threadIdx.x % P::tpr, row_walk<P>(r, a->cols), stats, kept);
}

// Stages over the rows of a contraction whose result exists only here (attention probabilities: scores, scaling, softmax).  A block
// takes sixteen rows of l against all rows of r: each wave contracts every fourth tile of sixteen columns with operands
// loaded straight into MFMA registers (no wave shares a row of r, and r is in the L2 for the blocks of the same batch item,
// which follow one another on one XCD), rounds the sums to the contraction's type and leaves them in LDS; then the row
// stages run as they do over a tensor.  P::scores_k: K, in whole steps of 32.
// Bound by the stages' vector instructions and the result's way to memory: bf16 4 x 8 x 512 x 512 from 64-element rows, f32 result,
// 26 us of kernels and 23.8 us a pass in two -> 21.9 us a pass in one; one query against 368 keys 10.2 -> 6.2.
template <int DT>
struct ScoreMma;
typedef float score4 __attribute__((ext_vector_type(4)));
typedef int score_words __attribute__((ext_vector_type(4)));
template <>
struct ScoreMma<HIPNX_BF16> {
  static __device__ __forceinline__ score4 step(score_words a, score_words b, score4 c) {
    typedef __bf16 v8 __attribute__((ext_vector_type(8)));
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(v8, a), __builtin_bit_cast(v8, b), c, 0, 0, 0);
  }
};
template <>
struct ScoreMma<HIPNX_F16> {
  static __device__ __forceinline__ score4 step(score_words a, score_words b, score4 c) {
    typedef _Float16 v8 __attribute__((ext_vector_type(8)));
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(v8, a), __builtin_bit_cast(v8, b), c, 0, 0, 0);
  }
};

template <typename P>
__device__ __forceinline__ void fused_scores_body() {
  KernArgs a = (KernArgs)__builtin_amdgcn_kernarg_segment_ptr();
  typedef score_words __attribute__((aligned(2))) words_any;
  constexpr int STEPS = P::scores_k / 32, TILES = STEPS <= 2 ? 4 : STEPS <= 4 ? 2 : 1;  // column tiles in flight: up to 32 registers of operands
  constexpr int DT = P::in_dt[P::scores];
  const int lane = threadIdx.x % WAVE, wave = threadIdx.x / WAVE;
  const int64_t cols = a->cols, M = a->scores_rows, tiles_m = (M + SCORE_ROWS - 1) / SCORE_ROWS;
  int64_t block = blockIdx.x;
  if (gridDim.x % 8 == 0) block = (int64_t)(blockIdx.x % 8) * (gridDim.x / 8) + blockIdx.x / 8;
  const int64_t item = block / tiles_m, m0 = (block - item * tiles_m) * SCORE_ROWS;
  const int64_t outer = item / a->scores_inner, inner = item - outer * a->scores_inner;
  {
    const uint16_t *l = (const uint16_t *)a->l + outer * a->l_outer + inner * a->l_inner, *r = (const uint16_t *)a->r + outer * a->r_outer + inner * a->r_inner;
    const int64_t m = m0 + lane % 16 < M ? m0 + lane % 16 : M - 1;  // (rows past the edge: any row; they are not used)
    score_words x[STEPS];
#pragma unroll
    for (int s = 0; s < STEPS; s++) x[s] = *reinterpret_cast<const words_any *>(l + m * a->l_ld + s * 32 + lane / 16 * 8);
    uint16_t *row = score_row<P>(lane % 16);
    const int shift = score_shift(item * M + m0 + lane % 16, cols, P::form == ROW_RAGGED);
    const bool whole = cols % 4 == 0;  // four neighbouring columns lie in the row together, eight bytes aligned
    for (int64_t n0 = wave * 16; n0 < cols; n0 += 64 * TILES) {
      score_words y[TILES][STEPS];
#pragma unroll
      for (int t = 0; t < TILES; t++) {
        int64_t n = n0 + t * 64 + lane % 16;
        n = n < cols ? n : cols - 1;
#pragma unroll
        for (int s = 0; s < STEPS; s++) y[t][s] = *reinterpret_cast<const words_any *>(r + n * a->r_ld + s * 32 + lane / 16 * 8);
      }
#pragma unroll
      for (int t = 0; t < TILES; t++) {
        score4 acc = {0, 0, 0, 0};
#pragma unroll
        for (int s = 0; s < STEPS; s++) acc = ScoreMma<DT>::step(y[t][s], x[s], acc);
        const int64_t n = n0 + t * 64 + lane / 16 * 4;  // a lane has four columns of row lane % 16
        uint16_t h[4];
#pragma unroll
        for (int e = 0; e < 4; e++) h[e] = DT == HIPNX_BF16 ? conv<float>::to_bf16(acc[e]) : conv<float>::to_f16(acc[e]);
        if (whole) {
          if (n < cols) *reinterpret_cast<uint2 *>(row + n + shift) = make_uint2(h[0] | (uint32_t)h[1] << 16, h[2] | (uint32_t)h[3] << 16);
        } else {
#pragma unroll
          for (int e = 0; e < 4; e++)
            if (n + e < cols) row[n + e + shift] = h[e];
        }
      }
    }
  }
  __syncthreads();
  for (int i = threadIdx.x / P::tpr; i < SCORE_ROWS && m0 + i < M; i += FBLOCK / P::tpr) {  // (a row's lanes go on or stop together)
    const int64_t r = item * M + m0 + i;
    RowStats stats = {};
    RowVector kept[(P::nv > 0 ? P::nv : 1) + 2];
    row_stage<P, 0>(a, r, threadIdx.x % P::tpr, row_walk<P>(r, cols), stats, kept);
  }
}

}  // namespace hipnx
