// Nx.dot as a dense batched contraction  out[b, m, n] = sum_k l[b, m, k] * r[b, n, k]:
// argument checks and the choice of kernel.
//
//   bf16 / f16 / f32 operand pairs (f32 accumulation) and s8 pairs (exact s32 accumulation):
//     the MFMA kernels (gemm_mfma.cuh, gemm_pingpong.cuh), which take both operand layouts and any K directly
//       (a partial slab of K is walked with zeros behind its end; rows and k-rows need not be whole 16-byte pieces).  What
//       is shorter than a piece is first copied, and K-inner rows on no dword that many tiles re-read (rows_worth_copying).
//   everything else (f64 whose K is not whole slabs, wide integers, mixed operand types, fewer than 256 outputs, and below
//     16 M multiply-adds a float K that is not whole 16-byte pieces, in every layout): dot_generic_kernel,
//     a plain tiled kernel accumulating in f64 or wrapping 64-bit integers, K cut into segments where few outputs would leave
//     the chip idle; dot_blocked_kernel for many outputs, dot_reduce_kernel for a handful, dot_small_batched_kernel for many small matrices.
//
// Algorithmic work: 2*B*M*N*K flop; minimum traffic bytes(l) + bytes(r) + bytes(out).
#include <type_traits>

#include <algorithm>
#include <cstdlib>

#include "gemm_launch.cuh"

namespace hipnx {

// Rows of K elements copied to a pitch of whole 16-byte pieces, zeros behind K: K-inner rows shorter than a piece, which the
// contraction kernels cannot take, and longer ones on no dword that many tiles re-read (rows_worth_copying).  A lane writes one
// piece; a piece inside its row is one load at whatever address it has, the row's last one is put together by elements.
// Bound by memory: reads and writes the operand once ([2000, 999] bf16, 8 MB moved: 3 us).
template <typename T>
__global__ void __launch_bounds__(256)
pad_rows_kernel(const T *__restrict__ in, unsigned char *__restrict__ out, int64_t rows, int64_t K, int pieces) {
  typedef v4i __attribute__((aligned(1))) v4i_any;
  constexpr int PER = 16 / sizeof(T);
  const int64_t total = rows * pieces;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < total; i += (int64_t)gridDim.x * 256) {
    const int64_t row = i / pieces;
    const int64_t k = (i - row * pieces) * PER;
    const T *src = in + row * K + k;
    v4i v = {0, 0, 0, 0};
    if (k + PER <= K) v = *reinterpret_cast<const v4i_any *>(src);
    else {
      T e[PER];
#pragma unroll
      for (int j = 0; j < PER; j++) e[j] = k + j < K ? src[j] : (T)0;
      __builtin_memcpy(&v, e, 16);
    }
    *reinterpret_cast<v4i *>(out + i * 16) = v;
  }
}

// Plain tiled contraction for every other type combination.  16 x 16 outputs per block, K
// walked in slabs of TK (64; 16 for a short K) through LDS; operands are decoded to CT (double or wrapping int64).
// lk / rk: 1 when the operand is K-inner ([rows, K]), 0 when K-outer ([K, rows]).
// LDT / RDT: the operands' types where they are known when the kernel is compiled (the four loads per operand and slab then
// all go out before one is converted), -1: read from ldt / rdt.
// Bound by the latency of a slab (about 1 us, mostly its loads), K / 64 of them in a row: few outputs over a long K leave the chip
// idle.  nseg > 1: the blocks along y are cut into segments of K of seg_len (whole slabs), whose sums go to
// partial[output * nseg + segment] for dot_reduce_finish_kernel.  In slabs of 16 and with K whole, before / now, us per call:
// f32 80 x 3 x 6377 394 / 20, 100 x 10 x 2001 118 / 12, 64 x 64 x 4095 264 / 15.5, bf16 5 x 300 x 9999 604 / 33.
template <typename CT, int TK, int LDT = -1, int RDT = -1>
__global__ void __launch_bounds__(256)
dot_generic_kernel(const void *__restrict__ l, const void *__restrict__ r, void *__restrict__ out, int ldt_, int rdt_,
                   int odt, int64_t M, int64_t N, int64_t K, int lk, int rk, CT *__restrict__ partial, int64_t seg_len, int nseg) {
  constexpr int T = 16, PER = T * TK / 256;
  const int ldt = LDT >= 0 ? LDT : ldt_, rdt = RDT >= 0 ? RDT : rdt_;
  __shared__ CT sA[T][TK + 1], sB[T][TK + 1];
  const int tid = threadIdx.x, tx = tid % T, ty = tid / T;
  // (tiles of M along x, which holds 2^31 - 1 groups: [2M, 3] . [3, 3] has 131072 of them; tiles of N along y)
  const int64_t b = blockIdx.z;
  const int seg = (int)(blockIdx.y % nseg);
  const int64_t m0 = (int64_t)blockIdx.x * T, n0 = (int64_t)(blockIdx.y / nseg) * T, m = m0 + ty, n = n0 + tx;
  const int64_t lbase = b * M * K, rbase = b * N * K;
  const int64_t k_begin = seg * seg_len, k_end = k_begin + seg_len < K ? k_begin + seg_len : K;
  CT acc = 0, a[PER], c[PER];
  auto request = [&](int64_t k0) {
#pragma unroll
    for (int q = 0; q < PER; q++) {
      // consecutive lanes along the operand's contiguous axis
      const int e = tid + q * 256;
      const int am = lk ? e / TK : e % T, ak = lk ? e % TK : e / T, bn = rk ? e / TK : e % T, bk = rk ? e % TK : e / T;
      const int64_t mm = m0 + am, nn = n0 + bn, ka = k0 + ak, kb = k0 + bk;
      a[q] = (mm < M && ka < k_end) ? load_one<CT>(l, ldt, lbase + (lk ? mm * K + ka : ka * M + mm)) : (CT)0;
      c[q] = (nn < N && kb < k_end) ? load_one<CT>(r, rdt, rbase + (rk ? nn * K + kb : kb * N + nn)) : (CT)0;
    }
  };
  request(k_begin);
  for (int64_t k0 = k_begin; k0 < k_end; k0 += TK) {
#pragma unroll
    for (int q = 0; q < PER; q++) {
      const int e = tid + q * 256;
      const int am = lk ? e / TK : e % T, ak = lk ? e % TK : e / T, bn = rk ? e / TK : e % T, bk = rk ? e % TK : e / T;
      sA[am][ak] = a[q];
      sB[bn][bk] = c[q];
    }
    __syncthreads();
    if (k0 + TK < k_end) request(k0 + TK);  // under this slab's arithmetic
    const int steps = k_end - k0 < TK ? (int)(k_end - k0) : TK;
    for (int k16 = 0; k16 < steps; k16 += 16) {  // (behind K both are zero)
#pragma unroll
      for (int kk = k16; kk < k16 + 16; kk++) {
        // (products of two f32 numbers or narrower ones are exact in f64: one rounding either way)
        if constexpr (std::is_same<CT, double>::value && LDT >= 0 && LDT != HIPNX_F64 && RDT >= 0 && RDT != HIPNX_F64) acc = __builtin_fma(sA[ty][kk], sB[tx][kk], acc);
        else if constexpr (std::is_same<CT, double>::value) acc = sA[ty][kk] * sB[tx][kk] + acc;
        else acc = (int64_t)((uint64_t)sA[ty][kk] * (uint64_t)sB[tx][kk] + (uint64_t)acc);
      }
    }
    __syncthreads();
  }
  if (m < M && n < N) {
    const int64_t o = b * M * N + m * N + n;
    if (nseg > 1) partial[o * nseg + seg] = acc;
    else store_one<CT>(out, odt, o, acc);
  }
}

// Many small matrices (a 3 x 3 transform per point, a 4 x 4 block per item): one lane per output over the whole batch,
// walking k in order -- the tiled kernel above spends a work-group of 256 lanes on each item's nine outputs.
template <typename CT>
__global__ void __launch_bounds__(256)
dot_small_batched_kernel(const void *__restrict__ l, const void *__restrict__ r, void *__restrict__ out, int ldt, int rdt,
                         int odt, int64_t batch, int M, int N, int K, int lk, int rk) {
  const int64_t total = batch * M * N;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < total; i += (int64_t)gridDim.x * 256) {
    const int64_t b = i / (M * N);
    const int mn = (int)(i - b * (M * N)), m = mn / N, n = mn - m * N;
    const int64_t lbase = b * M * K, rbase = b * N * K;
    CT acc = 0;
    for (int k = 0; k < K; k++) {
      const CT x = load_one<CT>(l, ldt, lbase + (lk ? m * K + k : k * M + m)), y = load_one<CT>(r, rdt, rbase + (rk ? n * K + k : k * N + n));
      if constexpr (std::is_same<CT, double>::value) acc = x * y + acc;
      else acc = (int64_t)((uint64_t)x * (uint64_t)y + (uint64_t)acc);
    }
    store_one<CT>(out, odt, i, acc);
  }
}

// The same contraction on 64 x 64 tiles with 4 x 4 outputs per lane: eight LDS reads per sixteen multiply-adds
// instead of two per one, each output still accumulated over k in order (the same bits as the kernel above).
// f64 / s32 / mixed-type 4096^3: 8.4 TFLOP/s there.
template <typename CT>
__global__ void __launch_bounds__(256)
dot_blocked_kernel(const void *__restrict__ l, const void *__restrict__ r, void *__restrict__ out, int ldt, int rdt,
                   int odt, int64_t M, int64_t N, int64_t K, int lk, int rk) {
  constexpr int TM = 64, TN = 64, TK = 16;
  __shared__ CT sA[TK][TM + 4], sB[TK][TN + 4];
  const int tid = threadIdx.x, tx = tid % 16, ty = tid / 16;
  const int64_t b = blockIdx.z, m0 = (int64_t)blockIdx.x * TM, n0 = (int64_t)blockIdx.y * TN;
  const int64_t lbase = b * M * K, rbase = b * N * K;
  CT acc[4][4];
#pragma unroll
  for (int i = 0; i < 4; i++)
#pragma unroll
    for (int j = 0; j < 4; j++) acc[i][j] = 0;
  for (int64_t k0 = 0; k0 < K; k0 += TK) {
#pragma unroll
    for (int q = 0; q < TM * TK / 256; q++) {
      const int e = tid + q * 256;
      // consecutive lanes along the operand's contiguous axis
      const int am = lk ? e / TK : e % TM, ak = lk ? e % TK : e / TM;
      const int bn = rk ? e / TK : e % TN, bk = rk ? e % TK : e / TN;
      const int64_t mm = m0 + am, nn = n0 + bn, ka = k0 + ak, kb = k0 + bk;
      sA[ak][am] = (mm < M && ka < K) ? load_one<CT>(l, ldt, lbase + (lk ? mm * K + ka : ka * M + mm)) : (CT)0;
      sB[bk][bn] = (nn < N && kb < K) ? load_one<CT>(r, rdt, rbase + (rk ? nn * K + kb : kb * N + nn)) : (CT)0;
    }
    __syncthreads();
#pragma unroll
    for (int kk = 0; kk < TK; kk++) {
      CT a[4], c[4];
#pragma unroll
      for (int i = 0; i < 4; i++) a[i] = sA[kk][ty * 4 + i];
#pragma unroll
      for (int j = 0; j < 4; j++) c[j] = sB[kk][tx * 4 + j];
#pragma unroll
      for (int i = 0; i < 4; i++)
#pragma unroll
        for (int j = 0; j < 4; j++) {
          if constexpr (std::is_same<CT, double>::value) acc[i][j] = a[i] * c[j] + acc[i][j];
          else acc[i][j] = (int64_t)((uint64_t)a[i] * (uint64_t)c[j] + (uint64_t)acc[i][j]);
        }
    }
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < 4; i++)
#pragma unroll
    for (int j = 0; j < 4; j++) {
      const int64_t m = m0 + ty * 4 + i, n = n0 + tx * 4 + j;
      if (m < M && n < N) store_one<CT>(out, odt, b * M * N + m * N + n, acc[i][j]);
    }
}

// A handful of outputs over a long contraction (the dot of two vectors, a [16, K] . [K, 16] Gram block): a work-group per
// output and segment of K, lanes along k, partial sums in f64 (wrapping 64-bit integers), then one small pass that adds
// an output's segments in order and encodes it.  The tiled kernels give such a problem one tile -- one work-group,
// or below 256 outputs one lane of the kernel above walking all of K (4M-element vectors: 0.26 s).
// l element (m, k) = l[m * l_sm + k * l_sk], r element (n, k) = r[n * r_sn + k * r_sk].
template <typename CT>
__global__ void __launch_bounds__(256)
dot_reduce_kernel(const void *__restrict__ l, const void *__restrict__ r, CT *__restrict__ partial, void *__restrict__ out, int ldt,
                  int rdt, int odt, int64_t M, int64_t N, int64_t K, int64_t l_sm, int64_t l_sk, int64_t r_sn, int64_t r_sk,
                  int64_t seg_len, int nseg, int vec) {
  constexpr int V = 8;
  const int64_t mn = blockIdx.y, b = blockIdx.z, m = mn / N, n = mn - m * N;
  const int seg = blockIdx.x;
  const int64_t k0 = (int64_t)seg * seg_len, k1 = k0 + seg_len < K ? k0 + seg_len : K;
  const int64_t lb = b * M * K + m * l_sm, rb = b * N * K + n * r_sn;
  CT acc = 0;
  auto mac = [&](CT x, CT y) {
    if constexpr (std::is_same<CT, double>::value) acc = x * y + acc;
    else acc = (int64_t)((uint64_t)x * (uint64_t)y + (uint64_t)acc);
  };
  if (vec) {  // both operands contiguous along k, every row and segment on a vector boundary
    for (int64_t k = k0 + (int64_t)threadIdx.x * V; k < k1; k += 256 * V) {
      CT x[V], y[V];
      load_vec<CT, V>(l, ldt, lb + k, x);
      load_vec<CT, V>(r, rdt, rb + k, y);
#pragma unroll
      for (int i = 0; i < V; i++) mac(x[i], y[i]);
    }
  } else {
    for (int64_t k = k0 + threadIdx.x; k < k1; k += 256) mac(load_one<CT>(l, ldt, lb + k * l_sk), load_one<CT>(r, rdt, rb + k * r_sk));
  }
  __shared__ CT sm[256];
  sm[threadIdx.x] = acc;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) {
      if constexpr (std::is_same<CT, double>::value) sm[threadIdx.x] = sm[threadIdx.x] + sm[threadIdx.x + w];
      else sm[threadIdx.x] = (int64_t)((uint64_t)sm[threadIdx.x] + (uint64_t)sm[threadIdx.x + w]);
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    if (nseg == 1) store_one<CT>(out, odt, b * M * N + mn, sm[0]);
    else partial[(b * M * N + mn) * nseg + seg] = sm[0];
  }
}

template <typename CT>
__global__ void __launch_bounds__(256)
dot_reduce_finish_kernel(const CT *__restrict__ partial, void *__restrict__ out, int odt, int64_t outputs, int nseg) {
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < outputs; i += (int64_t)gridDim.x * 256) {
    CT acc = partial[i * nseg];
    for (int s = 1; s < nseg; s++) {
      if constexpr (std::is_same<CT, double>::value) acc = acc + partial[i * nseg + s];
      else acc = (int64_t)((uint64_t)acc + (uint64_t)partial[i * nseg + s]);
    }
    store_one<CT>(out, odt, i, acc);
  }
}

}  // namespace hipnx

using namespace hipnx;

// defined in move.hip
extern "C" int hipnx_transpose(hipnx_ctx *ctx, int elem_bytes, int rank, const int64_t *in_dims, const int *perm,
                               const hipnx_buf *inb, hipnx_buf *out);

// Second pass of a contraction whose K was split over S work-groups per tile: out[i] = the S partial
// results of element i added in split order (f32 adds for the float types, wrapping 32-bit adds -- exact --
// for int8), then encoded once.
// SCALED: an int8 contraction's sums as f32 numbers times their scale, each step rounding once (gemm_epilogue).
template <typename AT, bool SCALED = false>
__global__ void __launch_bounds__(256)
splitk_combine_kernel(const AT *__restrict__ part, void *__restrict__ out, int odt, int64_t mn, int splits, int N = 0,
                      const float *__restrict__ scale = nullptr, int scale_mode = 0) {
  typedef typename std::conditional<std::is_same<AT, float>::value, float, int64_t>::type CT;
  auto scaled = [&](AT sum, int64_t i) -> float {
    const int64_t at = scale_mode == HIPNX_SCALE_ONE ? 0 : scale_mode == HIPNX_SCALE_PER_ROW ? i / N : i % N;
    return (float)sum * scale[at];
  };
  const int64_t nvec = mn / 4;
  for (int64_t v = (int64_t)blockIdx.x * 256 + threadIdx.x; v < nvec; v += (int64_t)gridDim.x * 256) {
    typedef __attribute__((ext_vector_type(4), aligned(4))) AT vec_t;
    vec_t acc = *reinterpret_cast<const vec_t *>(part + v * 4);
    // up to sixteen loads in flight, as many as there are ranges left, added in order of the ranges: what the pass waits for is round trips
    // (us per call with four in flight / so: f16 30 x 1000 x 8000 9.5 / 9.0, int8 8 x 500 x 4000 7.9 / 7.3, bf16 1 x 4096 x 11008 20.5 / 19.9, the pass alone, f32 512 x 10 in 64 ranges, 7.2 / 5.3)
    int s = 1;
    auto add = [&](auto count) {
      constexpr int B = decltype(count)::value;
      vec_t p[B];
#pragma unroll
      for (int u = 0; u < B; u++) p[u] = *reinterpret_cast<const vec_t *>(part + (int64_t)(s + u) * mn + v * 4);
#pragma unroll
      for (int u = 0; u < B; u++)
#pragma unroll
        for (int e = 0; e < 4; e++) acc[e] += p[u][e];
      s += B;
    };
    while (s + 16 <= splits) add(std::integral_constant<int, 16>{});
    if (s + 8 <= splits) add(std::integral_constant<int, 8>{});
    switch (splits - s) {
#define HIPNX_LEFT(N) case N: add(std::integral_constant<int, N>{}); break;
      HIPNX_LEFT(1) HIPNX_LEFT(2) HIPNX_LEFT(3) HIPNX_LEFT(4) HIPNX_LEFT(5) HIPNX_LEFT(6) HIPNX_LEFT(7)
#undef HIPNX_LEFT
    }
    if constexpr (SCALED) {
      float x[4];
#pragma unroll
      for (int e = 0; e < 4; e++) x[e] = scaled(acc[e], v * 4 + e);
      store_vec<float, 4>(out, HIPNX_F32, v * 4, x);
    } else {
      CT x[4];
#pragma unroll
      for (int e = 0; e < 4; e++) x[e] = (CT)acc[e];
      store_vec<CT, 4>(out, odt, v * 4, x);
    }
  }
  if (blockIdx.x == 0 && threadIdx.x < mn % 4) {
    const int64_t i = nvec * 4 + threadIdx.x;
    AT acc = part[i];
    for (int s = 1; s < splits; s++) acc += part[s * mn + i];
    if constexpr (SCALED) store_one<float>(out, HIPNX_F32, i, scaled(acc, i));
    else store_one<CT>(out, odt, i, (CT)acc);
  }
}

// A K-inner operand ([rows, K]) copied to rows of whole 16-byte pieces.
static int pad_rows(hipnx_ctx *ctx, int esz, int64_t rows, int64_t K, const hipnx_buf *in, hipnx_buf **out) {
  const int64_t pieces = (K * esz + 15) / 16;
  if (int st = hipnx_buf_alloc(ctx, (size_t)(rows * pieces * 16), out)) return st;
  Enter e(ctx);
  if (e.status) return e.status;
  if (int st = check_buf(ctx, in, (uint64_t)rows * K * esz, "dot operand")) return st;  // (the lock was dropped for the allocation)
  const dim3 grid((unsigned)std::min<int64_t>((rows * pieces + 255) / 256, 1 << 20)), block(256);
  switch (esz) {
    case 1: hipLaunchKernelGGL((pad_rows_kernel<uint8_t>), grid, block, 0, ctx->stream, (const uint8_t *)in->ptr, (unsigned char *)(*out)->ptr, rows, K, (int)pieces); break;
    case 2: hipLaunchKernelGGL((pad_rows_kernel<uint16_t>), grid, block, 0, ctx->stream, (const uint16_t *)in->ptr, (unsigned char *)(*out)->ptr, rows, K, (int)pieces); break;
    default: hipLaunchKernelGGL((pad_rows_kernel<uint32_t>), grid, block, 0, ctx->stream, (const uint32_t *)in->ptr, (unsigned char *)(*out)->ptr, rows, K, (int)pieces); break;
  }
  HIPNX_HIP(hipGetLastError());
  return HIPNX_OK;
}

// Operands contracted where they lie in a larger tensor, in bytes: from row to row (K-inner) or from k to k (K-outer), and from item
// to item along the two axes of the batch; `inner` items along the second.
struct DotView {
  int64_t inner, ld_l, bs_l, ts_l, ld_r, bs_r, ts_r;
};

// scale_mode != NONE: the scaled form (out_dt is then f32 over an s32 sum)
// view: strided operands, whose extents the caller has checked; only what the MFMA kernels take as it lies (otherwise HIPNX_EUNSUPPORTED,
// and nothing has been launched)
static int dot_impl(hipnx_ctx *ctx, int l_dt, int r_dt, int out_dt, int64_t batch, int64_t M, int64_t N,
                    int64_t K, int l_layout, int r_layout, const hipnx_buf *l, const hipnx_buf *r,
                    hipnx_buf *out, int scale_mode, const hipnx_buf *scale, const DotView *view = nullptr, bool any_k = false) {
  if (batch > 0 && M > 0 && N > 0 && K > 0) {  // (the products below are 64 bits wide)
    const __int128 most = INT64_MAX / 8;
    if ((__int128)M * N > most / batch || (__int128)M * K > most / batch || (__int128)N * K > most / batch)
      return set_error(HIPNX_EINVAL, "dot: extents beyond any buffer");
  }
  if (view && batch > 65535) return set_error(HIPNX_EUNSUPPORTED, "dot_strided: more than 65535 batch items");
  // More batch items than a grid's second dimension holds (100000 small matrices): runs of 65535 items, each over
  // borrowed handles on its part of the three buffers.
  if (batch > 65535 && M > 0 && N > 0 && l && r && out && dtype_size(l_dt) > 0 && dtype_size(r_dt) > 0 && out_dtype_size(out_dt) > 0 && K >= 0) {
    {
      Enter in(ctx);
      if (in.status) return in.status;
      if (int st = check_buf(ctx, l, (uint64_t)batch * M * K * dtype_size(l_dt), "dot lhs")) return st;
      if (int st = check_buf(ctx, r, (uint64_t)batch * N * K * dtype_size(r_dt), "dot rhs")) return st;
      if (int st = check_buf(ctx, out, (uint64_t)batch * M * N * out_dtype_size(out_dt), "dot out")) return st;
    }
    const size_t lb = (size_t)(M * K) * dtype_size(l_dt), rb = (size_t)(N * K) * dtype_size(r_dt), ob = (size_t)(M * N) * out_dtype_size(out_dt);
    for (int64_t b0 = 0; b0 < batch; b0 += 65535) {
      const int64_t nb = batch - b0 < 65535 ? batch - b0 : 65535;
      hipnx_buf *lw = nullptr, *rw = nullptr, *ow = nullptr;
      int st = hipnx_buf_wrap(ctx, (char *)l->ptr + b0 * lb, nb * lb > 0 ? nb * lb : 1, &lw);
      if (!st) st = hipnx_buf_wrap(ctx, (char *)r->ptr + b0 * rb, nb * rb > 0 ? nb * rb : 1, &rw);
      if (!st) st = hipnx_buf_wrap(ctx, (char *)out->ptr + b0 * ob, nb * ob, &ow);
      if (!st) st = dot_impl(ctx, l_dt, r_dt, out_dt, nb, M, N, K, l_layout, r_layout, lw, rw, ow, scale_mode, scale, nullptr, any_k);
      if (lw) hipnx_buf_destroy(lw);
      if (rw) hipnx_buf_destroy(rw);
      if (ow) hipnx_buf_destroy(ow);
      if (st) return st;
    }
    return HIPNX_OK;
  }
  bool mfma = false, l_pad = false, r_pad = false;
  const bool partials = l_dt == HIPNX_S8 ? scale_mode != HIPNX_SCALE_NONE || !is_float(out_dt) : l_dt != HIPNX_F64;  // (a split's sums are f32 / s32)
  // the MFMA kernels transpose K-outer operands themselves, k-rows that are not whole pieces too (not f64: its last slab would
  // have to be walked first, and it adds over k in order), but for k-rows shorter than one
  const int row_block = dtype_size(l_dt) == 1 ? 16 : dtype_size(l_dt) == 2 ? 8 : dtype_size(l_dt) == 4 ? 4 : 2;
  const bool l_ragged = l_layout == HIPNX_K_OUTER && M % row_block != 0, r_ragged = r_layout == HIPNX_K_OUTER && N % row_block != 0;
  const bool l_relay = l_ragged && (M < row_block || l_dt == HIPNX_F64);
  const bool r_relay = r_ragged && (N < row_block || l_dt == HIPNX_F64);
  {
    Enter in(ctx);
    if (in.status) return in.status;
    if (dtype_size(l_dt) < 0 || dtype_size(r_dt) < 0 || out_dtype_size(out_dt) < 0)
      return set_error(HIPNX_EINVAL, "dot: unknown element type");
    if (batch < 0 || M < 0 || N < 0 || K < 0) return set_error(HIPNX_EINVAL, "dot: negative extent");
    if ((l_layout != HIPNX_K_INNER && l_layout != HIPNX_K_OUTER) || (r_layout != HIPNX_K_INNER && r_layout != HIPNX_K_OUTER))
      return set_error(HIPNX_EINVAL, "dot: unknown operand layout");
    if (int st = check_buf(ctx, l, (uint64_t)batch * M * K * dtype_size(l_dt), "dot lhs")) return st;
    if (int st = check_buf(ctx, r, (uint64_t)batch * N * K * dtype_size(r_dt), "dot rhs")) return st;
    if (int st = check_buf(ctx, out, (uint64_t)batch * M * N * out_dtype_size(out_dt), "dot out")) return st;
    if (batch * M * N == 0) return HIPNX_OK;
    if (view && (l_ragged || r_ragged || K * dtype_size(l_dt) % 16 != 0))
      return set_error(HIPNX_EUNSUPPORTED, "dot_strided: operands that the kernels cannot take as they lie");
    if (batch > 65535) return set_error(HIPNX_EUNSUPPORTED, "dot: more than 65535 batch items");

    const bool float_pair = l_dt == r_dt && (l_dt == HIPNX_BF16 || l_dt == HIPNX_F16 || l_dt == HIPNX_F32 || l_dt == HIPNX_F64) && is_float(out_dt);
    const bool scaled = scale_mode != HIPNX_SCALE_NONE;
    const bool int8_pair = l_dt == HIPNX_S8 && r_dt == HIPNX_S8 && (scaled || !is_float(out_dt)) && K <= (1ll << 16);
    const int64_t row_bytes = K * dtype_size(l_dt);
    mfma = (float_pair || int8_pair) && K > 0 && M * N >= 256;
    if (mfma && l_dt == HIPNX_F64) mfma = row_bytes % SLAB == 0;  // (f64 otherwise adds over k in order, on the plain kernels)
    else if (mfma && row_bytes % 16 != 0) {
      // rows that are not whole pieces: below 16 M multiply-adds floats are summed in f64 on the plain kernels, whatever the
      // layout; int8 is exact on either.  Rows shorter than a piece are copied to one.
      l_pad = row_bytes < 16 && (l_layout == HIPNX_K_INNER || l_relay);
      r_pad = row_bytes < 16 && (r_layout == HIPNX_K_INNER || r_relay);
      if (l_pad || r_pad || l_dt != HIPNX_S8) mfma = (double)M * (double)N * (double)K * (double)batch >= 16777216.0;
      if (mfma && row_bytes >= 16) {
        const GemmChoice choice = gemm_choice(ctx->num_cus, l_dt, batch, M, N, K, l_layout == HIPNX_K_INNER || l_relay, r_layout == HIPNX_K_INNER || r_relay, partials);
        l_pad = l_layout == HIPNX_K_INNER && !l_relay && rows_worth_copying(ctx->num_cus, choice, batch, M, N, row_bytes, false);
        r_pad = r_layout == HIPNX_K_INNER && !r_relay && rows_worth_copying(ctx->num_cus, choice, batch, M, N, row_bytes, true);
      }
    }
    if (scaled) {
      // (below 16 M multiply-adds callers of a K off whole pieces make the conversion and the product calls of their own)
      if (any_k && row_bytes % 16 != 0 && (l_layout == HIPNX_K_INNER || r_layout == HIPNX_K_INNER || l_ragged || r_ragged) && (double)M * (double)N * (double)K * (double)batch < 16777216.0)
        return set_error(HIPNX_EUNSUPPORTED, "dot_scaled: a K off whole 16-byte pieces from 16 M multiply-adds on");
      if (!(int8_pair && mfma && (any_k || row_bytes % SLAB == 0))) return set_error(HIPNX_EUNSUPPORTED, "dot_scaled: s8 x s8 with K a multiple of 128 and at most 65536, M * N >= 256");
      if (scale_mode == HIPNX_SCALE_PER_ROW && batch != 1) return set_error(HIPNX_EUNSUPPORTED, "dot_scaled: a scale per row with more than one batch item");
      const int64_t need = scale_mode == HIPNX_SCALE_PER_COLUMN ? N : scale_mode == HIPNX_SCALE_PER_ROW ? M : 1;
      if (int st = check_buf(ctx, scale, (uint64_t)need * 4, "dot_scaled scale")) return st;
    }

    // at most 32 x 32 outputs over a contraction of 4096 elements or more: the reduction kernels
    // (also a matrix against one to four vectors in f32 or wider types, where the matrix is contiguous along k: an MFMA
    // tile would be all but empty, and its f32 work costs more than the bytes -- [1, 8192] . [8192, 8192]^T 105 us)
    const bool few_vectors = dtype_size(l_dt) >= 4 && dtype_size(r_dt) >= 4 && K >= 1024 &&
                             ((M <= 4 && r_layout == HIPNX_K_INNER) || (N <= 4 && l_layout == HIPNX_K_INNER));
    const bool few_outputs = !scaled && ((M <= 32 && N <= 32 && (K >= 4096 || (M * N <= 4 && K >= 128))) || few_vectors) && M * N <= 65535 && batch * M * N <= 65535 && !(!is_float(l_dt) && !is_float(r_dt) && is_float(out_dt));
    if (view && few_outputs) return set_error(HIPNX_EUNSUPPORTED, "dot_strided: a contraction whose sums are not for the matrix cores");
    if (few_outputs) {
      const bool any_float = is_float(l_dt) || is_float(r_dt);
      const int lk = l_layout == HIPNX_K_INNER, rk = r_layout == HIPNX_K_INNER;
      const int64_t l_sm = lk ? K : 1, l_sk = lk ? 1 : M, r_sn = rk ? K : 1, r_sk = rk ? 1 : N;
      const int64_t outputs = batch * M * N;
      int64_t nseg = (2 * (int64_t)ctx->num_cus + outputs - 1) / outputs;
      if (nseg > K / 2048) nseg = K / 2048;
      if (nseg > 1024) nseg = 1024;
      if (nseg < 1) nseg = 1;
      int64_t seg_len = ((K + nseg - 1) / nseg + 7) / 8 * 8;
      nseg = (K + seg_len - 1) / seg_len;
      const int vec = l_sk == 1 && r_sk == 1 && K % 8 == 0 && ((uintptr_t)l->ptr % 32 == 0) && ((uintptr_t)r->ptr % 32 == 0);
      void *ws = nullptr;
      size_t ws_cap = 0;
      if (nseg > 1)
        if (int st = pool_alloc(ctx, (size_t)(outputs * nseg) * 8, &ws, &ws_cap)) return st;
      dim3 grid((unsigned)nseg, (unsigned)(M * N), (unsigned)batch), block(256);
      if (any_float) {
        hipLaunchKernelGGL((dot_reduce_kernel<double>), grid, block, 0, ctx->stream, l->ptr, r->ptr, (double *)ws, out->ptr, l_dt, r_dt, out_dt, M, N, K,
                           l_sm, l_sk, r_sn, r_sk, seg_len, (int)nseg, vec);
        if (nseg > 1)
          hipLaunchKernelGGL((dot_reduce_finish_kernel<double>), dim3((unsigned)((outputs + 255) / 256)), block, 0, ctx->stream, (const double *)ws,
                             out->ptr, out_dt, outputs, (int)nseg);
      } else {
        hipLaunchKernelGGL((dot_reduce_kernel<int64_t>), grid, block, 0, ctx->stream, l->ptr, r->ptr, (int64_t *)ws, out->ptr, l_dt, r_dt, out_dt, M, N, K,
                           l_sm, l_sk, r_sn, r_sk, seg_len, (int)nseg, vec);
        if (nseg > 1)
          hipLaunchKernelGGL((dot_reduce_finish_kernel<int64_t>), dim3((unsigned)((outputs + 255) / 256)), block, 0, ctx->stream, (const int64_t *)ws,
                             out->ptr, out_dt, outputs, (int)nseg);
      }
      if (ws) pool_free(ctx, ws, ws_cap);  // later work is ordered on the same stream
      HIPNX_HIP(hipGetLastError());
      return HIPNX_OK;
    }

    // many small matrices (up to 64 outputs, K up to 64): a lane per output over the whole batch (16 x 16 x 16 items are
    // faster on the tiled kernels: 51 us against 175 us for 8192 of them)
    if (!scaled && !view && M * N <= 64 && K <= 64 && batch >= 64 && !(!is_float(l_dt) && !is_float(r_dt) && is_float(out_dt))) {
      const bool any_float = is_float(l_dt) || is_float(r_dt);
      const int lk = l_layout == HIPNX_K_INNER, rk = r_layout == HIPNX_K_INNER;
      const int64_t blocks = (batch * M * N + 255) / 256;
      dim3 gs((unsigned)(blocks < (1ll << 24) - 1 ? blocks : (1ll << 24) - 1)), block(256);
      if (any_float)
        hipLaunchKernelGGL((dot_small_batched_kernel<double>), gs, block, 0, ctx->stream, l->ptr, r->ptr, out->ptr, l_dt, r_dt, out_dt, batch, (int)M, (int)N, (int)K, lk, rk);
      else
        hipLaunchKernelGGL((dot_small_batched_kernel<int64_t>), gs, block, 0, ctx->stream, l->ptr, r->ptr, out->ptr, l_dt, r_dt, out_dt, batch, (int)M, (int)N, (int)K, lk, rk);
      HIPNX_HIP(hipGetLastError());
      return HIPNX_OK;
    }

    if (view && !mfma) return set_error(HIPNX_EUNSUPPORTED, "dot_strided: a contraction that is not for the matrix cores");
    if (!mfma) {
      const bool any_float = is_float(l_dt) || is_float(r_dt);
      if (!any_float && is_float(out_dt)) return set_error(HIPNX_EUNSUPPORTED, "dot: integer operands with a float output");
      dim3 grid((unsigned)((M + 15) / 16), (unsigned)((N + 15) / 16), (unsigned)batch), block(256);
      if ((N + 15) / 16 > 65535 || (M + 15) / 16 >= (1ll << 31) / 256)
        return set_error(HIPNX_EUNSUPPORTED, "dot: more than a million columns (or 134 million rows) on the plain kernel");
      const int lk = l_layout == HIPNX_K_INNER, rk = r_layout == HIPNX_K_INNER;
      // tiles of 64 x 64, sixteen outputs per lane, where they still give every CU two work-groups (512^3: 64 tiles, 143 us
      // against 53 us on 16 x 16 tiles)
      if (M >= 64 && N >= 64 && (N + 63) / 64 <= 65535 && ((M + 63) / 64) * ((N + 63) / 64) * batch >= 2 * (int64_t)ctx->num_cus) {
        dim3 g64((unsigned)((M + 63) / 64), (unsigned)((N + 63) / 64), (unsigned)batch);
        if (any_float)
          hipLaunchKernelGGL((dot_blocked_kernel<double>), g64, block, 0, ctx->stream, l->ptr, r->ptr, out->ptr, l_dt, r_dt, out_dt, M, N, K, lk, rk);
        else
          hipLaunchKernelGGL((dot_blocked_kernel<int64_t>), g64, block, 0, ctx->stream, l->ptr, r->ptr, out->ptr, l_dt, r_dt, out_dt, M, N, K, lk, rk);
        HIPNX_HIP(hipGetLastError());
        return HIPNX_OK;
      }
      // Few outputs over a long K (the weight gradient of a layer with a handful of classes: [6377, 80]^T . [6377, 3] is five
      // tiles): K is cut until every CU has two work-groups, where that saves more slabs than the second pass costs (four
      // and more: 1 to 3 us each against 5).  Not where a sum's order shows: an f64 operand or result adds over k in order.
      const bool any_f64 = l_dt == HIPNX_F64 || r_dt == HIPNX_F64 || out_dt == HIPNX_F64;
      const int64_t tiles = (int64_t)grid.x * grid.y * batch, slabs = (K + 63) / 64;
      int64_t nseg = any_f64 ? 1 : std::min<int64_t>(2 * (int64_t)ctx->num_cus / tiles, slabs / 2);
      int64_t seg_len = K;
      if (nseg > 1) {
        seg_len = (slabs + nseg - 1) / nseg * 64;
        nseg = (K + seg_len - 1) / seg_len;
      }
      if (nseg < 2 || slabs - seg_len / 64 < 4 || grid.y * nseg > 65535) nseg = 1, seg_len = K;
      void *ws = nullptr;
      size_t ws_cap = 0;
      if (nseg > 1 && pool_alloc(ctx, (size_t)(batch * M * N * nseg) * 8, &ws, &ws_cap) != HIPNX_OK) nseg = 1, seg_len = K;
      grid.y *= (unsigned)nseg;
      const dim3 finish((unsigned)std::min<int64_t>((batch * M * N + 255) / 256, 1 << 20));
#define HIPNX_GENERIC_K(CT, TK, ...) hipLaunchKernelGGL((dot_generic_kernel<CT, TK, ##__VA_ARGS__>), grid, block, 0, ctx->stream, l->ptr, r->ptr, out->ptr, l_dt, r_dt, out_dt, M, N, K, lk, rk, (CT *)ws, seg_len, (int)nseg)
#define HIPNX_GENERIC(CT, ...) do { if (K <= 32) HIPNX_GENERIC_K(CT, 16, ##__VA_ARGS__); else HIPNX_GENERIC_K(CT, 64, ##__VA_ARGS__); } while (0)
      if (any_float) {
        if (l_dt == HIPNX_F32 && r_dt == HIPNX_F32) HIPNX_GENERIC(double, HIPNX_F32, HIPNX_F32);
        else if (l_dt == HIPNX_BF16 && r_dt == HIPNX_BF16) HIPNX_GENERIC(double, HIPNX_BF16, HIPNX_BF16);
        else if (l_dt == HIPNX_F16 && r_dt == HIPNX_F16) HIPNX_GENERIC(double, HIPNX_F16, HIPNX_F16);
        else HIPNX_GENERIC(double);
        if (nseg > 1)
          hipLaunchKernelGGL((dot_reduce_finish_kernel<double>), finish, block, 0, ctx->stream, (const double *)ws, out->ptr, out_dt, batch * M * N, (int)nseg);
      } else {
        HIPNX_GENERIC(int64_t);
        if (nseg > 1)
          hipLaunchKernelGGL((dot_reduce_finish_kernel<int64_t>), finish, block, 0, ctx->stream, (const int64_t *)ws, out->ptr, out_dt, batch * M * N, (int)nseg);
      }
#undef HIPNX_GENERIC
#undef HIPNX_GENERIC_K
      if (ws) pool_free(ctx, ws, ws_cap);  // later work is ordered on the same stream
      HIPNX_HIP(hipGetLastError());
      return HIPNX_OK;
    }
  }

  // MFMA path: operands the kernels cannot take as they are, copied
  const int esz = dtype_size(l_dt);
  hipnx_buf *lt = nullptr, *rt = nullptr;
  int st = HIPNX_OK;
  if (l_relay) {
    st = hipnx_buf_alloc(ctx, (size_t)(batch * M * K * esz), &lt);
    if (!st) {
      int64_t dims[3] = {batch, K, M};
      int perm[3] = {0, 2, 1};
      st = hipnx_transpose(ctx, esz, 3, dims, perm, l, lt);
    }
  }
  if (!st && r_relay) {
    st = hipnx_buf_alloc(ctx, (size_t)(batch * N * K * esz), &rt);
    if (!st) {
      int64_t dims[3] = {batch, K, N};
      int perm[3] = {0, 2, 1};
      st = hipnx_transpose(ctx, esz, 3, dims, perm, r, rt);
    }
  }
  for (int side = 0; side < 2 && !st; side++) {
    bool &pad = side ? r_pad : l_pad;
    if (!pad) continue;
    hipnx_buf *&turned = side ? rt : lt, *padded = nullptr;
    st = pad_rows(ctx, esz, batch * (side ? N : M), K, turned ? turned : side ? r : l, &padded);
    if (st == HIPNX_ENOMEM && K * esz >= 16) {  // (such rows are copied for speed alone: without room for it they are read as they lie)
      pad = false;
      st = HIPNX_OK;
      continue;
    }
    if (turned) hipnx_buf_destroy(turned);  // (back to the pool: later work is ordered on the same stream)
    turned = padded;
  }
  if (!st) {
    Enter in(ctx);
    st = in.status;
    // the lock was dropped for the re-layout above: the operands may have been freed meanwhile
    if (!st) st = check_buf(ctx, l, (uint64_t)batch * M * K * dtype_size(l_dt), "dot lhs");
    if (!st) st = check_buf(ctx, r, (uint64_t)batch * N * K * dtype_size(r_dt), "dot rhs");
    if (!st) st = check_buf(ctx, out, (uint64_t)batch * M * N * out_dtype_size(out_dt), "dot out");
    if (!st && scale_mode != HIPNX_SCALE_NONE) st = check_buf(ctx, scale, 4, "dot_scaled scale");
    if (!st) {
      const void *lp = lt ? lt->ptr : l->ptr, *rp = rt ? rt->ptr : r->ptr;
      const bool l_kin = l_layout == HIPNX_K_INNER || l_relay, r_kin = r_layout == HIPNX_K_INNER || r_relay;
      const GemmChoice choice = gemm_choice(ctx->num_cus, l_dt, batch, M, N, K, l_kin, r_kin, partials);
      GemmArgs a{};
      a.l = (const unsigned char *)lp;
      a.r = (const unsigned char *)rp;
      a.out = out->ptr;
      a.odt = out_dt;
      const int64_t row_bytes = K * esz, nslab = (row_bytes + SLAB - 1) / SLAB;
      const int64_t pitch = (row_bytes + 15) / 16 * 16;
      a.M = M; a.N = N; a.Kb = nslab * SLAB;
      a.ld_l = !l_kin ? M * esz : l_pad ? pitch : row_bytes;
      a.ld_r = !r_kin ? N * esz : r_pad ? pitch : row_bytes;
      a.bs_l = l_pad ? M * pitch : M * row_bytes;
      a.bs_r = r_pad ? N * pitch : N * row_bytes;
      if (view) {
        a.ld_l = view->ld_l, a.bs_l = view->bs_l, a.ts_l = view->ts_l;
        a.ld_r = view->ld_r, a.bs_r = view->bs_r, a.ts_r = view->ts_r;
        a.batch_inner = (int)view->inner;
      }
      const bool ragged = (l_ragged && !l_relay) || (r_ragged && !r_relay);
      a.tail_l = gemm_tail(row_bytes, esz, ragged, l_kin, l_pad);
      a.tail_r = gemm_tail(row_bytes, esz, ragged, r_kin, r_pad);
      a.scale = scale_mode != HIPNX_SCALE_NONE ? (const float *)scale->ptr : nullptr;
      a.scale_mode = scale_mode;
      const int cfg = choice.cfg;
      int splits = choice.splits;
      const int64_t per_split = (nslab + splits - 1) / splits;
      void *ws = nullptr;
      size_t ws_cap = 0;
      if (splits > 1 && pool_alloc(ctx, (size_t)splits * M * N * 4, &ws, &ws_cap) != HIPNX_OK) splits = 1;
      if (splits > 1) {
        GemmArgs p = a;
        p.Kb = per_split * SLAB;
        p.all_slabs = (int)nslab;
        p.batch_inner = 0;
        p.bs_l = l_kin ? p.Kb : (p.Kb / esz) * a.ld_l;  // split s begins p.Kb bytes (or that many k-rows) further on
        p.bs_r = r_kin ? p.Kb : (p.Kb / esz) * a.ld_r;
        p.out = ws;
        p.scale_mode = HIPNX_SCALE_NONE;
        p.odt = l_dt == HIPNX_S8 ? HIPNX_S32 : HIPNX_F32;
        switch (l_dt) {
          case HIPNX_BF16: st = launch_gemm_bf16(ctx, cfg, l_kin, r_kin, p, splits); break;
          case HIPNX_F16: st = launch_gemm_f16(ctx, cfg, l_kin, r_kin, p, splits); break;
          case HIPNX_F32: st = launch_gemm_f32(ctx, cfg, l_kin, r_kin, p, splits); break;
          case HIPNX_F64: st = launch_gemm_f64(ctx, cfg, l_kin, r_kin, p, splits); break;
          default: st = launch_gemm_s8(ctx, cfg, l_kin, r_kin, p, splits); break;
        }
        if (!st) {
          const int64_t mn = M * N;
          dim3 grid((unsigned)std::min<int64_t>((mn / 4 + 255) / 256, 1 << 20)), block(256);
          if (scale_mode != HIPNX_SCALE_NONE)
            hipLaunchKernelGGL((splitk_combine_kernel<int, true>), grid, block, 0, ctx->stream, (const int *)ws, out->ptr, out_dt, mn, splits, (int)N, a.scale, scale_mode);
          else if (l_dt == HIPNX_S8) hipLaunchKernelGGL((splitk_combine_kernel<int>), grid, block, 0, ctx->stream, (const int *)ws, out->ptr, out_dt, mn, splits);
          else hipLaunchKernelGGL((splitk_combine_kernel<float>), grid, block, 0, ctx->stream, (const float *)ws, out->ptr, out_dt, mn, splits);
          hipError_t e = hipGetLastError();
          if (e != hipSuccess) st = hip_fail(e, "split-K combine launch");
        }
        pool_free(ctx, ws, ws_cap);  // later work is ordered on the same stream
      } else
      switch (l_dt) {
        case HIPNX_BF16: st = launch_gemm_bf16(ctx, cfg, l_kin, r_kin, a, batch); break;
        case HIPNX_F16: st = launch_gemm_f16(ctx, cfg, l_kin, r_kin, a, batch); break;
        case HIPNX_F32: st = launch_gemm_f32(ctx, cfg, l_kin, r_kin, a, batch); break;
        case HIPNX_F64: st = launch_gemm_f64(ctx, cfg, l_kin, r_kin, a, batch); break;
        default: st = launch_gemm_s8(ctx, cfg, l_kin, r_kin, a, batch); break;
      }
    }
  }
  // handing the workspaces back to the pool is safe: later work is ordered on the same stream
  if (lt) hipnx_buf_destroy(lt);
  if (rt) hipnx_buf_destroy(rt);
  return st;
}

extern "C" int hipnx_dot(hipnx_ctx *ctx, int l_dt, int r_dt, int out_dt, int64_t batch, int64_t M, int64_t N,
                         int64_t K, int l_layout, int r_layout, const hipnx_buf *l, const hipnx_buf *r,
                         hipnx_buf *out) {
  return dot_impl(ctx, l_dt, r_dt, out_dt, batch, M, N, K, l_layout, r_layout, l, r, out, HIPNX_SCALE_NONE, nullptr);
}

extern "C" int hipnx_dot_strided(hipnx_ctx *ctx, int l_dt, int r_dt, int out_dt, int64_t batch_outer, int64_t batch_inner, int64_t M,
                                 int64_t N, int64_t K, int l_layout, int r_layout, const int64_t *l_strides, const int64_t *r_strides,
                                 const hipnx_buf *l, const hipnx_buf *r, hipnx_buf *out) {
  const int lsz = dtype_size(l_dt), rsz = dtype_size(r_dt);
  if (lsz < 0 || rsz < 0) return set_error(HIPNX_EINVAL, "dot_strided: unknown element type");
  if (!l_strides || !r_strides || batch_outer < 0 || batch_inner < 0 || M < 0 || N < 0 || K < 0 || (batch_inner > 0 && batch_outer > INT64_MAX / batch_inner))
    return set_error(HIPNX_EINVAL, "dot_strided: bad extents or strides");
  if ((l_layout != HIPNX_K_INNER && l_layout != HIPNX_K_OUTER) || (r_layout != HIPNX_K_INNER && r_layout != HIPNX_K_OUTER))
    return set_error(HIPNX_EINVAL, "dot_strided: unknown operand layout");
  const int64_t batch = batch_outer * batch_inner;
  if (batch > 0 && M > 0 && N > 0 && K > 0) {
    Enter in(ctx);
    if (in.status) return in.status;
    for (int side = 0; side < 2; side++) {
      const int64_t *s = side ? r_strides : l_strides, rows = side ? N : M;
      const bool kin = (side ? r_layout : l_layout) == HIPNX_K_INNER;
      for (int i = 0; i < 3; i++)
        if (s[i] < 0 || s[i] > (1ll << 40)) return set_error(HIPNX_EINVAL, "dot_strided: a stride of %lld elements", (long long)s[i]);
      // runs that overlap within an item, or that are read as neighbours without being ones, are no operand
      if (s[2] < (kin ? K : rows)) return set_error(HIPNX_EINVAL, "dot_strided: rows of an operand overlap");
      const uint64_t bytes = strided_bytes(batch_outer, s[0], batch_inner, s[1], kin ? rows : K, s[2], kin ? K : rows, side ? rsz : lsz);
      if (int st = check_buf(ctx, side ? r : l, bytes, side ? "dot_strided rhs" : "dot_strided lhs")) return st;
    }
  }
  const DotView v{batch_inner, l_strides[2] * lsz, l_strides[0] * lsz, l_strides[1] * lsz, r_strides[2] * rsz, r_strides[0] * rsz, r_strides[1] * rsz};
  return dot_impl(ctx, l_dt, r_dt, out_dt, batch, M, N, K, l_layout, r_layout, l, r, out, HIPNX_SCALE_NONE, nullptr, &v);
}

extern "C" int hipnx_dot_scaled(hipnx_ctx *ctx, int l_dt, int r_dt, int64_t batch, int64_t M, int64_t N, int64_t K,
                                int l_layout, int r_layout, const hipnx_buf *l, const hipnx_buf *r, int scale_mode,
                                const hipnx_buf *scale, hipnx_buf *out) {
  if (scale_mode != HIPNX_SCALE_PER_COLUMN && scale_mode != HIPNX_SCALE_PER_ROW && scale_mode != HIPNX_SCALE_ONE)
    return set_error(HIPNX_EINVAL, "dot_scaled: scale mode %d", scale_mode);
  return dot_impl(ctx, l_dt, r_dt, HIPNX_F32, batch, M, N, K, l_layout, r_layout, l, r, out, scale_mode, scale);
}

extern "C" int hipnx_dot_scaled_any_k(hipnx_ctx *ctx, int l_dt, int r_dt, int64_t batch, int64_t M, int64_t N, int64_t K,
                                      int l_layout, int r_layout, const hipnx_buf *l, const hipnx_buf *r, int scale_mode,
                                      const hipnx_buf *scale, hipnx_buf *out) {
  if (scale_mode != HIPNX_SCALE_PER_COLUMN && scale_mode != HIPNX_SCALE_PER_ROW && scale_mode != HIPNX_SCALE_ONE)
    return set_error(HIPNX_EINVAL, "dot_scaled_any_k: scale mode %d", scale_mode);
  return dot_impl(ctx, l_dt, r_dt, HIPNX_F32, batch, M, N, K, l_layout, r_layout, l, r, out, scale_mode, scale, nullptr, true);
}
