// Axis reductions of a long, narrow slab: [red, inner] summed (or multiplied, ...) over `red` where a row is shorter than a
// work-group's reach (a table's columns, the gradient of a bias of ten classes).  See reduce_kernels.cuh for the wider ones.
#include "reduce_kernels.cuh"

namespace hipnx {

// Bound by memory.  The slab is read as flat vectors of eight elements: `lanes` lanes of a work-group cover g = lanes * 8 /
// inner whole rows, so a lane stays on the same columns for its whole walk, and the g rows are folded in LDS by halves.
// The last folded row is cut off at the end of the slab, wherever that is.  (Folding the rows by viewing the slab as
// [red / g, g * inner] and reducing twice took six launches, the last of them 41 dependent f64 loads deep in one
// work-group: f32 [671088, 100] 56 + 5 + 9 + 21 us, now 59 + 5 us.)
template <typename R, typename CT, int IDT, bool NT>
__global__ void __launch_bounds__(BLOCK)
reduce_narrow_kernel(const void *__restrict__ in, typename R::acc_t *__restrict__ partial, void *__restrict__ out, int idt_, int odt,
                     int64_t total, int inner, int lanes) {
  const int idt = IDT >= 0 ? IDT : idt_;
  __shared__ typename R::acc_t sm[BLOCK * E];
  const int lane = threadIdx.x, period = lanes * E;
  if (lane < lanes) {
    typename R::acc_t acc[E];
#pragma unroll
    for (int i = 0; i < E; i++) acc[i] = R::init();
    // four folded rows at a time, all four loads in flight, then the next four of this work-group: the grid sweeps the
    // slab together, from its end to its start -- what wrote it went the other way, and of a slab larger than the
    // last-level cache it is the end that is still there (f32 [671088, 100]
    // 67 -> 59 us, 46 where its writer was the call before)
    const int64_t run = 4 * (int64_t)period;
    for (int64_t q = (total - 1) / run - blockIdx.x; q >= 0; q -= gridDim.x) {
      const int64_t f = q * run + (int64_t)lane * E;
      if (f >= total) continue;
      if (f + 3 * (int64_t)period + E <= total) {
        CT v[4][E];
#pragma unroll
        for (int u = 0; u < 4; u++) load_vec<CT, E, true, NT>(in, idt, f + u * (int64_t)period, v[u]);
#pragma unroll
        for (int u = 0; u < 4; u++)
#pragma unroll
          for (int i = 0; i < E; i++) acc[i] = R::accumulate(acc[i], v[u][i], 0);
      } else {  // the last folded rows, cut off where the slab ends
        for (int64_t g = f; g < total; g += period)
#pragma unroll
          for (int i = 0; i < E; i++)
            if (g + i < total) acc[i] = R::accumulate(acc[i], load_one<CT>(in, idt, g + i), 0);
      }
    }
#pragma unroll
    for (int i = 0; i < E; i++) sm[lane * E + i] = acc[i];
  }
  __syncthreads();
  for (int rows = period / inner; rows > 1;) {
    const int half = (rows + 1) / 2;
    for (int j = threadIdx.x; j < (rows - half) * inner; j += BLOCK) sm[j] = R::combine(sm[j], sm[j + half * inner]);
    __syncthreads();
    rows = half;
  }
  if ((int)threadIdx.x < inner) {
    if (gridDim.x == 1) finalize(out, odt, threadIdx.x, sm[threadIdx.x]);
    else partial[(int64_t)blockIdx.x * inner + threadIdx.x] = sm[threadIdx.x];
  }
}

// partial[nseg, inner] -> out[inner]: a work-group per 8 columns, its 32 rows of lanes each fold a slice of the segments
// (few dependent round trips to L2, which is all this costs: 512 segments are four steps of four loads)
constexpr int NARROW_X = 8, NARROW_Y = BLOCK / NARROW_X;
template <typename R>
__global__ void __launch_bounds__(BLOCK)
combine_narrow_kernel(const typename R::acc_t *__restrict__ partial, void *__restrict__ out, int odt, int inner, int nseg) {
  typedef typename R::acc_t acc_t;
  __shared__ acc_t sm[NARROW_Y][NARROW_X];
  const int tx = threadIdx.x % NARROW_X, ty = threadIdx.x / NARROW_X, c = blockIdx.x * NARROW_X + tx;
  acc_t acc = R::init();
  if (c < inner) {
    int s = ty;
    for (; s + 3 * NARROW_Y < nseg; s += 4 * NARROW_Y) {
      acc_t a[4];
#pragma unroll
      for (int u = 0; u < 4; u++) a[u] = partial[(int64_t)(s + u * NARROW_Y) * inner + c];
#pragma unroll
      for (int u = 0; u < 4; u++) acc = R::combine(acc, a[u]);
    }
    for (; s < nseg; s += NARROW_Y) acc = R::combine(acc, partial[(int64_t)s * inner + c]);
  }
  sm[ty][tx] = acc;
  __syncthreads();
  for (int h = NARROW_Y / 2; h > 0; h /= 2) {
    if (ty < h) sm[ty][tx] = R::combine(sm[ty][tx], sm[ty + h][tx]);
    __syncthreads();
  }
  if (ty == 0 && c < inner) finalize(out, odt, c, sm[0][tx]);
}

template <typename R, typename CT, int IDT>
static int run_narrow_t(hipnx_ctx *ctx, int idt, int odt, int64_t red, int64_t inner, const void *in, void *out) {
  const int esize = dtype_size(idt), cols = (int)inner;
  const int unit = cols % 8 == 0 ? cols / 8 : cols % 4 == 0 ? cols / 4 : cols % 2 == 0 ? cols / 2 : cols;  // lanes of the fewest rows that are whole vectors
  const int lanes = BLOCK / unit * unit;
  const int64_t total = red * inner, run = 4 * (int64_t)lanes * E, runs = (total + run - 1) / run;
  // two work-groups per CU (f32 [671088, 100] held by the cache 46 / 44 / 45 / 48 us with 1 / 2 / 4 / 8, bf16 [1000003, 33]
  // 21 / 19 / 19 / 21; a narrower element leaves less in flight per lane), and two runs or more each
  const int64_t want = (int64_t)ctx->num_cus * (esize >= 2 ? 2 : 4), half = (runs + 1) / 2;
  const int64_t groups = half < want ? half : want;
  typename R::acc_t *partial = nullptr;
  void *ws = nullptr;
  size_t ws_cap = 0;
  if (groups > 1) {
    if (int st = pool_alloc(ctx, sizeof(typename R::acc_t) * (size_t)(groups * inner), &ws, &ws_cap)) return st;
    partial = (typename R::acc_t *)ws;
  }
  const dim3 grid((unsigned)groups), block(BLOCK);
  // (non-temporal as in run_reduce_t: far larger than the last-level cache and one access per vector)
  if (IDT >= 0 && total * esize >= (256ll << 20) && esize * E <= 16)
    hipLaunchKernelGGL((reduce_narrow_kernel<R, CT, IDT, (IDT >= 0)>), grid, block, 0, ctx->stream, in, partial, out, idt, odt, total, cols, lanes);
  else
    hipLaunchKernelGGL((reduce_narrow_kernel<R, CT, IDT, false>), grid, block, 0, ctx->stream, in, partial, out, idt, odt, total, cols, lanes);
  if (groups > 1)
    hipLaunchKernelGGL((combine_narrow_kernel<R>), dim3((unsigned)((cols + NARROW_X - 1) / NARROW_X)), block, 0, ctx->stream, partial, out, odt, cols, (int)groups);
  if (ws) pool_free(ctx, ws, ws_cap);  // later work on the stream is ordered behind the launches
  HIPNX_HIP(hipGetLastError());
  return HIPNX_OK;
}

// The element types compiled in: with the type a run-time argument a vector costs some hundred instructions, and a row that
// leaves half of the lanes idle waits for those (s16 [262144, 129], 129 of 256 lanes: 77 us, compiled in 19).  The 32-bit
// unsigned and 64-bit types are left: f64 and u64 [262144, 129] 195 and 162 us.
template <typename R, typename CT>
static int run_narrow(hipnx_ctx *ctx, int idt, int odt, int64_t red, int64_t inner, const void *in, void *out) {
#define HIPNX_NARROW_AS(T) if (idt == T) return run_narrow_t<R, CT, T>(ctx, idt, odt, red, inner, in, out);
  if constexpr (std::is_floating_point<CT>::value) {
    HIPNX_NARROW_AS(HIPNX_F32) HIPNX_NARROW_AS(HIPNX_BF16) HIPNX_NARROW_AS(HIPNX_F16)
  } else {
    HIPNX_NARROW_AS(HIPNX_S32) HIPNX_NARROW_AS(HIPNX_U8) HIPNX_NARROW_AS(HIPNX_S16) HIPNX_NARROW_AS(HIPNX_U16)
  }
#undef HIPNX_NARROW_AS
  return run_narrow_t<R, CT, -1>(ctx, idt, odt, red, inner, in, out);
}

// the accumulators of reduce_op (reduce.hip, reduce_select.hip)
template <int OP>
static int narrow_op(hipnx_ctx *ctx, int idt, int odt, int64_t red, int64_t inner, const void *in, void *out) {
  constexpr bool selects = OP != HIPNX_RED_SUM && OP != HIPNX_RED_PRODUCT;
  if constexpr (selects)
    if (is_float(idt) && idt != HIPNX_F64) return run_narrow<PlainReducer<float, OP, false>, float>(ctx, idt, odt, red, inner, in, out);
  if (is_float(idt)) return run_narrow<PlainReducer<double, OP, false>, double>(ctx, idt, odt, red, inner, in, out);
  if constexpr (OP == HIPNX_RED_MAX || OP == HIPNX_RED_MIN)
    if (idt == HIPNX_U64) return run_narrow<PlainReducer<int64_t, OP, true>, int64_t>(ctx, idt, odt, red, inner, in, out);
  return run_narrow<PlainReducer<int64_t, OP, false>, int64_t>(ctx, idt, odt, red, inner, in, out);
}

int reduce_narrow(hipnx_ctx *ctx, int op, int idt, int odt, int64_t red, int64_t inner, const void *in, void *out) {
  switch (op) {
    case HIPNX_RED_SUM: return narrow_op<HIPNX_RED_SUM>(ctx, idt, odt, red, inner, in, out);
    case HIPNX_RED_PRODUCT: return narrow_op<HIPNX_RED_PRODUCT>(ctx, idt, odt, red, inner, in, out);
    case HIPNX_RED_MAX: return narrow_op<HIPNX_RED_MAX>(ctx, idt, odt, red, inner, in, out);
    case HIPNX_RED_MIN: return narrow_op<HIPNX_RED_MIN>(ctx, idt, odt, red, inner, in, out);
    case HIPNX_RED_ALL: return narrow_op<HIPNX_RED_ALL>(ctx, idt, odt, red, inner, in, out);
    default: return narrow_op<HIPNX_RED_ANY>(ctx, idt, odt, red, inner, in, out);
  }
}

}  // namespace hipnx
