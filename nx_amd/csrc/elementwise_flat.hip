// Binary operations of a dense [rows, cols] tensor with a row [cols] or one value per row where a row is not whole vectors of
// eight elements (a table of 100 features and their means, a bias of 10 classes): float types, one type throughout.  And
// two forms of mixed types: a mean's quotient of sums and a whole number, and values times a mask.
#include <type_traits>

#include "elementwise_ops.cuh"
#include "elementwise_vec.cuh"
#include "internal.h"

namespace hipnx {

// Bound by memory: a lane takes 16 bytes of the flat output, whatever rows they lie in, and the same of the dense operand;
// the other operand comes from a row or a column that the caches hold.  (The general kernel does the same with the
// operands' forms, strides and outer axes as run-time arguments and 64-bit offsets, some hundred instructions per
// vector: f32 [671088, 100] less a row 132 us back to back, now 89 (6.0 TB/s); 122 and 77 right behind a pass that read
// the table.)
//   L_DENSE: the left operand is the dense one.  PER_ROW: the other holds one value per row, `step` elements apart.
template <int OP, int FIX, bool L_DENSE, bool PER_ROW>
__global__ void __launch_bounds__(BLOCK)
binary_flat_kernel(const void *__restrict__ dense, const void *__restrict__ other, void *__restrict__ out, uint32_t total, uint32_t cols,
                   FastDiv32 fd, int64_t step) {
  constexpr int E = vec_elems(FIX, FIX);
  const uint32_t f0 = (blockIdx.x * (uint32_t)BLOCK + threadIdx.x) * E;
  if (f0 >= total) return;
  uint32_t row = fastdiv(f0, fd), col = f0 - row * cols;
  const bool whole = total - f0 >= (uint32_t)E;
  float a[E], b[E], c[E];
  if (whole) load_vec<float, E>(dense, FIX, f0, a);
  else {
#pragma unroll
    for (int i = 0; i < E; i++) a[i] = f0 + i < total ? load_one<float>(dense, FIX, f0 + i) : 1.0f;
  }
  if constexpr (PER_ROW) {
    if (cols >= (uint32_t)E) {  // the vector lies in one row or two
      const float first = load_one<float>(other, FIX, row * step);
      const float second = col + E > cols && f0 + (cols - col) < total ? load_one<float>(other, FIX, (row + 1) * step) : first;
#pragma unroll
      for (int i = 0; i < E; i++) b[i] = col + i < cols ? first : second;
    } else {
#pragma unroll
      for (int i = 0; i < E; i++) {
        b[i] = f0 + i < total ? load_one<float>(other, FIX, row * step) : 1.0f;
        if (++col == cols) col = 0, row++;
      }
    }
  } else if (cols % E == 0) {  // (rows of 4-byte elements that are whole 16-byte vectors)
    load_vec<float, E>(other, FIX, col, b);
  } else {
#pragma unroll
    for (int i = 0; i < E; i++) {
      b[i] = load_one<float>(other, FIX, col);
      if (++col == cols) col = 0;
    }
  }
#pragma unroll
  for (int i = 0; i < E; i++) c[i] = L_DENSE ? binary_apply<OP, float, false>(a[i], b[i]) : binary_apply<OP, float, false>(b[i], a[i]);
  if (whole) store_vec<float, E>(out, FIX, f0, c);
  else {
#pragma unroll
    for (int i = 0; i < E; i++)
      if (f0 + i < total) store_one<float>(out, FIX, f0 + i, c[i]);
  }
}

template <int OP, int FIX>
static void launch_flat(const hipnx_ctx *ctx, bool l_dense, bool per_row, const void *dense, const void *other, void *out, uint32_t total,
                        uint32_t cols, int64_t step) {
  constexpr int PER_BLOCK = vec_elems(FIX, FIX) * BLOCK;
  const dim3 grid((total + PER_BLOCK - 1) / PER_BLOCK), block(BLOCK);
  const FastDiv32 fd = make_fastdiv(cols);
  if (l_dense && per_row) hipLaunchKernelGGL((binary_flat_kernel<OP, FIX, true, true>), grid, block, 0, ctx->stream, dense, other, out, total, cols, fd, step);
  else if (l_dense) hipLaunchKernelGGL((binary_flat_kernel<OP, FIX, true, false>), grid, block, 0, ctx->stream, dense, other, out, total, cols, fd, step);
  else if (per_row) hipLaunchKernelGGL((binary_flat_kernel<OP, FIX, false, true>), grid, block, 0, ctx->stream, dense, other, out, total, cols, fd, step);
  else hipLaunchKernelGGL((binary_flat_kernel<OP, FIX, false, false>), grid, block, 0, ctx->stream, dense, other, out, total, cols, fd, step);
}

template <int OP>
static bool flat_op(const hipnx_ctx *ctx, int dt, bool l_dense, bool per_row, const void *dense, const void *other, void *out, uint32_t total,
                    uint32_t cols, int64_t step) {
  if constexpr (binary_int_only(OP) || binary_can_raise(OP, true)) return false;
  else {
    if (dt == HIPNX_F32) launch_flat<OP, HIPNX_F32>(ctx, l_dense, per_row, dense, other, out, total, cols, step);
    else if (dt == HIPNX_BF16) launch_flat<OP, HIPNX_BF16>(ctx, l_dense, per_row, dense, other, out, total, cols, step);
    else if (dt == HIPNX_F16) launch_flat<OP, HIPNX_F16>(ctx, l_dense, per_row, dense, other, out, total, cols, step);
    else return false;
    return true;
  }
}

template <int... OPS>
static bool flat_any(std::integer_sequence<int, OPS...>, const hipnx_ctx *ctx, int op, int dt, bool l_dense, bool per_row, const void *dense,
                     const void *other, void *out, uint32_t total, uint32_t cols, int64_t step) {
  bool took = false;
  (void)((op == OPS ? (took = flat_op<OPS>(ctx, dt, l_dense, per_row, dense, other, out, total, cols, step), true) : false) || ...);
  return took;
}

// W consecutive elements a lane.  NUMBER: the right operand is one element.
// (The kernel that reads its operands' types as it runs is some thousand instructions, which a launch of a few waves spends its time
// fetching, the more so behind a pass that went through the caches.  us, there / here: 100 f32 sums over an s32 count behind
// 268 MB 8.0 / 4.8, 300 behind 24 MB 6.4 / 1.5; f32 [4096, 512] times a u8 mask 5.4 / 4.0 a call.)
template <int OP, typename CT, int LDT, int RDT, int W, bool NUMBER>
__global__ void __launch_bounds__(BLOCK)
binary_mixed_kernel(const void *__restrict__ l, const void *__restrict__ r, void *__restrict__ out, uint32_t n) {
  const uint32_t f0 = (blockIdx.x * (uint32_t)BLOCK + threadIdx.x) * W;
  if (f0 >= n) return;
  CT a[W], b[W], c[W];
  if (n - f0 >= (uint32_t)W) {
    load_vec<CT, W>(l, LDT, f0, a);
    if constexpr (NUMBER) {
      b[0] = load_one<CT>(r, RDT, 0);
#pragma unroll
      for (int i = 1; i < W; i++) b[i] = b[0];
    } else load_vec<CT, W>(r, RDT, f0, b);
#pragma unroll
    for (int i = 0; i < W; i++) c[i] = binary_apply<OP, CT, false>(a[i], b[i]);
    store_vec<CT, W>(out, LDT, f0, c);
  } else {
    for (uint32_t f = f0; f < n; f++)
      store_one<CT>(out, LDT, f, binary_apply<OP, CT, false>(load_one<CT>(l, LDT, f), load_one<CT>(r, RDT, NUMBER ? 0 : f)));
  }
}

// Flat operands of n elements, ls / rs 1 or (one element for all) 0, the result of the float operand's type:
//   float / one s32 number, computed in f64 as any operation with a 32-bit integer is, of up to 2^16 elements (a lane each; more are
//   bound by memory, not by the launch);
//   f32 * u8, either way round (a product commutes), below 2^31 elements.
bool binary_mixed(const hipnx_ctx *ctx, int op, int l_dt, int r_dt, int out_dt, const void *l, const void *r, void *out, int64_t n, int64_t ls, int64_t rs) {
  if (op == HIPNX_DIVIDE && r_dt == HIPNX_S32 && l_dt == out_dt && (ls == 1 || n == 1) && (rs == 0 || n == 1) && n <= (1 << 16)) {
    const dim3 grid((unsigned)((n + BLOCK - 1) / BLOCK)), block(BLOCK);
    if (l_dt == HIPNX_F32) hipLaunchKernelGGL((binary_mixed_kernel<HIPNX_DIVIDE, double, HIPNX_F32, HIPNX_S32, 1, true>), grid, block, 0, ctx->stream, l, r, out, (uint32_t)n);
    else if (l_dt == HIPNX_BF16) hipLaunchKernelGGL((binary_mixed_kernel<HIPNX_DIVIDE, double, HIPNX_BF16, HIPNX_S32, 1, true>), grid, block, 0, ctx->stream, l, r, out, (uint32_t)n);
    else if (l_dt == HIPNX_F16) hipLaunchKernelGGL((binary_mixed_kernel<HIPNX_DIVIDE, double, HIPNX_F16, HIPNX_S32, 1, true>), grid, block, 0, ctx->stream, l, r, out, (uint32_t)n);
    else return false;
    return true;
  }
  const bool masked = l_dt == HIPNX_F32 && r_dt == HIPNX_U8, mask_first = l_dt == HIPNX_U8 && r_dt == HIPNX_F32;
  if (op == HIPNX_MULTIPLY && out_dt == HIPNX_F32 && (masked || mask_first) && ls == 1 && rs == 1 && n < (1ll << 31)) {
    const dim3 grid((unsigned)((n + 4 * BLOCK - 1) / (4 * BLOCK))), block(BLOCK);
    hipLaunchKernelGGL((binary_mixed_kernel<HIPNX_MULTIPLY, float, HIPNX_F32, HIPNX_U8, 4, false>), grid, block, 0, ctx->stream, masked ? l : r, masked ? r : l, out, (uint32_t)n);
    return true;
  }
  return false;
}

// Strides per row (l0, r0) and column (l1, r1; 0 or 1) of both operands; total < 2^31.  Taken where one operand is as dense as
// the output and the other repeats along the rows or along the columns.
bool binary_flat(const hipnx_ctx *ctx, int op, int dt, const void *l, const void *r, void *out, int64_t total, int64_t cols,
                 int64_t l0, int64_t l1, int64_t r0, int64_t r1) {
  auto dense = [&](int64_t s0, int64_t s1) { return s1 == 1 && s0 == cols; };
  auto repeats = [&](int64_t s0, int64_t s1) { return (s1 == 1 && s0 == 0) || (s1 == 0 && s0 > 0); };
  const bool l_dense = dense(l0, l1) && repeats(r0, r1);
  if (!l_dense && !(dense(r0, r1) && repeats(l0, l1))) return false;
  const int64_t step = l_dense ? r0 : l0;
  return flat_any(std::make_integer_sequence<int, HIPNX_NBINARY>{}, ctx, op, dt, l_dense, (l_dense ? r1 : l1) == 0, l_dense ? l : r,
                  l_dense ? r : l, out, (uint32_t)total, (uint32_t)cols, step);
}

}  // namespace hipnx
