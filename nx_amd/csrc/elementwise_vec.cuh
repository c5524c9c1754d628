// What the element-wise kernels share: the vector of a lane and the division of an index by an invariant extent.
#pragma once
#include "dtypes.cuh"

namespace hipnx {

constexpr int E = 8;
// A lane's vector when the element types are known at compile time: 16 bytes of the WIDEST type involved -- 8 elements of
// 1 or 2 bytes, 4 of 4 bytes, 2 of 8 bytes.  One 16-byte access per lane with the lanes side by side is what streams
// fastest here: a wave instruction then covers whole cache lines, where two adjacent 16-byte accesses per lane (eight
// f32) make every instruction touch twice the lines it fills (f32 multiply: 8.4 M elements 11.3 -> 9.4 us, 268 M
// elements 5.8 -> 6.2 TB/s; bf16 -> f32 conversion of 8.4 M elements 9.6 -> 7.6 us).  The narrower side of a
// conversion or comparison moves 8, 4 or 2 bytes per lane, still lanes side by side.
constexpr int fixed_type_bytes(int dt) {
  return dt < 0 ? 0
         : (dt == HIPNX_U8 || dt == HIPNX_S8) ? 1
         : (dt == HIPNX_U16 || dt == HIPNX_S16 || dt == HIPNX_F16 || dt == HIPNX_BF16 || dt == HIPNX_BF16_RNE) ? 2
         : (dt == HIPNX_U32 || dt == HIPNX_S32 || dt == HIPNX_F32) ? 4 : 8;
}
constexpr int vec_elems(int fix_in, int fix_out) {
  const int a = fixed_type_bytes(fix_in), b = fixed_type_bytes(fix_out), w = a > b ? a : b;
  return w == 8 ? 2 : w == 4 ? 4 : 8;  // (types known at run time only: 8 elements)
}
constexpr int BLOCK = 256;

// Division of an index below 2^31 by an invariant divisor below 2^31 as one multiplication: the 64-bit
// division the compiler emits costs every wave some hundred scalar and vector instructions, more than the
// rest of an 8-element vector's work.
struct FastDiv32 {
  uint32_t mul, shr;
};
static FastDiv32 make_fastdiv(uint32_t d) {
  uint32_t shr = 0;
  while ((1ull << shr) < d) shr++;
  return FastDiv32{(uint32_t)(((1ull << 32) * ((1ull << shr) - d)) / d + 1), shr};
}
__device__ __forceinline__ uint32_t fastdiv(uint32_t n, FastDiv32 f) { return (__umulhi(n, f.mul) + n) >> f.shr; }

}  // namespace hipnx
