// The block cipher of Nx.Random (nx/lib/nx/random.ex:236-281), shared by the kernels of random.hip and by groups compiled at run time.
#pragma once
#include "dtypes.cuh"

namespace hipnx {

__device__ __forceinline__ uint32_t rotl32(uint32_t x, int r) { return (x << r) | (x >> (32 - r)); }

// 20 rounds on one counter pair, key already split into the three schedule words
__device__ __forceinline__ void threefry_pair(uint32_t &x1, uint32_t &x2, uint32_t key1, uint32_t key2) {
  uint32_t k1 = key2, k2 = key1 ^ key2 ^ 0x1BD11BDAu, k3 = key1;
  x1 += key1;
  x2 += key2;
  constexpr int R[2][4] = {{13, 15, 26, 6}, {17, 29, 16, 24}};
#pragma unroll
  for (int g = 1; g <= 5; g++) {
#pragma unroll
    for (int r = 0; r < 4; r++) {
      x1 += x2;
      x2 = rotl32(x2, R[(g - 1) & 1][r]) ^ x1;
    }
    x1 += k1;
    x2 += k2 + (uint32_t)g;
    const uint32_t t = k1; k1 = k2; k2 = k3; k3 = t;
  }
}

// Key number `index` of the `parts` that split/2 makes of a key (random.ex:148-152): words 2 index and 2 index + 1 of the cipher over
// the counters 0 .. 2 parts - 1.  Uniform in, uniform out: scalar instructions.
__device__ __forceinline__ void threefry_sub_key(uint32_t &key1, uint32_t &key2, uint32_t parts, uint32_t index) {
  uint32_t word[2];
#pragma unroll
  for (int w = 0; w < 2; w++) {
    const uint32_t f = 2 * index + w, j = f < parts ? f : f - parts;
    uint32_t a = j, b = parts + j;
    threefry_pair(a, b, key1, key2);
    word[w] = f < parts ? a : b;
  }
  key1 = word[0];
  key2 = word[1];
}

}  // namespace hipnx
