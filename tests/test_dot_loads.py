"""What the contraction kernels read: their loaders (nx_amd/csrc/gemm_loaders.cuh), compiled for the host, walk every lane, slab and
tile of an operand.  No load may leave the operand, and the slab in LDS holds the operand's elements, zeros behind the end of K."""
import shutil
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent
CLANG = shutil.which("amdclang++") or "/opt/rocm/llvm/bin/clang++"
PROGRAM = r"""
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <type_traits>
#include <vector>
#define __device__
#define __forceinline__ inline
#define __builtin_amdgcn_perm byte_permute

typedef unsigned char byte;
// bytes 0-3 of a selector are the second word's, 4-7 the first's
static unsigned byte_permute(unsigned a, unsigned b, unsigned sel) {
  const uint64_t both = ((uint64_t)a << 32) | b;
  unsigned out = 0;
  for (int i = 0; i < 4; i++) out |= (unsigned)((both >> (((sel >> (8 * i)) & 7) * 8)) & 255) << (8 * i);
  return out;
}
static const byte *first, *behind;  // the operand
static int lane_now;
static long outside, wrong, loads;

namespace hipnx {
typedef int v4i __attribute__((ext_vector_type(4)));
static const unsigned g_zero16[4] = {};
static v4i load_piece(const byte *p) {
  v4i v = {-1, -1, -1, -1};
  loads++;
  if (p < first || p + 16 > behind) outside++;
  else memcpy(&v, p, 16);
  return v;
}
static void lds_dma16(const byte *g, byte *lds) {
  const v4i v = g == (const byte *)g_zero16 ? v4i{0, 0, 0, 0} : load_piece(g);
  memcpy(lds + 16 * lane_now, &v, 16);
}
static void lds_dma16_at(const byte *base, unsigned off, byte *lds) { lds_dma16(base + off, lds); }
static const byte *wave_uniform(const byte *p) { return p; }
}
#include "@LOADERS@"
using namespace hipnx;

// the operand in memory of its own size; the rows (K-inner) or columns (K-outer) of item `item` from `row0` on, slab by slab
struct Operand {
  bool k_inner;
  int es;
  int64_t batch, rows, K, ld, item_bytes;
  std::vector<byte> data;
  Operand(bool kin, int es_, int64_t b, int64_t r, int64_t k) : k_inner(kin), es(es_), batch(b), rows(r), K(k), ld((kin ? k : r) * es_), item_bytes(r * k * es_), data(b * item_bytes) {
    for (byte &x : data) x = (byte)(1 + rand() % 255);  // (no zeros)
    first = data.data();
    behind = first + data.size();
  }
  const byte *item(int64_t b) const { return data.data() + b * item_bytes; }
  const byte *element(int64_t b, int64_t row, int64_t k) const { return item(b) + (k_inner ? row * ld + k * es : k * ld + row * es); }
};

// LDS as [row][k] (slot: where a row keeps its chunk) or as [k][row]
template <int ES, int ROWS, class Slot>
static void compare(const Operand &o, int64_t b, int64_t row0, int64_t k0, bool k_major, const byte *lds, Slot slot) {
  for (int r = 0; r < ROWS && row0 + r < o.rows; r++)
    for (int k = 0; k < SLAB / ES; k++) {
      const byte zero[8] = {}, *want = k0 + k < o.K ? o.element(b, row0 + r, k0 + k) : zero;
      const byte *got = k_major ? lds + k * ROWS * ES + slot(k, r * ES / 16) * 16 + r * ES % 16 : lds + r * SLAB + slot(r, k * ES / 16) * 16 + k * ES % 16;
      if (memcmp(got, want, ES)) wrong++;
    }
}

template <int ES, int ROWS, class Walk>
static void every_tile(const Operand &o, bool ragged, Walk walk) {
  const int tail = gemm_tail(o.K * ES, ES, ragged, o.k_inner, false);
  const int64_t nslab = (o.K * ES + SLAB - 1) / SLAB;
  for (int64_t b = 0; b < o.batch; b++)
    for (int64_t row0 = 0; row0 < o.rows; row0 += ROWS)
      for (int64_t s = 0; s < nslab; s++) {
        std::vector<byte> lds(ROWS * SLAB, (byte)0xEE);
        walk(b, row0, s, s == nslab - 1 ? tail : 0, lds.data());
      }
}

template <class F>
static void lanes(int waves, F f) {
  for (int w = 0; w < waves; w++)
    for (lane_now = 0; lane_now < 64; lane_now++) f(w, lane_now);
}

template <class L, int ES, int ROWS, int WAVES, bool KIN>
static void dma(const Operand &o, bool ragged) {
  every_tile<ES, ROWS>(o, ragged, [&](int64_t b, int64_t row0, int64_t s, int tail, byte *lds) {
    std::vector<L> at(WAVES * 64);
    const int64_t k0 = s * (KIN ? SLAB : SLAB / ES);
    lanes(WAVES, [&](int w, int l) { at[w * 64 + l].init(o.item(b), o.ld, row0, o.rows, w, l); });
    lanes(WAVES, [&](int w, int l) {
      const L &x = at[w * 64 + l];
      if constexpr (KIN) {
        if (tail) x.issue_partial(k0, tail, lds, w, l);
        else if constexpr (requires { x.issue(k0, lds, w); }) x.issue(k0, lds, w);
        else x.issue(k0, lds);
      } else {
        if (tail) x.issue_partial(k0, o.ld, tail, lds, w, l);
        else if constexpr (requires { x.issue(k0, o.ld, lds, w); }) x.issue(k0, o.ld, lds, w);
        else x.issue(k0, o.ld, lds);
      }
    });
    if (tail)
      lanes(WAVES, [&](int w, int l) {
        if constexpr (KIN) at[w * 64 + l].finish_partial(k0, tail, lds, w, l);
        else at[w * 64 + l].finish_partial(k0, o.ld, tail, lds, w, l);
      });
    constexpr bool rows_low_bits = std::is_same<L, PPKInnerLoader<ROWS, WAVES>>::value;
    compare<ES, ROWS>(o, b, row0, s * (SLAB / ES), !KIN, lds, [&](int i, int chunk) {
      if constexpr (!KIN) return tr_slot_w<ES, ROWS * ES>(i, chunk);
      else return rows_low_bits ? lds_slot16(i, chunk) : lds_slot(i, chunk);
    });
  });
}

template <int ES, int ROWS, int THREADS>
static void staged(const Operand &o, bool ragged) {
  every_tile<ES, ROWS>(o, ragged, [&](int64_t b, int64_t row0, int64_t s, int tail, byte *lds) {
    for (int t = 0; t < THREADS; t++) {
      KOuterStage<ES, ROWS, THREADS> stage;
      if (tail) stage.fetch_partial(o.item(b), o.ld, row0, o.rows, s * (SLAB / ES), tail, t);
      else stage.fetch(o.item(b), o.ld, row0, o.rows, s * (SLAB / ES), t);
      stage.store(lds, t);
    }
    compare<ES, ROWS>(o, b, row0, s * (SLAB / ES), false, lds, [](int i, int chunk) { return lds_slot(i, chunk); });
  });
}

template <int ES, bool KIN, class F>
static void sizes(const char *name, int rows_from, F f) {
  outside = wrong = loads = 0;
  constexpr int KS = SLAB / ES;
  for (int64_t rows : {1, 2, 7, 8, 9, 15, 16, 17, 31, 33, 64, 65, 100, 127, 128, 129, 131, 144, 256, 259, 300})
    for (int64_t K : {1, 3, 7, 8, 15, 16, 17, KS - 1, KS, KS + 1, 2 * KS, 2 * KS + 5, 3 * KS - 16 / ES})
      for (int64_t batch : {1, 2}) {
        if (rows < rows_from || (KIN && K * ES < 16) || (ES == 8 && (rows % 2 || K % KS))) continue;  // (copied first, or another kernel's)
        Operand o(KIN, ES, batch, rows, K);
        const bool ragged = !KIN && rows * ES % 16 != 0;
        f(o, ragged);
        if (!ragged) f(o, true);  // (the other operand's are)
      }
  printf("%s %ld %ld %ld\n", name, loads, outside, wrong);
}

int main() {
#define INNER(L, ES, ROWS, WAVES) sizes<ES, true>(#L " " #ES " " #ROWS " " #WAVES, 1, dma<L<ROWS, WAVES>, ES, ROWS, WAVES, true>)
#define OUTER(L, ES, ROWS, WAVES) sizes<ES, false>(#L " " #ES " " #ROWS " " #WAVES, 16 / ES, dma<L<ES, ROWS, WAVES>, ES, ROWS, WAVES, false>)
#define STAGED(ES, ROWS, THREADS) sizes<ES, false>("KOuterStage " #ES " " #ROWS " " #THREADS, 16 / ES, staged<ES, ROWS, THREADS>)
  INNER(KInnerLoader, 1, 64, 2); INNER(KInnerLoader, 2, 32, 2); INNER(KInnerLoader, 2, 128, 4); INNER(KInnerLoader, 4, 128, 8); INNER(KInnerLoader, 8, 64, 4);
  INNER(PPKInnerLoader, 1, 64, 4); INNER(PPKInnerLoader, 2, 128, 4); INNER(PPKInnerLoader, 2, 256, 8); INNER(PPKInnerLoader, 4, 128, 4);
  OUTER(KOuterDmaLoader, 2, 128, 4); OUTER(KOuterDmaLoader, 2, 256, 8); OUTER(KOuterDmaLoader, 1, 256, 8);
  OUTER(PPKOuterLoader, 1, 64, 4); OUTER(PPKOuterLoader, 1, 128, 4); OUTER(PPKOuterLoader, 1, 256, 8); OUTER(PPKOuterLoader, 2, 128, 4); OUTER(PPKOuterLoader, 2, 256, 8);
  STAGED(1, 64, 128); STAGED(1, 128, 256); STAGED(2, 32, 128); STAGED(2, 128, 256); STAGED(4, 32, 256); STAGED(4, 64, 128); STAGED(4, 128, 512); STAGED(8, 128, 256);
}
"""


def test_every_load_of_a_contraction_lies_in_its_operand_and_lds_holds_the_slab(tmp_path):
    (tmp_path / "loads.cpp").write_text(PROGRAM.replace("@LOADERS@", str(ROOT / "nx_amd" / "csrc" / "gemm_loaders.cuh")))
    subprocess.run([CLANG, "-std=c++20", "-O1", "-Wno-everything", "-o", str(tmp_path / "loads"), str(tmp_path / "loads.cpp")], check=True)
    lines = subprocess.run([str(tmp_path / "loads")], capture_output=True, text=True, check=True).stdout.splitlines()
    assert len(lines) == 25
    for line in lines:
        loads, outside, wrong = map(int, line.split()[-3:])
        assert loads > 1000 and outside == 0 and wrong == 0, line
