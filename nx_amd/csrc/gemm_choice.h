// The rules of a contraction on the matrix cores: its tile, the number of ranges its K is cut into, and whether an operand whose rows
// are not whole pieces is copied first.  Host code without the device's headers: a function of sizes and types.
#pragma once
#include <algorithm>
#include <cstdint>

#include "../../include/hipnx.h"

namespace hipnx {

constexpr int SLAB = 128;  // bytes of K per row per slab

// tile configurations of gemm_pipelined_kernel<DT, WM, WN, TM, TN, ...>
enum {
  GEMM_CFG_256x128 = 3,  // 256 x 128, the two-group kernel with half-width wave tiles: 2-byte types whose 256 x 256 grid is too small
  GEMM_CFG_256 = 0,  // 256 x 256, 8 waves (4 x 2, each 64 x 128): large square-ish problems
  GEMM_CFG_128 = 1,  // 128 x 128: mid-size and batched problems; 4 waves (2 x 2, each 64 x 64), or two such groups sharing K
  GEMM_CFG_64 = 2,  // 64 x 64 on the two-group kernel (2-byte K-inner pairs, int8): small and mid-size problems, few rows; otherwise 64 x 32, 2 waves
  GEMM_CFG_64x128 = 4, // 64 x 128, wherever the cost models below have it cheapest: the two-group kernel (2-byte, int8) or 4 waves (2 x 2, each 32 x 64)
  GEMM_CFG_32x128 = 6, // 32 x 128, 4 waves (1 x 4, each 32 x 32): 2-byte weights stored K-outer, few rows or small problems
  GEMM_CFG_128x32 = 5  // 128 x 32, 4 waves (4 x 1, each 32 x 32): many rows against up to 32 columns (a layer with a few outputs)
};

struct GemmChoice {
  int cfg, splits, rows, cols;
};
// The tile of a contraction on the matrix cores and the number of ranges K is cut into.
// partials: whether ranges' sums may be kept apart (as s32 for int8) and added by a second launch.
static inline GemmChoice gemm_choice(int64_t num_cus, int l_dt, int64_t batch, int64_t M, int64_t N, int64_t K, bool l_kin, bool r_kin, bool partials) {
  const int esz = l_dt == HIPNX_S8 ? 1 : l_dt == HIPNX_BF16 || l_dt == HIPNX_F16 ? 2 : l_dt == HIPNX_F32 ? 4 : 8;
  const int64_t nslab = (K * esz + SLAB - 1) / SLAB;
  // tile choice: the largest tile that still gives every CU work; few rows against a long
  // weight matrix stream the weights with many small tiles
  const int64_t t256 = ((M + 255) / 256) * ((N + 255) / 256) * batch;
  const int64_t t128 = ((M + 127) / 128) * ((N + 127) / 128);
  const int64_t tw = ((M + 255) / 256) * ((N + 127) / 128) * batch;
  const bool two_byte = l_dt == HIPNX_BF16 || l_dt == HIPNX_F16;
  const bool big_ok = M >= 192 && N >= 192;
  int cfg;
  // few rows: 64-row tiles (f32: whatever its cost model below picks), except for a 2-byte K-outer operand
  // (x . W with W stored [K, N]), which only the 128-row kernels read by transposing loads
  // (64 x 4096 x 4096 bf16: 72 us on 64 x 32 tiles, 16.5 us there)
  const bool wide = l_dt == HIPNX_F32 || l_dt == HIPNX_F64;  // (an f64 slab costs the matrix pipes what an f32 one does)
  if (M <= 64 && !wide && !(two_byte && !(l_kin && r_kin) && N >= 128)) cfg = GEMM_CFG_64;
  else if (t256 * 4 >= num_cus * 3 && big_ok) cfg = GEMM_CFG_256;
  else if (two_byte && M >= 192 && N >= 128 && t128 * batch > num_cus)
    // More 128 x 128 tiles than CUs: half-width tiles of the two-group kernel while they fit the CUs in one
    // round, even where they leave some idle (1280 x 4096 x 4096, 160 tiles: 66 us; as 320 tiles of
    // 128 x 128 in two rounds: 76 us); where they would need a second round, full tiles on what is then more
    // than half of the CUs (3072^3: 144 tiles of 256 x 256 72 us, 288 half-width tiles 100 us)
    cfg = tw <= num_cus || !big_ok ? GEMM_CFG_256x128 : GEMM_CFG_256;
  else if (l_dt == HIPNX_S8 && big_ok && t256 * 2 >= num_cus)
    cfg = GEMM_CFG_256;  // int8 has no half-width tile: full tiles from half of the CUs on (3072^3: 46 us against 57 us)
  else cfg = GEMM_CFG_128;
  // many rows against at most 32 columns (a layer with a few outputs): a 128-column tile would be three
  // quarters empty or more, and its MFMA work is what bounds f32
  if (N <= 32 && M > 64 && cfg == GEMM_CFG_128) cfg = GEMM_CFG_128x32;
  // A grid of 128 x 128 tiles that leaves three quarters of the CUs idle (a few hundred rows against a long
  // weight matrix: 128 x 4096 x 4096 is 32 tiles walking 64 slabs each) splits K over S work-groups per tile:
  // f32 (s32) partial results in pool workspace, then one pass that adds them in split order.
  int splits = 1;
  auto per_split = [&](int cand) { return (nslab + cand - 1) / cand; };
  auto reaches = [&](int cand) { return per_split(cand) * (cand - 1) < nslab; };  // (every split has a slab)
  const bool splittable = (cfg == GEMM_CFG_128 || cfg == GEMM_CFG_128x32) && batch == 1 && partials;
  if (wide && cfg == GEMM_CFG_128x32) {
    // (0.6 us per slab of a 128 x 32 tile; the split as below)
    const int64_t cus = num_cus, tiles = t128 * batch;
    double best = 10.0 + (double)((tiles + cus - 1) / cus) * (double)nslab * 0.6;
    if (splittable)
      for (int cand = 2; cand <= 64; cand *= 2) {
        if (tiles * cand > cus || nslab / cand < 2 || !reaches(cand)) continue;
        const double t = 10.0 + (double)per_split(cand) * 0.6 + 5.0 + 2.0 * (double)cand * (double)(M * N) * 4.0 / 8.0e6;
        if (t < best) { best = t; splits = cand; }
      }
  } else if (wide) {
    // An f32 slab is eight times the MFMA work of a 2-byte one, so a grid that leaves CUs idle is cut much earlier: the
    // cheapest, by the figures below, of 128 x 128, 64 x 128 (up to 64 rows a 128-row tile would be half empty; and
    // a last round that leaves most CUs idle ends sooner in halves) and 64 x 32 tiles, the first two also with K
    // split up to 64 ways, 2 slabs or more each.  512^3: 41 -> 18 us; 256 x 256 x 16384: 84 -> 40 us.
    //   A work-group takes `alone` us per slab while it has its CU to itself, waiting for memory much of it; up to
    //   `resident` of them (as the LDS holds) share a CU and take `shared` us per slab and work-group together,
    //   near what the MFMAs take: a split that puts two or three work-groups on a CU pays for its second pass
    //   (784 x 512 x 4096, 52 tiles: 4 splits 58 us, 8 splits 50; 1000 x 700 x 1500, 96 tiles: 2 splits 45 us,
    //   8 splits 33; 300 x 1000 x 900, 40 tiles: 64 x 32 tiles 29 us, 6 splits of 64 x 128 16; 2048^3: 128 x 128
    //   174 us, 64 x 128, two to a CU, 152).  Fitted to f32 contractions of 100 to 8192 a side in three layouts,
    //   within a tenth.  (Both operands K-inner: 128 x 128 tiles on the two-group kernel, which holds its CU alone,
    //   and six stages of 64 x 32 tiles, two to a CU.)
    //   64 x 128 tiles, and an operand that is not K-inner: the figures of eight waves to a work-group (two_waves_a_simd, gemm_launch.cuh); two and
    //   three work-groups of 64 x 32 that start together share a CU no better than `pair` (1024^3, 512 of them: 46 us; two splits
    //   of 64 x 128 31; 6000 x 100 x 500 24.8 / 17.9; 4096 x 512 x 784 40.7 -> 35.3; 2048^3 152 -> 144, both K-outer 160 -> 150).
    struct Tile { int cfg, rows, cols, resident; double alone, pair, shared; };
    const bool kk = l_kin && r_kin, oo = !l_kin && !r_kin, f64 = l_dt == HIPNX_F64;
    const Tile tiles[3] = {
        {GEMM_CFG_128, 128, 128, f64 || kk ? 1 : 2, f64 ? 2.6 : kk ? 2.05 : 2.25, 0, f64 ? 2.6 : kk ? 2.05 : 2.15},
        {GEMM_CFG_64x128, 64, 128, f64 ? 1 : 3, f64 ? 1.3 : 1.25, 0, f64 ? 1.3 : kk || oo ? 1.15 : 1.12},
        {GEMM_CFG_64, 64, 32, f64 ? 1 : kk ? 2 : 6, f64 ? 0.55 : kk ? 0.75 : 0.9, f64 || kk ? 0 : 1.38, f64 ? 0.55 : kk ? 0.65 : 0.36}};
    if (cfg == GEMM_CFG_128) {
      const int64_t cus = num_cus;
      double best = 0;
      for (const Tile &t : tiles) {
        const int64_t count = ((M + t.rows - 1) / t.rows) * ((N + t.cols - 1) / t.cols) * batch;
        for (int cand : {1, 2, 3, 4, 6, 8, 12, 16, 24, 32, 48, 64}) {
          if (cand > 1 && (!splittable || t.cfg == GEMM_CFG_64 || count * cand > t.resident * cus || nslab / cand < 2 || !reaches(cand))) continue;
          const int64_t per_cu = (count * cand + cus - 1) / cus, last = per_cu % t.resident;
          double us = (double)per_split(cand) * ((double)(per_cu - last) * t.shared + (last ? std::max(last > 1 && last == per_cu ? std::max(t.alone, t.pair) : t.alone, (double)last * t.shared) : 0.0));
          // a split's second launch, then the partial results written and read once (mostly from cache: ~8 MB per us)
          if (cand > 1) us += 5.0 + 2.0 * (double)cand * (double)(M * N) * 4.0 / 8.0e6;
          if (best == 0 || us < best) { best = us; cfg = t.cfg; splits = cand; }
        }
      }
    }
  } else if (l_kin && (two_byte || l_dt == HIPNX_S8) && (cfg == GEMM_CFG_128 || cfg == GEMM_CFG_64)) {
    // The cheapest tile and number of ranges of K.  A work-group (`resident` of them share a CU) takes `slab` us a slab, up to `fill` more by how
    // many of its rows there are (those past the edge are the last one read again), `off` more where rows do not begin on cache lines, and up to
    // `press` more by how much of the chip walks at once (what work-groups share is the way from L2 and beyond); `base` is a launch with an
    // empty walk, `round` what a further round of work-groups costs beside its slabs, `stream` a megabyte of the operands from memory; a second
    // launch adds the ranges' partial results, written and read once (`second`, and `megabyte` of them).  Fitted to 885 contractions of 1 to
    // 4000 rows, each under up to 25 tiles and ranges (profiles/dot_tile_choice.md): of what is within a third of the best, within a thirteenth in the
    // middle, the ninth decile within a fifth (int8 a third).  The choice takes 1.6 % longer than the best of them in the geometric mean; without `fill`, `press`
    // and `stream` 3.6 %, as full grids that stream long weights were taken to go as fast as a lone work-group.  us per call, by thresholds (128 x 128
    // tiles in up to sixteen ranges; 64 rows and fewer: 64 x 64) / without the three / so: bf16 128 x 11008 x 4096 24.2 / 29.6 / 24.4, 200 x 4000 x 4000
    // 18.5 / 22.9 / 18.7, 96 x 4096 x 4096 with K-outer weights 18.5 / 20.7 / 16.6; 500^3 10.3 / 6.0 / 6.0, 1000^3 10.9 / 6.8 / 6.8, 168 x 4000 x 1600 13.7 / 8.8 / 8.8;
    // int8 256 x 1024 x 8192 31.2 / 11.6 / 11.6.
    struct Tile { int cfg, rows, cols, resident; double base, round, slab, fill, off, press, stream, second, megabyte; };
    static const Tile table[4][3] = {
        {{GEMM_CFG_128, 128, 128, 1, 4.688, 1.675, 0.198, 0.106, 0.118, 0.254, 0.02, 3.086, 0.139},
         {GEMM_CFG_64, 64, 64, 1, 4.267, 1.392, 0.076, 0.064, 0.069, 0.084, 0.023, 2.517, 0.115},
         {GEMM_CFG_64x128, 64, 128, 1, 4.281, 1.335, 0.158, 0.086, 0.104, 0.103, 0.057, 2.768, 0.174}},
        {{GEMM_CFG_128, 128, 128, 1, 5.053, 1.319, 0.298, 0.068, 0.085, 0.176, 0.039, 2.945, 0.158},
         {GEMM_CFG_32x128, 32, 128, 2, 4.26, 0.213, 0.22, 0.033, 0.067, 0.126, 0.096, 2.134, 0.219},
         {GEMM_CFG_64x128, 64, 128, 1, 4.606, 1.736, 0.24, 0.055, 0.074, 0.083, 0.059, 2.583, 0.174}},
        {{GEMM_CFG_128, 128, 128, 1, 10.243, 2.339, 0.071, 0.2, 0.22, 0.27, 0.0, 0.0, 0.139},
         {GEMM_CFG_64, 64, 64, 1, 5.258, 2.102, 0.029, 0.102, 0.114, 0.067, 0.011, 2.052, 0.121},
         {GEMM_CFG_64x128, 64, 128, 1, 7.512, 2.258, 0.066, 0.128, 0.193, 0.175, 0.033, 0.265, 0.145}},
        {{GEMM_CFG_128, 128, 128, 1, 8.651, 3.069, 0.222, 0.159, 0.187, 0.147, 0.047, 0.0, 0.141},
         {GEMM_CFG_64, 64, 64, 1, 4.808, 2.171, 0.07, 0.074, 0.134, 0.102, 0.167, 2.164, 0.065},
         {GEMM_CFG_64x128, 64, 128, 1, 6.975, 3.166, 0.165, 0.084, 0.153, 0.179, 0.077, 0.615, 0.113}}};
    const Tile *tiles = table[(two_byte ? 0 : 2) + (r_kin ? 0 : 1)];
    const double off = K * esz % 128 ? 1.0 : 0.0, operands = (double)batch * (double)(M + N) * (double)K * esz / 1e6, results = (double)(M * N) * 8.0 / 1e6;
    double counts[3], slabs[3], best = 0;
    for (int i = 0; i < 3; i++) {
      const Tile &t = tiles[i];
      counts[i] = (double)(((M + t.rows - 1) / t.rows) * ((N + t.cols - 1) / t.cols) * batch);
      slabs[i] = t.slab + t.fill * (double)std::min<int64_t>(M, t.rows) / t.rows + off * t.off;
    }
    const int most = batch == 1 && partials ? (int)std::min<int64_t>(16, nslab / 2) : 1;
    double least = 0;  // what a second launch makes any of them take
    for (int i = 0; i < 3; i++) least = i ? std::min(least, tiles[i].base + tiles[i].second) : tiles[i].base + tiles[i].second;
    for (int cand = 1; cand == 1 || (cand <= most && best > least); cand++) {
      const int64_t per = per_split(cand);
      if (per * (cand - 1) >= nslab) continue;  // (every range has a slab)
      for (int i = 0; i < 3; i++) {
        const Tile &t = tiles[i];
        const double groups = counts[i] * cand, at_once = (double)(t.resident * num_cus);
        const double rounds = (double)(int64_t)((groups + at_once - 1) / at_once);  // (whole numbers: the quotient is not rounded past one)
        double us = t.base + t.round * (rounds - 1) + (double)per * (rounds * slabs[i] + t.press * groups / (double)num_cus) + t.stream * operands;
        if (cand > 1) us += t.second + t.megabyte * cand * results;
        if (best == 0 || us < best) { best = us; cfg = t.cfg; splits = cand; }
      }
    }
  } else if (splittable && t128 * 2 <= num_cus && nslab >= (t128 * 4 <= num_cus ? 32 : 64))
    // (the second pass and the partial results cost about 10 us: worth it from K = 32 slabs on -- 64 where
    // the grid already covers more than a quarter of the CUs -- with at least 8 slabs left per split and no
    // more work-groups than CUs; 1024 x 2048 x 2048, 128 tiles of 32 slabs, is faster whole: 21 us against
    // 22 us in two halves and 27 us in four quarters)
    for (int cand = 16; cand >= 2; cand /= 2)
      if (t128 * cand <= num_cus && nslab / cand >= 8 && reaches(cand)) { splits = cand; break; }
  const int rows = cfg == GEMM_CFG_256 || cfg == GEMM_CFG_256x128 ? 256 : cfg == GEMM_CFG_32x128 ? 32 : cfg == GEMM_CFG_64 || cfg == GEMM_CFG_64x128 ? 64 : 128;
  const int cols = cfg == GEMM_CFG_256 ? 256 : cfg == GEMM_CFG_64 ? 64 : cfg == GEMM_CFG_128x32 ? 32 : 128;
  return {cfg, splits, rows, cols};
}

// Whether a K-inner operand is copied to rows of whole pieces though the kernels take its rows as they lie.  Sixteen bytes at an
// address that is no multiple of four cost a CU three times its intake of aligned ones (measured from L2: 30 TB/s aligned, 18
// with rows on any multiple of four -- never worth a copy --, 15 on any multiple of two, 11.7 on any byte), which a tile pays per
// slab where its multiplications do not cover it; a copy costs a launch and reads and writes the operand once.  So the
// operand that many tiles re-read is copied, the long one that few do is not.  us per call, both copied / neither / by this rule:
// int8 512 x 11007 x 11005 142 / 157 / 119, 512 x 1001 x 11006 56 / 66 / 53, 128 x 11007 x 4094 43 / 32 / 29; bf16 168 x 4000 x 1597
// 25.3 / 25.7 / 21.1.
static inline bool rows_worth_copying(int64_t num_cus, const GemmChoice &c, int64_t batch, int64_t M, int64_t N, int64_t row_bytes, bool right) {
  if (row_bytes % 4 == 0) return false;
  const int64_t groups = ((M + c.rows - 1) / c.rows) * ((N + c.cols - 1) / c.cols) * batch * c.splits;
  const int64_t slabs = ((row_bytes + SLAB - 1) / SLAB + c.splits - 1) / c.splits;
  const double intake = 78e3, flops = 7.8e6;  // bytes and 2-byte multiply-adds x 2 a CU takes per us
  const double aligned = (double)(c.rows + c.cols) * SLAB / intake, side = (double)(right ? c.cols : c.rows) * SLAB / intake * (row_bytes % 2 ? 1.4 : 0.85);
  const double work = (double)c.rows * c.cols * SLAB / flops;
  const double extra = (double)((groups + num_cus - 1) / num_cus) * (double)slabs * std::max(0.0, aligned + side - std::max(aligned, work));
  const double copy = 2.5 + (double)batch * (double)(right ? N : M) * (double)row_bytes * 2.0 / 4.5e6;
  return extra > copy;
}

// What exists of the last slab of K: bytes of each row of a K-inner operand, k of a K-outer one; 0, the slab is whole and walked as every other.
// ragged: an operand is K-outer with k-rows that are not whole pieces.  The end of its last k-row, behind which there may be nothing, is
// read with care, which the kernels do for a partial slab only: a whole last slab is walked as one.  copied: to rows of whole pieces.
static inline int gemm_tail(int64_t row_bytes, int esz, bool ragged, bool k_inner, bool copied) {
  const int64_t over = row_bytes % SLAB, last = over == 0 && ragged ? SLAB : over;
  return (int)(!k_inner ? last / esz : copied ? (last + 15) / 16 * 16 : last);
}

}  // namespace hipnx
