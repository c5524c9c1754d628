"""The rule of a contraction's tile and ranges of K (nx_amd/csrc/gemm_choice.h), compiled for the host, against the
times measured under every choice (profiles/dot_tile_choice.md)."""
import math
import re
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent
RANGES = [1, 2, 3, 4, 5, 6, 8, 10, 12, 16]
TILES = ["128 x 128", "64 x 64", "64 x 128", "32 x 128"]
CFG = {1: "128 x 128", 2: "64 x 64", 4: "64 x 128", 6: "32 x 128"}
PROGRAM = r"""
#include "%s"
#include <cstdio>
using namespace hipnx;
int main() {
  long long two, kin, M, N, K, batch;
  while (scanf("%%lld %%lld %%lld %%lld %%lld %%lld", &two, &kin, &batch, &M, &N, &K) == 6) {
    const GemmChoice c = gemm_choice(256, two ? HIPNX_BF16 : HIPNX_S8, batch, M, N, K, true, kin != 0, batch == 1);
    printf("%%d %%d\n", c.cfg, c.splits);
  }
}
"""


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    d = tmp_path_factory.mktemp("choice")
    (d / "choice.cpp").write_text(PROGRAM % (ROOT / "nx_amd" / "csrc" / "gemm_choice.h"))
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-o", str(d / "choice"), str(d / "choice.cpp")], check=True)

    def ask(lines):
        out = subprocess.run([str(d / "choice")], input="\n".join(" ".join(map(str, q)) for q in lines), capture_output=True, text=True, check=True)
        return [tuple(map(int, x.split())) for x in out.stdout.splitlines()]
    return ask


def measured():
    for line in (ROOT / "profiles" / "dot_tile_choice.md").read_text().splitlines():
        cells = [c.strip() for c in line.strip("|").split("|")]
        m = re.match(r"(int8|bf16) (\d+) x (\d+) x (\d+)$", cells[0])
        if m:
            times = {(t, n): float(v) for t, cell in zip(TILES, cells[3:7]) for n, v in zip(RANGES, cell.split()) if v != "-"}
            yield m.group(1), cells[1] == "K-inner", *map(int, m.groups()[1:]), float(cells[2]), times


def time_of(times, tile, ranges):
    known = sorted(n for t, n in times if t == tile)
    low, high = max(n for n in known if n <= ranges), min((n for n in known if n >= ranges), default=max(known))
    a, b = times[tile, low], times[tile, high]
    return a if low == high else a + (b - a) * (ranges - low) / (high - low)


def test_the_choice_is_near_the_best_measured_one_and_no_slower_than_thresholds_were(rules):
    rows = list(measured())
    assert len(rows) > 100
    choices = rules([(int(t == "bf16"), int(kin), 1, M, N, K) for t, kin, M, N, K, _, _ in rows])
    apart = []
    for (t, kin, M, N, K, before, times), (cfg, ranges) in zip(rows, choices):
        us, best = time_of(times, CFG[cfg], ranges), min(times.values())
        # (two programs' loops took `before` and the others, 0.3 us a call apart; two runs of one differ by 2 %)
        assert us <= 1.03 * before + 0.4 and us <= 1.16 * best, (t, kin, M, N, K, CFG[cfg], ranges, us, best, before)
        apart.append(math.log(us / best))
    assert math.exp(sum(apart) / len(apart)) < 1.012


def test_ranges_have_slabs_and_are_whole_where_partial_results_are_not_kept(rules):
    """Any extents: the ranges are those that the launch takes (every one has a slab, two at least where there are several), and a batch has one."""
    sizes = [(M, N, K) for M in (1, 8, 33, 64, 65, 128, 300, 2000) for N in (8, 127, 128, 5000) for K in (1, 63, 64, 65, 200, 1000, 4097, 65536)]
    for two in (0, 1):
        for kin in (0, 1):
            one = rules([(two, kin, 1, *s) for s in sizes])
            for (M, N, K), (cfg, ranges) in zip(sizes, one):
                slabs = -(-K * (1 + two) // 128)
                per = -(-slabs // ranges)
                assert 1 <= ranges <= 16 and per * (ranges - 1) < slabs and (ranges == 1 or slabs >= 2 * ranges)
                assert cfg != 6 or (two and not kin)
            assert all(ranges == 1 for _, ranges in rules([(two, kin, 3, *s) for s in sizes]))
