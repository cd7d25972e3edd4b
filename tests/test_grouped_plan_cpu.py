"""The grouped call's plan (csrc/mer_grouped_plan.hpp), compiled and run on
the CPU: a call that is no larger than another in any size needs no more
scratch, so it never makes a workspace grow that served the larger one, and
every region and K part lies inside what was asked for.  The kernel chosen is
the one that was measured to be the faster."""
from __future__ import annotations

import os
import shutil
import subprocess

import pytest

from conftest import PKG_NAME, ROOT
from grouped_f16_cases import LONG_ROWS, LONG_ROWS_QMM, MANY

CSRC = os.path.join(ROOT, PKG_NAME, "csrc")

MAIN = r"""
#include "mer_grouped_plan.hpp"
#include <stdio.h>
using namespace mer;
static int bad = 0;
#define CHECK(c) do { if (!(c) && bad++ < 20) printf("line %d: %s (dm %zu dff %zu tok %u k %u table %u q8 %d)\n", __LINE__, #c, dm, dff, tok, k, tab, (int)q8); } while (0)
int main() {
  const size_t dims[] = {64, 512, 2048, 4032, 4096, 4160, 7168, 8192, 14336, 16384};
  const uint32_t toks[] = {1, 15, 16, 17, 63, 64, 65, 333, 511, 512, 1023, 1024, 1727, 1728, 1791, 1792, 1888, 1920, 2048, 3776, 3840, 4096};
  const uint32_t tabs[] = {1, 2, 7, 8, 60, 64, 128, 256, 1024, 4096};
  const uint32_t ks[] = {1, 2, 8};
  const unsigned nd = sizeof dims / sizeof *dims, nt = sizeof toks / sizeof *toks, ne = sizeof tabs / sizeof *tabs;
  unsigned long n = 0, split = 0, big = 0;
  for (unsigned a = 0; a < nd; ++a) for (unsigned b = 0; b < nd; ++b) for (unsigned c = 0; c < nt; ++c)
    for (unsigned d = 0; d < 3; ++d) for (unsigned e = 0; e < ne; ++e) for (int q = 0; q < 3; ++q) {
      const size_t dm = dims[a], dff = dims[b];
      const uint32_t tok = toks[c], k = ks[d], tab = tabs[e];
      const bool q4 = q < 2, q8 = q == 1;
      if (tok * k > kMaxGroupedPairs) continue;
      const GroupedPlan p = plan_grouped(q4, q8, dm, dff, tok, k, tab);
      const size_t pairs = tok * k, one = pairs * dm, hb = dff / 32;
      ++n; split += p.n_parts > 1; big += p.mode != kGroupDigits;
      CHECK(p.plist >= 64 && p.pair_ok >= p.plist + pairs && p.tiles >= p.pair_ok + pairs);
      CHECK(p.xg >= p.tiles + p.max_tiles * sizeof(GroupTile) / 4);
      CHECK(p.hg >= p.xg + tok * dm && p.xs >= p.hg + pairs * dff && p.hs >= p.xs + tok && p.partial >= p.hs + pairs);
      CHECK(p.need >= p.partial + one && p.want >= p.partial + p.n_parts * one);
      CHECK((p.plist | p.pair_ok | p.tiles | p.xg | p.hg | p.xs | p.hs | p.partial) % 64 == 0);
      CHECK(p.n_parts >= 1 && p.n_parts <= 4 && (p.n_parts == 1 || p.mode != kGroupDigits));
      CHECK((p.n_parts - 1) * p.part_blocks < hb && p.n_parts * p.part_blocks >= hb);
      CHECK(p.n_parts == 1 || p.part_blocks % 4 == 0);
      // no more than the records, lists and one part of sums take in any mode
      CHECK(p.need <= 64 + 3 * pairs + 4 * (pairs / 16 + (pairs < tab ? pairs : tab)) + tok * dm + pairs * dff + one + tok + 8 * 63);
      GroupedPlan small = p;  // what a scratch of `need` floats serves
      fit_parts(small, (uint32_t)pairs, dm, dff, p.need);
      CHECK(small.n_parts == 1 && small.part_blocks == hb);
      // each size one step up, alone
      auto le = [&](size_t m, size_t f, uint32_t t, uint32_t kk, uint32_t l, bool qq) {
        const GroupedPlan g = plan_grouped(q4, qq, m, f, t, kk, l);
        CHECK(p.need <= g.need && p.want <= g.want);
      };
      if (a + 1 < nd) le(dims[a + 1], dff, tok, k, tab, q8);
      if (b + 1 < nd) le(dm, dims[b + 1], tok, k, tab, q8);
      if (c + 1 < nt && toks[c + 1] * k <= kMaxGroupedPairs) le(dm, dff, toks[c + 1], k, tab, q8);
      if (d + 1 < 3 && tok * ks[d + 1] <= kMaxGroupedPairs) le(dm, dff, tok, ks[d + 1], tab, q8);
      if (e + 1 < ne) le(dm, dff, tok, k, tabs[e + 1], q8);
      if (q4) le(dm, dff, tok, k, tab, !q8);
    }
  printf("%lu plans, %lu with K parts, %lu with 64-pair tiles, %d failures\n", n, split, big, bad);
  return bad || !split || !big;
}
"""


@pytest.fixture(scope="module")
def run_plan(tmp_path_factory):
    gxx = shutil.which("g++")
    if not gxx:
        pytest.skip("g++ not available")

    def run(main):
        d = tmp_path_factory.mktemp("plan")
        (d / "plan.cpp").write_text(main)
        r = subprocess.run([gxx, "-std=c++17", "-O1", "-Wall", "-Wextra", "-Werror", "-I", CSRC, str(d / "plan.cpp"),
                            "-o", str(d / "plan")], capture_output=True, text=True)
        assert r.returncode == 0, r.stderr[-2000:]
        out = subprocess.run([str(d / "plan")], capture_output=True, text=True, timeout=300)
        return out.returncode, out.stdout

    return run


def test_scratch_regions_and_growth(run_plan):
    rc, out = run_plan(MAIN)
    assert rc == 0, out


CHOICE = r"""
#include "mer_grouped_plan.hpp"
#include <stdio.h>
#include <stdlib.h>
int main(int argc, char **argv) {
  for (int i = 1; i + 6 < argc; i += 7) {
    const mer::GroupedPlan p = mer::plan_grouped(atoi(argv[i]) == 4, atoi(argv[i + 1]) != 0, atoi(argv[i + 2]), atoi(argv[i + 3]),
                                                 atoi(argv[i + 4]), atoi(argv[i + 5]), atoi(argv[i + 6]));
    printf("%d", p.mode == mer::kGroupDigits ? 0 : (int)p.n_parts);
  }
  return 0;
}
"""

# dtype, qmm, d_model, d_ff, tokens, top_k, experts -> int8 / f16 us measured on
# routes picked at random (z: with a Zipf exponent); only where the two differ
# by more than runs do
MEASURED = [
    ((4, 0, 7168, 2048, 256, 8, 256), 2043, 1943),
    ((4, 0, 7168, 2048, 512, 8, 256), 2806, 2066),
    ((4, 1, 7168, 2048, 256, 8, 256), 1985, 2122),
    ((4, 1, 7168, 2048, 320, 8, 256), 2063, 2142),
    ((4, 1, 7168, 2048, 512, 8, 256), 2694, 2227),
    ((5, 0, 7168, 2048, 256, 8, 256), 2870, 3069),
    ((5, 0, 7168, 2048, 512, 8, 256), 3745, 3229),
    ((4, 1, 4096, 14336, 32, 2, 8), 277, 324),
    ((4, 1, 4096, 14336, 64, 2, 8), 409, 334),
    ((5, 0, 4096, 14336, 48, 2, 8), 371, 429),
    ((5, 0, 4096, 14336, 96, 2, 8), 610, 463),
    ((5, 0, 2048, 768, 192, 8, 128), 189, 217),
    ((5, 0, 2048, 768, 320, 8, 128), 272, 224),
    ((4, 1, 2048, 768, 320, 8, 128), 208, 169),
    ((4, 1, 4096, 4096, 128, 4, 64), 557, 646),
    ((5, 0, 4096, 4096, 256, 4, 64), 1065, 935),
    ((4, 0, 8192, 8192, 96, 4, 32), 1265, 1165),
    ((5, 0, 4096, 1536, 48, 1, 1), 46, 137),
    ((5, 0, 4096, 384, 235, 1, 4), 43, 119),         # z 0.9
    ((4, 0, 3264, 1152, 41, 2, 2), 41, 106),
    ((4, 1, 1088, 960, 64, 1, 1), 26, 67),
    ((5, 0, 832, 384, 218, 1, 1), 23, 52),
    ((4, 1, 4096, 896, 16, 4, 4), 40, 91),
    ((4, 0, 1600, 448, 272, 1, 8), 33, 67),          # z 0.8
    ((4, 0, 704, 512, 57, 4, 8), 24, 47),
    ((4, 0, 1152, 3968, 114, 3, 19), 119, 149),      # z 1.0
    ((5, 0, 512, 13760, 17, 2, 2), 134, 73),
    ((5, 0, 1280, 10176, 20, 2, 2), 118, 73),
    ((4, 0, 1280, 6784, 410, 3, 128), 666, 527),     # z 0.7
]


@pytest.fixture(scope="module")
def choice(tmp_path_factory):
    """Sizes -> K parts of the f16 kernel, 0 for the int8 kernel."""
    gxx = shutil.which("g++")
    if not gxx:
        pytest.skip("g++ not available")
    d = tmp_path_factory.mktemp("choice")
    (d / "choice.cpp").write_text(CHOICE)
    subprocess.run([gxx, "-std=c++17", "-I", CSRC, str(d / "choice.cpp"), "-o", str(d / "choice")], check=True)

    def ask(cases):
        r = subprocess.run([str(d / "choice"), *[str(v) for c in cases for v in c]], check=True, capture_output=True, text=True)
        assert len(r.stdout) == len(cases)
        return [int(c) for c in r.stdout]

    return ask


def test_kernel_choice_is_the_faster_one(choice):
    got = choice([m[0] for m in MEASURED])
    wrong = [m for m, parts in zip(MEASURED, got) if (parts > 0) != (m[2] < m[1])]
    assert not wrong, wrong


def test_sizes_of_the_f16_tests_run_f16(choice):
    cases = LONG_ROWS + LONG_ROWS_QMM + MANY
    wrong = [(c, parts) for c, parts in zip(cases, choice([c[:7] for c in cases])) if parts != c[7]]
    assert not wrong, wrong
