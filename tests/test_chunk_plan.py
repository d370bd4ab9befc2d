"""The key-range split planner of the chunk kernels (ellm_amd/csrc/chunk_plan.hpp, host code) against an
exact simulation of the dispatch it models: workgroups dealt in id order to the free slot that
opens first."""
import os
import shutil
import subprocess

import pytest

import plan_probe

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "ellm_amd", "csrc")

PROBE = r"""
#include "chunk_plan.hpp"
#include <algorithm>
#include <cstdio>
#include <vector>
using namespace ellm;
static uint64_t simulate(uint32_t items, uint32_t slots, uint32_t len, uint32_t n, uint32_t rest) {
  std::vector<uint64_t> free_at(slots, 0);
  uint64_t end = 0;
  for (uint32_t s = 0; s < n; ++s)
    for (uint32_t i = 0; i < items; ++i) {
      auto it = std::min_element(free_at.begin(), free_at.end());
      *it += (s == n - 1) ? rest : len;
      end = std::max(end, *it);
    }
  return end;
}
int main() {
  const uint32_t tiles_set[] = {1, 7, 16, 17, 33, 64, 129, 130, 513, 2048};
  const uint32_t items_set[] = {1, 4, 8, 16, 24, 96, 128, 192, 255, 256, 300};
  const uint32_t slots_set[] = {256, 512};
  const uint32_t max_set[] = {1, 2, 5, 64, 4096};
  const double cost_set[] = {0.0, 0.1, 1.0, 6.7};
  for (uint32_t tiles : tiles_set) for (uint32_t items : items_set) for (uint32_t slots : slots_set)
  for (uint32_t max_split : max_set) for (double cost : cost_set) for (uint32_t min_tiles : {4u, 8u}) {
    const KeySplit k = plan_key_split(tiles, items, slots, min_tiles, max_split, cost);
    const uint32_t rest = tiles - (k.n_split - 1) * k.split_tiles;
    const KeySplit again = plan_key_split(tiles, items, slots, min_tiles, max_split, cost);
    printf("%u %u %u %u %u %g %u %u %u %llu %llu %llu %u %u\n", tiles, items, slots, min_tiles, max_split, cost,
           k.split_tiles, k.n_split, rest,
           (unsigned long long)key_split_makespan(items, slots, k.split_tiles, k.n_split, rest),
           (unsigned long long)simulate(items, slots, k.split_tiles, k.n_split, rest),
           (unsigned long long)simulate(items, slots, tiles, 1, tiles), again.split_tiles, again.n_split);
  }
  return 0;
}
"""


@pytest.fixture(scope="module")
def rows(tmp_path_factory):
    gxx = shutil.which("g++")
    if not gxx:
        pytest.skip("no g++")
    d = tmp_path_factory.mktemp("plan")
    src = d / "probe.cpp"
    src.write_text(PROBE)
    exe = d / "probe"
    subprocess.run([gxx, "-O2", "-std=c++17", "-I", CSRC, str(src), "-o", str(exe)], check=True, timeout=300)
    out = subprocess.run([str(exe)], check=True, capture_output=True, text=True, timeout=300).stdout
    return [[float(x) for x in line.split()] for line in out.splitlines()]


def test_plans_are_well_formed(rows):
    assert len(rows) > 1000
    for tiles, items, slots, min_tiles, max_split, cost, length, n, rest, est, sim, unsplit, l2, n2 in rows:
        assert 1 <= n <= max(max_split, 1)
        assert (n - 1) * length + rest == tiles and 1 <= rest <= length     # the pieces tile the walk, the last is the short one
        assert n == 1 or length >= min_tiles
        assert (l2, n2) == (length, n)                                       # the memo returns the same answer


def test_estimate_never_undershoots_the_simulated_dispatch_by_much(rows):
    """The closed form is what the planner minimises; it must track the simulation: never below it
    (it would pick plans that look better than they are) beyond one short piece, and within one long
    piece above."""
    for tiles, items, slots, min_tiles, max_split, cost, length, n, rest, est, sim, unsplit, l2, n2 in rows:
        assert est + rest >= sim, (tiles, items, slots, length, n, est, sim)
        assert est <= sim + length, (tiles, items, slots, length, n, est, sim)


def test_a_split_is_only_chosen_when_it_pays(rows):
    for tiles, items, slots, min_tiles, max_split, cost, length, n, rest, est, sim, unsplit, l2, n2 in rows:
        if n > 1:
            assert est + n * cost < unsplit, (tiles, items, slots, cost, length, n, est, unsplit)


def test_known_shapes(rows):
    """24 sequences x 4 kv heads on 8192 keys (129 tiles): the twelve-wave kernel (one workgroup a unit)
    gets two long pieces and a short one per plane; with twice the slots the plan is five equal pieces."""
    by = {(r[0], r[1], r[2], r[3], r[4], r[5]): r for r in rows}
    r = by[(129, 96, 256, 4, 5, 1.0)]
    assert (r[6], r[7], r[8]) == (52, 3, 25) and r[10] == 52
    r = by[(129, 96, 512, 4, 64, 1.0)]
    assert (r[6], r[7]) == (26, 5)


def test_the_chunk_cases_reach_the_kernels_they_are_there_for():
    from test_gpu_parity import PREFILL, kernel_of

    seen = set()
    for name, bcap, b, hq, hkv, cap, p0, s in PREFILL:
        kernel, waves, n_split, _ = plan_probe.chunk_plan(bcap, b, hq, hkv, p0, s)
        want, want_waves = kernel_of(name)
        assert kernel == want and (want_waves is None or waves == want_waves), (name, kernel, waves)
        seen.add((kernel, waves, n_split > 1))
    assert seen >= {("stream", w, True) for w in (4, 8, 12)} | {("stream", 4, False), ("pingpong", 0, True), ("pingpong", 0, False),
                                                               ("short", 1, False), ("short", 2, False)}


def test_tiles_go_straight_to_lds_in_unsplit_tile_walks_of_4096_keys_and_more():
    direct, plan = plan_probe.chunk_is_direct, plan_probe.chunk_plan
    for b, hq, hkv, s in ((25, 64, 1, 9), (25, 32, 4, 49), (3, 32, 4, 600), (26, 32, 4, 64)):
        for keys, want in ((4095, False), (4096, True), (4097, True), (131072, True)):
            assert plan(b, b, hq, hkv, keys - s, s)[:3] == ("pingpong", 0, 1)
            assert direct(b, b, hq, hkv, keys - s, s) == want, (b, hq, hkv, s, keys)
    assert plan(1, 1, 32, 4, 8192, 64)[0] == "pingpong" and plan(1, 1, 32, 4, 8192, 64)[2] > 1 and not direct(1, 1, 32, 4, 8192, 64)
    assert plan(24, 24, 32, 4, 8191, 13)[0] == "stream" and not direct(24, 24, 32, 4, 8191, 13)


def test_walks_of_129_to_192_workgroups_are_cut_in_two_where_that_is_faster():
    """Five of eight units of a shader engine busy: the second pieces run in two rounds on the other three; six:
    in three rounds on two.  Not where the partial rows cost more than that gives, nor with most units busy."""
    plan = plan_probe.chunk_plan
    for s, p0, pieces in ((1030, 4100, 2), (1030, 30000, 2), (1167, 12000, 2), (1344, 4100, 2), (1344, 12000, 2), (1536, 12000, 2),
                          (1536, 4100, 2),
                          (1030, 1000, 1), (1480, 2000, 1), (1537, 30000, 1)):
        assert plan(1, 1, 32, 4, p0, s)[:3] == ("pingpong", 0, pieces), (s, p0)
    assert plan(18, 18, 32, 4, 4096, 64)[2] == 1 and plan(18, 18, 32, 4, 8192, 64)[2] == 2    # 99 us against 96, 184 against 190
    assert plan(1, 1, 64, 8, 4100, 660)[2] == 1 and plan(1, 1, 64, 8, 12000, 660)[2] == 2     # 111 against 109, 262 against 272
    assert plan(1, 1, 8, 1, 0, 5000)[2] == 2
    assert plan(40, 1, 32, 4, 12000, 1536, most=1536)[2] == 1                                 # no room for the partial rows


def test_short_walks_that_leave_units_idle_run_on_32x32x16():
    form, plan = plan_probe.chunk_form, plan_probe.chunk_plan
    for bf16, want in ((True, "wide"), (False, "registers")):
        assert form(1, 1, 32, 4, 1400, 1536, bf16=bf16) == want                               # units busy for 0.57 of the time
        assert form(19, 19, 32, 4, 1200, 64, bf16=bf16) == want                               # 49 MB of K and V
    for bf16 in (True, False):
        assert form(1, 1, 32, 4, 1000, 1200, bf16=bf16) == "wide"                             # 0.47
        assert form(1, 1, 32, 4, 700, 2048, bf16=bf16) == "registers"                         # 0.64
        assert form(22, 22, 32, 4, 2000, 64, bf16=bf16) == "registers"                        # 93 MB
        assert form(1, 1, 32, 4, 4100, 1600, bf16=bf16) == "direct"
        assert plan(1, 1, 8, 1, 0, 4000)[2] == 2 and form(1, 1, 8, 1, 0, 4000, bf16=bf16) == "wide"           # cut in two, 0.37
        assert plan(1, 1, 32, 4, 2000, 300)[2] > 2 and form(1, 1, 32, 4, 2000, 300, bf16=bf16) == "wide"     # pieces of 9 tiles, 0.59
        assert plan(1, 1, 32, 4, 6000, 300)[2] > 2 and form(1, 1, 32, 4, 6000, 300, bf16=bf16) == "registers"
