"""The index arithmetic of flexmm_amd/csrc/work_split.h, compiled by the host
compiler: the parts of a range are consecutive, cover it and differ in length
by at most one, up to ranges of 2^31 - 1; the orders of blocks and evaluation
items over the XCDs take every one exactly once."""
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "flexmm_amd",
                    "csrc")

HARNESS = r"""
#include "work_split.h"
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <vector>
using namespace fmm;

template <int PARTS>
static int parts(int b, int e) {
  int at = b;
  const int64_t n = e > b ? (int64_t)e - b : 0;
  for (int k = 0; k < PARTS; ++k) {
    const Span s = part_of<PARTS>(b, e, k);
    const int64_t len = (int64_t)s.e - s.b;
    if (s.b != at || len < n / PARTS || len > n / PARTS + 1) {
      std::printf("part %d of %d of [%d, %d): [%d, %d)\n", k, PARTS, b, e, s.b, s.e);
      return 1;
    }
    at = s.e;
  }
  return (int64_t)at != b + n;
}

int main(int argc, char** argv) {
  if (argc == 4 && !std::strcmp(argv[1], "parts")) {
    const int b = std::atoi(argv[2]), e = std::atoi(argv[3]);
    return parts<1>(b, e) | parts<4>(b, e);
  }
  // every logical index once, and the neighbours of a chunk on one XCD
  if (argc == 4 && !std::strcmp(argv[1], "blocks")) {
    const int n = std::atoi(argv[2]), chunk = std::atoi(argv[3]);
    std::vector<int> xcd(n, -1);
    for (int b = 0; b < n; ++b) {
      const int l = xcd_block(b, n, chunk);
      if (l < 0 || l >= n || xcd[l] >= 0) return 1;
      xcd[l] = b % kNumXcd;
    }
    for (int l = 0; l + 1 < n; ++l) {
      if (chunk == 0 && xcd[l + 1] < xcd[l]) return 1;
      if (chunk > 0 && l < n / (kNumXcd * chunk) * (kNumXcd * chunk) && (l + 1) % chunk &&
          xcd[l + 1] != xcd[l])
        return 1;
    }
    return 0;
  }
  // every item by ns waves of one block, in any grid of at least its blocks
  if (argc == 6 && !std::strcmp(argv[1], "items")) {
    const int ni = std::atoi(argv[2]), icap = std::atoi(argv[3]), chunk = std::atoi(argv[4]),
              ns = std::atoi(argv[5]);
    std::vector<int> waves(ni, 0), block(ni, -1);
    for (int b = 0; b < eval_grid(icap, chunk, ns); ++b)
      for (int w = 0; w < kEvalWaves; ++w) {
        const int i = xcd_item(b, w, ni, chunk, ns);
        if (i < 0) continue;
        if (i >= ni || (ns > 1 && waves[i] && block[i] != b)) return 1;
        ++waves[i];
        block[i] = b;
        // a block whose waves share an item takes no other
        if (ns == kEvalWaves && i != xcd_item(b, 0, ni, chunk, ns)) return 1;
      }
    for (int i = 0; i < ni; ++i)
      if (waves[i] != ns) return 1;
    return 0;
  }
  if (argc == 9 && !std::strcmp(argv[1], "waves")) {
    const auto v = [&](int k) { return std::atoll(argv[k]); };
    std::printf("%d", item_waves(v(2), v(3), v(4), v(5), v(6), (int)v(7), v(8) != 0));
    return 0;
  }
  if (argc == 4 && !std::strcmp(argv[1], "broad")) {
    std::printf("%d", broad_sources(std::atoi(argv[2]), std::atoll(argv[3])));
    return 0;
  }
  if (argc == 4 && !std::strcmp(argv[1], "even_items")) {
    std::printf("%d", even_items(std::atoi(argv[2]), std::atoll(argv[3])));
    return 0;
  }
  return 2;
}
"""


@pytest.fixture(scope="module")
def harness(tmp_path_factory):
    d = tmp_path_factory.mktemp("work_split")
    (d / "h.cpp").write_text(HARNESS)
    exe = d / "h"
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-I" + CSRC,
                    str(d / "h.cpp"), "-o", str(exe)], check=True)
    return lambda *a: subprocess.run([str(exe)] + [str(v) for v in a], capture_output=True,
                                     text=True)


@pytest.mark.parametrize("b", [0, 1, 12345])
@pytest.mark.parametrize("n", [0, 1, 2, 3, 4, 5, 7, 8, 63, 64, 65, 1000, 2 ** 29 - 1, 2 ** 29,
                               2 ** 29 + 1, 715827883, 2 ** 30, 2 ** 30 + 3, 2 ** 31 - 2,
                               2 ** 31 - 1])
def test_parts_cover_the_range(harness, b, n):
    r = harness("parts", b, min(b + n, 2 ** 31 - 1))
    assert r.returncode == 0, r.stdout


def test_a_range_that_ends_before_it_begins_is_empty(harness):
    assert harness("parts", 5, 3).returncode == 0


COUNTS = [1, 7, 8, 31, 32, 33, 255, 256, 257, 1000, 4099]


@pytest.mark.parametrize("chunk", [0, 1, 4, 8, 32])
@pytest.mark.parametrize("n", COUNTS)
def test_block_order_is_a_bijection(harness, n, chunk):
    assert harness("blocks", n, chunk).returncode == 0


@pytest.mark.parametrize("ns", [1, 4])
@pytest.mark.parametrize("chunk", [0, 8, 32])
@pytest.mark.parametrize("n", COUNTS)
def test_items_are_taken_once(harness, n, chunk, ns):
    for icap in (n, n + 1, n + 65, 3 * n):
        assert harness("items", n, icap, chunk, ns).returncode == 0, icap


# 1000 evaluation boxes.  (items, targets per box, sources per box, S2M boxes,
# levels, self) -> waves per item; 1000 boxes of 6 levels: broad, not complete
@pytest.mark.parametrize("icap,per_box,per_leaf,n_up,levels,own,waves", [
    (1, 4, 1, 100, 20, 0, 4), (2048, 4, 0, 100, 20, 0, 4), (2048, 3, 500, 1000, 6, 1, 1),
    (2049, 9, 8, 1000, 6, 1, 1), (2049, 9, 9, 1000, 6, 1, 4), (16384, 9, 9, 100, 20, 1, 4),
    (2049, 9, 15, 100, 20, 0, 1), (4096, 9, 16, 100, 20, 0, 4),
    (4097, 9, 15, 1000, 6, 0, 1), (4097, 9, 16, 1000, 6, 0, 4), (4097, 9, 16, 205, 6, 0, 4),
    (4097, 9, 16, 204, 6, 0, 1), (4097, 9, 31, 1000, 20, 0, 1), (4097, 9, 32, 1000, 20, 0, 4),
    (4097, 9, 32, 500, 20, 0, 4), (4097, 9, 95, 499, 20, 0, 1), (4097, 9, 96, 499, 20, 0, 4),
    (4097, 9, 16, 2000, 20, 0, 1), (4097, 9, 32, 2000, 20, 0, 4),
    (16384, 9, 96, 100, 20, 0, 4), (16385, 9, 500, 1000, 6, 1, 1)])
def test_waves_per_item(harness, icap, per_box, per_leaf, n_up, levels, own, waves):
    n = per_leaf * min(n_up, 1000)
    r = harness("waves", icap, per_box * 1000, 1000, n, n_up, levels, own)
    assert r.returncode == 0 and int(r.stdout) == waves


@pytest.mark.parametrize("per_leaf,waves", [(31, 1), (32, 4)])
def test_complete_trees_need_more_sources(harness, per_leaf, waves):
    r = harness("waves", 4200, 9 * 4096, 4096, per_leaf * 4096, 4096, 7, 0)
    assert r.returncode == 0 and int(r.stdout) == waves


@pytest.mark.parametrize("levels,ne,even", [
    (1, 1, 1), (2, 4, 1), (2, 3, 0), (7, 4096, 1), (7, 4093, 1), (7, 4064, 1), (7, 4063, 0),
    (9, 65024, 1), (9, 65023, 0), (9, 61447, 0), (16, 4 ** 15, 1), (17, 4 ** 15, 0)])
def test_even_items(harness, levels, ne, even):
    r = harness("even_items", levels, ne)
    assert r.returncode == 0 and int(r.stdout) == even


@pytest.mark.parametrize("levels,n_up,broad", [
    (1, 1, 1), (2, 1, 1), (3, 3, 0), (3, 4, 1), (8, 4096, 1), (8, 3277, 1), (8, 3276, 0),
    (10, 4080, 0), (16, 4 ** 14, 1), (17, 4 ** 16, 0)])
def test_broad_sources(harness, levels, n_up, broad):
    r = harness("broad", levels, n_up)
    assert r.returncode == 0 and int(r.stdout) == broad
