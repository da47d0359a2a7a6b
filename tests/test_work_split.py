"""The index arithmetic of flexmm_amd/csrc/work_split.h, compiled by the host
compiler: the parts of a range are consecutive, cover it and differ in length
by at most one, up to ranges of 2^31 - 1."""
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
