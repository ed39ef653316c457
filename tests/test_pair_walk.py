"""The walk over two runs' particle pairs (fof_pairwalk.h), compiled for the
host: every lane visits its pairs in order and all of them, where the number
of pairs passes 2^32 too."""
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "cm_halofinder_amd", "csrc")

# Per pair of sizes: lanes first .. 15 in steps of `lanes`, the pair's number
# rebuilt in 64 bits.
MAIN = r"""
#include "fof_pairwalk.h"
#include <cstdio>
#include <cstdlib>
int main(int c, char **v) {
  const uint32_t m1 = strtoul(v[1], 0, 10), m2 = strtoul(v[2], 0, 10), lanes = strtoul(v[3], 0, 10);
  const uint64_t total = (uint64_t)m1 * m2;
  for (uint32_t q = 0; q < fof::kPairLanes; q += lanes) {
    uint64_t at = q;
    fof::PairWalk p(q, m2);
    for (; p.i < m1; p.step(), at += fof::kPairLanes)
      if (p.j >= m2 || (uint64_t)p.i * m2 + p.j != at) return printf("lane %u at %llu\n", q, (unsigned long long)at), 1;
    if (at < total) return printf("lane %u ends at %llu\n", q, (unsigned long long)at), 1;
  }
  return 0;
}
"""


@pytest.fixture(scope="module")
def walk(tmp_path_factory):
    d = tmp_path_factory.mktemp("walk")
    (d / "main.cpp").write_text(MAIN)
    subprocess.run(["g++", "-O2", "-std=c++17", "-I", CSRC, str(d / "main.cpp"), "-o", str(d / "walk")], check=True)
    return lambda *a: subprocess.run([str(d / "walk"), *map(str, a)], capture_output=True, text=True, timeout=100)


def test_every_small_pair(walk):
    for m1 in (1, 2, 3, 5, 15, 16, 17, 40):
        for m2 in (1, 2, 3, 5, 15, 16, 17, 33):
            r = walk(m1, m2, 1)
            assert r.returncode == 0, (m1, m2, r.stdout)


@pytest.mark.parametrize("m1,m2", [(65536, 65536), (65537, 65536), (3, 1 << 31), (1 << 31, 3)])
def test_pairs_beyond_2_32(walk, m1, m2):
    r = walk(m1, m2, 15)  # the first lane and the last
    assert r.returncode == 0, r.stdout
