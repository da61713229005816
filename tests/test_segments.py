"""The walks over a pair list's slots at the largest list there is (2^31 - 1):
constant expressions, so that an overflow or an endless walk does not compile."""
import os
import subprocess

import phafd_amd.build as B

SOURCE = r"""
#include <climits>
#include "segments.hpp"
using namespace phafd;
constexpr int M = INT_MAX;
// slots a walk of G lanes takes of [s, e), each lane until it is past the end
constexpr long long lanes(int s, int e, int G) {
  long long n = 0;
  for (int l = 0; l < G; l++) {
    LaneWalk w(s, e, l);
    while (w.on()) { n++; w.next(G); }
  }
  return n;
}
constexpr long long chunks(int s, int e, int most) {
  long long n = 0;
  for (int c = s, d = 0; c < e; c = d) {
    d = chunk_end(c, e, most);
    n += d - c;
  }
  return n;
}
static_assert(lanes(0, 0, 8) == 0 && lanes(5, 6, 8) == 1 && lanes(3, 40, 16) == 37);
static_assert(chunks(0, 0, 2048) == 0 && chunks(7, 2055, 2048) == 2048 && chunks(7, 2056, 2048) == 2049);
static_assert(lanes(M, M, 16) == 0 && lanes(M - 1, M, 16) == 1 && lanes(M - 7, M, 8) == 7 && lanes(M - 300, M, 16) == 300);
static_assert(chunks(M, M, 2048) == 0 && chunks(M - 1, M, 2048) == 1 && chunks(M - 2048, M, 2048) == 2048);
static_assert(chunks(M - 5000, M, 2048) == 5000);
"""


def test_walks_end_at_the_largest_slot(tmp_path):
    src = tmp_path / "limits.cpp"
    src.write_text(SOURCE)
    r = subprocess.run(["g++", "-std=c++17", "-fsyntax-only", "-I" + B.CSRC, str(src)], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    # the check has teeth: an int cursor in steps of 16 does not compile there
    src.write_text(SOURCE.replace("LaneWalk w(s, e, l);\n    while (w.on()) { n++; w.next(G); }",
                                  "for (int c = s + l; c < e; c += G) n++;"))
    assert subprocess.run(["g++", "-std=c++17", "-fsyntax-only", "-I" + B.CSRC, str(src)],
                          capture_output=True).returncode != 0
