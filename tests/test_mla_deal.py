"""How MLA decode deals tiles to runs: the header that its kernels count with, on the CPU."""

import ctypes
import os
import random
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(__file__), "..", "parallax_amd", "ops", "csrc")

# the kernels' find_run with one sequence after the other in place of a wave
SHIM = r"""
#include "mla_deal.h"
static int div_up(int n, int d) { return n > 0 ? (n + d - 1) / d : 0; }
extern "C" int deal(const int* tiles, int B, int runs, int shortest, int more, int* out) {
  int total = 0;
  for (int b = 0; b < B; ++b) total += tiles[b];
  int even = div_up(total, runs);
  if (even < shortest) even = shortest;
  const int least = least_length(even, even + more, runs, [&](int length) {
    int n = 0;
    for (int b = 0; b < B; ++b) n += div_up(tiles[b], length);
    return n;
  });
  const bool whole = least <= even + more;
  const int per = whole ? least : even;
  for (int run = 0; run < runs; ++run) {
    Run r = {0, 0, 0, 1};
    const int begin = whole ? run : run * per;
    for (int b = 0, first = 0; b < B; ++b) {
      const int n = whole ? div_up(tiles[b], per) : tiles[b];
      if (begin >= first && begin < first + n)
        r = whole ? run_of_sequence(b, run - first, tiles[b], n, div_up)
                  : run_of_list(b, begin, first, per, total);
      first += n;
    }
    out[run * 4] = r.seq, out[run * 4 + 1] = r.at, out[run * 4 + 2] = r.todo;
    out[run * 4 + 3] = r.per;
  }
  return least;
}
"""


@pytest.fixture(scope="module")
def deal(tmp_path_factory):
    d = tmp_path_factory.mktemp("deal")
    (d / "deal.cpp").write_text(SHIM)
    subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", "-I", CSRC,
                    str(d / "deal.cpp"), "-o", str(d / "deal.so")], check=True)
    f = ctypes.CDLL(str(d / "deal.so")).deal

    def call(tiles, runs, shortest, more):
        out = (ctypes.c_int * (4 * runs))()
        least = f((ctypes.c_int * len(tiles))(*tiles), len(tiles), runs, shortest, more, out)
        return least, [tuple(out[i:i + 4]) for i in range(0, 4 * runs, 4)]
    return call


def _up(n, d):
    return -(-n // d)


@pytest.mark.parametrize("runs", [1, 128, 256])
@pytest.mark.parametrize("shortest,more", [(2, 0), (2, 1), (2, 3), (4, 9), (4, 16)])
def test_every_tile_once_and_no_longer_than_need_be(deal, runs, shortest, more):
    rng = random.Random(runs * 100 + more)
    lists = [[0], [1], [0, 0, 7], [1] * 300, [4096], [3] * 128, [17] * 99 + [0] * 20]
    for _ in range(400):
        top = int(2 ** rng.uniform(0, 10))
        lists.append([rng.choice((top, rng.randint(0, top)))
                      for _ in range(rng.randint(1, 200))])
    wholes = 0
    for tiles in lists:
        least, dealt = deal(tiles, runs, shortest, more)
        even = max(_up(sum(tiles), runs), shortest)
        fits = [n for n in range(even, even + more + 1)
                if sum(_up(t, n) for t in tiles) <= runs]
        assert least == (fits[0] if fits else even + more + 1), tiles
        wholes += bool(fits)
        seen = [0] * sum(tiles)
        first = [sum(tiles[:b]) for b in range(len(tiles))]
        for seq, at, todo, per in dealt:
            if todo <= 0:
                continue
            assert todo <= per <= (fits[0] if fits else even)
            if fits:
                assert at + todo <= tiles[seq]
            for t in range(first[seq] + at, first[seq] + at + todo):
                seen[t] += 1
        assert all(n == 1 for n in seen), tiles
    assert runs == 1 or 0 < wholes < len(lists)
