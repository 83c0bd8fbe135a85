"""The GEMM kernels' loads in the tiles of a K that is no multiple of 128, walked on the CPU: csrc/
buf_offsets.h, whose functions form every offset of those loads, compiled for the host and asked for each
lane of each step. A load must lie inside the matrix it reads (the last expert's, with nothing behind it)
or past the size that the unit checks its vector offset against, where it gives zeros; a row of
activations must be read inside its K bytes and without an offset that wraps."""
import subprocess

import pytest

from conftest import REPO

WALK = r"""
#include <cstdio>
#include <cstdlib>
#include "buf_offsets.h"
using namespace w4a8;

static void fail(const char* what, int K, int N, int g, int kt, int lane, BufOffset o) {
  printf("%s: K=%d N=%d group=%d tile %d lane %d: offsets %u + %u\n", what, K, N, g, kt, lane, o.v, o.s);
  exit(1);
}
// inside the matrix, or wholly past the size that the vector offset is checked against
static void load(const char* what, BufOffset o, uint64_t size, uint64_t bytes, uint64_t checked, int K, int N, int g, int kt,
                 int lane) {
  const uint64_t at = (uint64_t)o.v + o.s;
  if (!(at + size <= bytes || o.v >= checked)) fail(what, K, N, g, kt, lane, o);
}
static void load(const char* what, BufOffset o, uint64_t size, uint64_t bytes, int K, int N, int g, int kt, int lane) {
  load(what, o, size, bytes, bytes, K, N, g, kt, lane);
}

int main(int argc, char** argv) {
  const int K = atoi(argv[1]), N = atoi(argv[2]), KT = (K + 127) / 128, ktail = K - (KT - 1) * 128;
  const uint64_t ldx = K + 16 * atoi(argv[3]);
  // activations: three rows, the first at offset 0 (it also stands for rows without data)
  for (int kt = 0; kt < KT; ++kt)
    for (int half = 0; half < 2; ++half)
      for (int lane = 0; lane < 64; ++lane)
        for (uint64_t row = 0; row < 3; ++row) {
          const uint32_t from = a_piece((uint32_t)(row * ldx), half, lane) + kABias;
          const BufOffset o = {a_step(from, a_back(half, lane, ktail), kt == KT - 1 ? ~0u : 0u), (uint32_t)(kt * 128)};
          if (o.v > from) fail("activations (below zero)", K, N, 0, kt, lane, o);
          const uint64_t at = (uint64_t)o.v + o.s - kABias, in = (uint64_t)kt * 128 + 64 * half + 16 * (lane >> 4);
          if (at < row * ldx || at + 16 > row * ldx + K) fail("activations", K, N, 0, kt, lane, o);
          // the piece itself wherever it lies inside K
          if (in + 16 <= (uint64_t)K && at != row * ldx + in) fail("activations (place)", K, N, 0, kt, lane, o);
        }
  for (int kt = 0; kt < KT; ++kt) {
    // the kernels hand `ragged` to the steps that may load the last tile; steps before it are in range either way
    const bool ragged = kt == KT - 1;
    for (int lane = 0; lane < 64; ++lane)
      for (int strip = 0; strip < N / 16; ++strip) {
        for (int g = 32; g <= 64; g *= 2) {
          if (K % g) continue;
          const int gpt = 128 / g;
          const uint64_t groups = K / g, z_bytes = groups * (N / 8) * 4, s_bytes = groups * N * 2;
          for (int h = 0; h < 2; ++h)
            load("zero words", row_step(zero_word(lane, strip * 16 + (lane & 15), gpt, N),
                                        (uint32_t)((kt * gpt + h * (gpt / 2)) * (N / 8) * 4), ragged), 4, z_bytes, K, N, g, kt, lane);
          for (int c = 0; c < gpt; ++c)
            load("scales", row_step(scale_piece(c, strip, lane & 1, N), (uint32_t)(kt * gpt * N * 2), ragged), 16, s_bytes, K,
                 N, g, kt, lane);
        }
        // decode kernels: the descriptor starts at the tile's rows; a row for every block
        const uint64_t left = e8m0_bytes_left(kt, K, N), from = (uint64_t)kt * 4 * N;
        if (from + left != (uint64_t)K / 32 * N) fail("E8M0 descriptor", K, N, 32, kt, lane, {0, (uint32_t)from});
        for (int ss = 0; ss < 8; ++ss) {
          const uint32_t row = e4m3_row(kt, ss, K, N);
          load("e4m3 row", {(uint32_t)(strip * 16 + (lane & 15)), row}, 1, (uint64_t)K / 16 * N, ~0ull, K, N, 16,
               kt, lane);
          if (kt * 128 + ss * 16 < K && row != (uint32_t)((kt * 8 + ss) * N)) fail("e4m3 row (place)", K, N, 16, kt, lane, {0, row});
        }
        if (K % 32 == 0)
          load("E8M0 bytes", row_step(e8m0_word(lane, strip, N), (uint32_t)(kt * 4 * N), ragged), 4, (uint64_t)K / 32 * N, K,
               N, 32, kt, lane);
        for (int h = 0; h < 2; ++h)
          load("e4m3 bytes", row_step(e4m3_byte(lane, h, strip, N), (uint32_t)(kt * 8 * N), true), 1, (uint64_t)K / 16 * N, K,
               N, 16, kt, lane);
      }
  }
  return 0;
}
"""


@pytest.fixture(scope="module")
def walk(tmp_path_factory):
    d = tmp_path_factory.mktemp("walk")
    (d / "walk.cpp").write_text(WALK)
    subprocess.run(["g++", "-O1", "-std=c++17", "-I", str(REPO / "minisglang-rdna4_amd" / "csrc"), str(d / "walk.cpp"),
                    "-o", str(d / "walk")], check=True)
    return d / "walk"


@pytest.mark.parametrize("K", [160, 192, 224, 256, 480, 544, 1088])
@pytest.mark.parametrize("N", [16, 48, 1040])
@pytest.mark.parametrize("pad", [0, 3])
def test_ragged_tile_loads_stay_inside(walk, K, N, pad):
    r = subprocess.run([str(walk), str(K), str(N), str(pad)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout
