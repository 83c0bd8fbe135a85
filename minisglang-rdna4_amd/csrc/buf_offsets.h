// Offsets of the GEMM kernels' buffer loads on a K that ends inside a 128-wide tile. Plain functions,
// so that a host program can walk every lane of every load (tests/test_ragged_offsets.py).
//
// Of a load's two offsets only the vector one is checked against the descriptor's size; the scalar one is
// added behind the check. A load that may fall outside its matrix therefore carries everything in the
// vector offset, where a read past the end gives zeros (the prefill kernels), or moves the descriptor's
// start and size in its place (the decode kernels, whose lanes it costs nothing); and no vector offset goes
// below zero.
#pragma once
#include <stdint.h>

#if defined(__HIPCC__)
#include <hip/hip_runtime.h>
#define W4A8_HD __host__ __device__ __forceinline__
#else
#define W4A8_HD inline
#endif

namespace w4a8 {

struct BufOffset {
  uint32_t v, s;  // per lane and range-checked; wave-uniform and not
};

// A 16-byte piece of an activation row: lane l of block half h of row block b reads row (l & 15) of it
W4A8_HD uint32_t a_piece(uint32_t row_off, int half, int lane) { return row_off + 64 * half + 16 * (lane >> 4); }
// 128 for the lanes whose piece of a tile with ktail inputs lies past them, else 0
W4A8_HD uint32_t a_back(int half, int lane, int ktail) { return 64 * half + 16 * (lane >> 4) >= ktail ? 128u : 0u; }
// last: all ones for the last tile of K, else 0. There the lanes with `back` read the tile before (the
// operand read masks theirs out). The piece's offset is from kABias bytes ahead of the activations, where
// the descriptor starts, so that the lanes of row 0 that step back do not go below zero; every address
// read lies inside its row.
constexpr int kABias = 128;
W4A8_HD uint32_t a_step(uint32_t biased_piece, uint32_t back, uint32_t last) { return biased_piece - (back & last); }

// Zero word of channel n: lane l of a strip reads codes K 16q.. of the tile and K 64 + 16q.. (q = l >> 4),
// of groups q * gpt / 8 and that + gpt / 2 (gpt groups per tile; one for groups of 128 and more)
W4A8_HD uint32_t zero_word(int lane, int n, int gpt, int N) {
  return (uint32_t)((((lane >> 4) * gpt / 8) * (N / 8) + n / 8) * 4);
}
// 16 bytes of the fp16 scales of group g of a tile: half h of a strip's 16 channels
W4A8_HD uint32_t scale_piece(int g, int strip, int half, int N) { return (uint32_t)((g * N + strip * 16 + half * 8) * 2); }
// dword of the E8M0 bytes of a tile: lane m & 15's 32-block m >> 2, channels 4 (m & 3).. of a strip
W4A8_HD uint32_t e8m0_word(int lane, int strip, int N) {
  const int m = lane & 15;
  return (uint32_t)((m >> 2) * N + strip * 16 + (m & 3) * 4);
}
// e4m3 scale byte of block 2q + h of a tile, channel lane & 15 of a strip
W4A8_HD uint32_t e4m3_byte(int lane, int h, int strip, int N) {
  return (uint32_t)((2 * (lane >> 4) + h) * N + strip * 16 + (lane & 15));
}
// Decode kernels: bytes from tile kt's first E8M0 row to the end of the scales, the size of the descriptor
// that starts there; and where the e4m3 row of block ss of tile kt starts, the last row again for blocks past K
W4A8_HD uint32_t e8m0_bytes_left(int kt, int K, int N) { return (uint32_t)((K / 32 - kt * 4) * N); }
W4A8_HD uint32_t e4m3_row(int kt, int ss, int K, int N) {
  const uint32_t row = (uint32_t)((kt * 8 + ss) * N), last = (uint32_t)((K / 16 - 1) * N);
  return row < last ? row : last;
}
// a scale or zero load, its rows starting at byte `so` of the matrix; ragged: in a tile that may have
// fewer rows than the load covers
W4A8_HD BufOffset row_step(uint32_t off, uint32_t so, bool ragged) {
  return ragged ? BufOffset{off + so, 0u} : BufOffset{off, so};
}

}  // namespace w4a8
