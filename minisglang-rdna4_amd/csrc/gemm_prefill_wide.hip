// The dense int4 prefill GEMM (groups of 128+) on 256 x 256 tiles, for activations in operand order
// (GemmArgs::a_tiled), symmetric with their row-sum seeds or with zero points; the math and the bits of
// gemm_prefill_dma.hip's tiles.
//
// What bounds the 256 x 128 tile there is not its MFMAs but what goes with each: 1 KiB of LDS operands
// per MFMA, and a barrier every 16 of them. A 256 x 256 tile halves the barriers and takes a quarter
// off the LDS reads, and each weight strip is unpacked for 256 rows by one workgroup instead of two.
// It has to fit two waves per SIMD in 256 registers and 160 KiB of LDS:
//   * a wave owns 128 x 64 outputs (128 accumulators). It holds the K step's four strips (32 registers)
//     and streams its eight row blocks, one ahead. A strip's partial of row block r is scaled into the
//     accumulators right before the strip's MFMA of row block r + 1 (four MFMAs after its own, so
//     nothing waits), which keeps one set of partials live instead of two;
//   * two stages of 32 KiB activations, 32 KiB unpacked weights, scales and seeds. Activations, scales
//     and seeds go to LDS by LDS-DMA at the start of the step before theirs, which is twice as long as a
//     256 x 128 step; the 4-bit weights are loaded to registers two steps ahead and unpacked one ahead.
// Whole calls, operand order on 256 x 128 -> 256 x 256, us: K=4096 N=28672 M=8192 1134 -> 955 (2.0
// PFLOP/s), N=6144 M=8192 259 -> 220, N=4096 M=8192 181 -> 153, K=14336 N=4096 M=4096 308 -> 267, K=1024
// N=4096 M=4096 37.0 -> 32.1. With zero points, row-major codes on the tiles they take -> operand order on
// this one: K=4096 N=28672 M=8192 1167 -> 1006, N=14336 M=3000 239 -> 208, N=4096 M=8192 177 -> 159.
// The unpack placed one row block earlier or later, the DMAs ahead of the step's LDS reads, and a raised
// wave priority around the MFMAs all measured within 1%.
#include "prefill.h"

namespace w4a8 {

template <int I, int N, typename F>
__device__ __forceinline__ void wide_steps(F f) {
  if constexpr (I < N) {
    f(IC<I>{});
    wide_steps<I + 1, N>(f);
  }
}

template <int WM, int WN, int RB, int NSB, int MODE>
__global__ void __launch_bounds__(WM * WN * 64) __attribute__((amdgpu_waves_per_eu(2, 2)))
gemm_wide_kernel(const GemmArgs p) {
  static_assert(MODE == kPSym || MODE == kPAsym, "int4, groups of 128 or more");
  constexpr bool kZ = MODE == kPAsym;  // weights decoded as e4m3(q - z), no seeds
  constexpr int T = WM * WN * 64, NW = WM * WN;
  constexpr int BM = WM * RB * 16, BN = WN * NSB * 16, NSTRIP = BN / 16;
  constexpr int kA = BM * 128, kB = BN * 128, kS = BN * 2;
  constexpr int kScaleOff = kA, kSeedOff = kScaleOff + kS, kDma = kSeedOff + (kZ ? 0 : BM * 4);
  constexpr int A_PER = BM / 8 / NW, B_PER = NSTRIP * 64 / T;
  constexpr int W_PER = B_PER * (kZ ? 2 : 1);  // loads of a step's weights (and zero words) per thread
  static_assert(A_PER * NW == BM / 8 && B_PER * T == NSTRIP * 64, "blocks / waves");
  constexpr int kScaleW = BN / 128, kSeedW = BM / 64;  // waves whose dword DMAs cover the scales, the seeds
  static_assert(NW % kScaleW == 0 && NW % kSeedW == 0, "every wave issues one DMA of each");

  // what the DMAs write and what the waves write in arrays of their own, so that the compiler does not
  // make the unpacked weights' writes wait for the DMAs just issued
  __shared__ __align__(16) unsigned char sa0[kDma];
  __shared__ __align__(16) unsigned char sa1[kDma];
  __shared__ __align__(16) unsigned char sb0[kB];
  __shared__ __align__(16) unsigned char sb1[kB];
  auto astage = [&](auto I) __attribute__((always_inline)) -> unsigned char* {
    if constexpr (decltype(I)::value == 0) return sa0;
    else return sa1;
  };
  auto bstage = [&](auto I) __attribute__((always_inline)) -> unsigned char* {
    if constexpr (decltype(I)::value == 0) return sb0;
    else return sb1;
  };

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave / WN, wn = wave % WN;
  const int bx = (int)blockIdx.x;
  const int64_t blk_row0 = (int64_t)blockIdx.y * BM;
  const int N = (int)p.N, KT = (int)p.KT, nstrips = N / kTileN;
  const int gshift = 31 - __builtin_clz((unsigned)(p.group / kTileK));

  // global strip of LDS strip s, as in gemm_dma_kernel
  auto gstrip = [&](int s, bool& ok) __attribute__((always_inline)) {
    int gs;
    if (p.silu) {
      constexpr int hj = NSB / 2;
      const int j = s % NSB;
      const int h = bx * (NSTRIP / 2) + (s / NSB) * hj + (j < hj ? j : j - hj);
      gs = j < hj ? h : nstrips / 2 + h;
      ok = h < nstrips / 2;
    } else {
      gs = bx * NSTRIP + s;
      ok = gs < nstrips;
    }
    return ok ? gs : nstrips - 1;
  };

  const uint32_t w_bytes = (uint32_t)((size_t)nstrips * KT * kTileBytes);
  const uint32_t s_bytes = (uint32_t)((size_t)(KT >> gshift) * N * 2);
  const uint32_t seed_bytes = kZ ? 0u : (uint32_t)((size_t)KT * p.seeds_ld * 4);
  const uint32_t z_bytes = kZ ? (uint32_t)((size_t)(KT >> gshift) * (N / 8) * 4) : 0u;

  // per-lane source offsets (rows past M read the last 16-row block / seed; their outputs are not stored)
  uint32_t a_voff[A_PER];
  const int64_t nblk16 = (p.M + 15) / 16;
#pragma unroll
  for (int i = 0; i < A_PER; ++i) {
    const int b = wave + i * NW;
    int64_t rbg = blk_row0 / 16 + (b >> 1);
    rbg = rbg < nblk16 ? rbg : nblk16 - 1;
    a_voff[i] = (uint32_t)((rbg * KT * 2 + (b & 1)) * 1024 + lane * 16);
  }
  int64_t sr = blk_row0 + 64 * (wave % kSeedW) + lane;
  sr = sr < p.seeds_ld ? sr : p.seeds_ld - 1;
  const uint32_t seed_voff = (uint32_t)(sr * 4);
  bool ok_;
  const int sd = 64 * (wave % kScaleW) + lane;  // dword of the tile's scale row: two channels of strip sd / 8
  const uint32_t s_voff = (uint32_t)((gstrip(sd >> 3, ok_) * 16 + (sd & 7) * 2) * 2);
  uint32_t b_voff[B_PER], z_voff[B_PER];
#pragma unroll
  for (int i = 0; i < B_PER; ++i) {
    const int c = (int)threadIdx.x + i * T, gs = gstrip(c >> 6, ok_);
    b_voff[i] = (uint32_t)(((size_t)gs * KT * 64 + (c & 63)) * 16);
    z_voff[i] = (uint32_t)((gs * 2 + ((c >> 3) & 1)) * 4);
  }
  __shared__ uint4 zlut[kZ ? 16 : 1];
  if (kZ && threadIdx.x < 16) zlut[threadIdx.x] = zero_point_lut((int)threadIdx.x);

  __shared__ float e_sc[BM];
  const int er = (int)threadIdx.x;
  float er_sc = 0.f;
  if (er < BM && blk_row0 + er < p.M) er_sc = p.act_scales[blk_row0 + er];

  v4u rbw[2][B_PER];
  uint32_t rzp[2][B_PER];
  // Tail: loads past the last step read empty buffers, as in gemm_dma_kernel
  auto live_of = [&](int kt, auto Tail) __attribute__((always_inline)) {
    return decltype(Tail)::value ? (uint32_t)__builtin_amdgcn_readfirstlane(kt < KT ? -1 : 0) : 0xffffffffu;
  };
  auto issue_dma = [&](auto I, int kt, auto Tail) __attribute__((always_inline)) {
    unsigned char* st = astage(I);
    const uint32_t live = live_of(kt, Tail);
    if constexpr (decltype(Tail)::value) kt = kt < KT ? kt : KT - 1;
    const BufRsrc rs_a = make_rsrc(p.xq, live), rs_s = make_rsrc(p.scales, s_bytes & live);
    const BufRsrc rs_seed = make_rsrc(p.seeds, seed_bytes & live);
    const uint32_t so = (uint32_t)__builtin_amdgcn_readfirstlane(kt * 2048);
#pragma unroll
    for (int i = 0; i < A_PER; ++i) lds_dma16(rs_a, st + (wave + i * NW) * 1024, a_voff[i], so);
    lds_dma4(rs_s, st + kScaleOff + (wave % kScaleW) * 256, s_voff,
             (uint32_t)__builtin_amdgcn_readfirstlane((kt >> gshift) * N * 2));
    if constexpr (!kZ)
      lds_dma4(rs_seed, st + kSeedOff + (wave % kSeedW) * 256, seed_voff,
               (uint32_t)__builtin_amdgcn_readfirstlane(kt * (int)p.seeds_ld * 4));
  };
  auto issue_w = [&](auto R_, int kt, auto Tail) __attribute__((always_inline)) {
    constexpr int R = decltype(R_)::value;
    const uint32_t live = live_of(kt, Tail);
    const BufRsrc rs_w = make_rsrc(p.wt, w_bytes & live), rs_z = make_rsrc(p.zeros, z_bytes & live);
    if constexpr (decltype(Tail)::value) kt = kt < KT ? kt : KT - 1;
    const uint32_t so = (uint32_t)__builtin_amdgcn_readfirstlane(kt * kTileBytes);
#pragma unroll
    for (int i = 0; i < B_PER; ++i) rbw[R][i] = bload128v(rs_w, b_voff[i], so);
    if constexpr (kZ) {
      const uint32_t so_z = (uint32_t)__builtin_amdgcn_readfirstlane((kt >> gshift) * (N / 8) * 4);
#pragma unroll
      for (int i = 0; i < B_PER; ++i) rzp[R][i] = bload32(rs_z, z_voff[i], so_z);
    }
  };
  auto commit = [&](auto I, int i) __attribute__((always_inline)) {  // chunk i of the stage's weights
    constexpr int R = decltype(I)::value;
    unsigned char* sb = bstage(I);
    const int c = (int)threadIdx.x + i * T, s = c >> 6, l = c & 63;
    const uint4 w = make_uint4(rbw[R][i].x, rbw[R][i].y, rbw[R][i].z, rbw[R][i].w);
    v8i u;
    if constexpr (kZ) {
      const uint4 t = zlut[(rzp[R][i] >> (4 * (lane & 7))) & 15u];
      u = unpack_tile_lut(w, t, t);
    } else {
      u = unpack_tile_int4(w);
    }
    *reinterpret_cast<uint4*>(sb + ((s * 2 + 0) * 64 + l) * 16) = make_uint4(u[0], u[1], u[2], u[3]);
    *reinterpret_cast<uint4*>(sb + ((s * 2 + 1) * 64 + l) * 16) = make_uint4(u[4], u[5], u[6], u[7]);
  };

  v4f acc[RB][NSB];
#pragma unroll
  for (int rb = 0; rb < RB; ++rb)
#pragma unroll
    for (int j = 0; j < NSB; ++j) acc[rb][j] = v4f{0.f, 0.f, 0.f, 0.f};
  uint32_t oa = (uint32_t)(wm * RB * 2048 + lane * 16);
  uint32_t ob = (uint32_t)(wn * NSB * 2048 + lane * 16);
  uint32_t os = (uint32_t)(kScaleOff + (wn * NSB * 16 + (lane & 15)) * 2);
  uint32_t oe = (uint32_t)(kSeedOff + (wm * RB * 16 + 4 * (lane >> 4)) * 4);
  asm volatile("" : "+v"(oa), "+v"(ob), "+v"(os), "+v"(oe));

  // step kt (stage kt % 2): the DMAs of kt + 1 after the first row block's MFMAs, the weight loads of
  // kt + 2 after the second's, the weights of kt + 1 unpacked after the third's and the fifth's; then
  // wait for the DMAs (the weight loads stay in flight) and meet at the barrier
  auto step = [&](auto C, int kt, auto Tail) __attribute__((always_inline)) {
    if (decltype(Tail)::value && kt >= KT) return;
    constexpr int c = decltype(C)::value, n = 1 - c;
    const unsigned char* st = astage(C);
    const unsigned char* sb = bstage(C);
    v8i b[NSB];
    float sc[NSB];
    v8i a0 = lds_operand(st + oa, 0);
    v4f e0 = kZ ? v4f{0.f, 0.f, 0.f, 0.f} : *reinterpret_cast<const v4f*>(st + oe);
#pragma unroll
    for (int j = 0; j < NSB; ++j) b[j] = lds_operand(sb + ob + j * 2048, 0);
#pragma unroll
    for (int j = 0; j < NSB; ++j) sc[j] = f16_to_f32(*reinterpret_cast<const uint16_t*>(st + os + j * 32));
    v4f cj[NSB];
#pragma unroll
    for (int rb = 0; rb < RB; ++rb) {
      v8i a1;
      v4f e1;
      if (rb + 1 < RB) {
        a1 = lds_operand(st + oa + (rb + 1) * 2048, 0);
        e1 = kZ ? v4f{0.f, 0.f, 0.f, 0.f} : *reinterpret_cast<const v4f*>(st + oe + (rb + 1) * 64);
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int j = 0; j < NSB; ++j) {
        if (rb > 0) {
#pragma unroll
          for (int r = 0; r < 4; ++r) acc[rb - 1][j][r] += sc[j] * cj[j][r];
        }
        cj[j] = mfma_f8f8(a0, b[j], e0);
      }
      if (rb > 0) {
#pragma unroll
        for (int j = 0; j < NSB; ++j) {
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
          __builtin_amdgcn_sched_group_barrier(0x002, 4, 0);
        }
      }
      if (rb == 0) issue_dma(IC<n>{}, kt + 1, Tail);
      if (rb == 1) issue_w(IC<c>{}, kt + 2, Tail);  // behind the DMAs: the wait below counts on it
      if (rb == 2) commit(IC<n>{}, 0);
      if (rb == 4 && B_PER > 1) commit(IC<n>{}, B_PER - 1);
      if (rb + 1 < RB) {
        a0 = a1;
        e0 = e1;
      }
    }
#pragma unroll
    for (int j = 0; j < NSB; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) acc[RB - 1][j][r] += sc[j] * cj[j][r];
    __builtin_amdgcn_sched_barrier(0);
    wait_vm_lgkm0<W_PER>();
    __builtin_amdgcn_s_barrier();
  };
  static_assert(B_PER <= 2, "weight chunks per thread");

  issue_dma(IC<0>{}, 0, IC<1>{});
  issue_w(IC<0>{}, 0, IC<1>{});
  __builtin_amdgcn_sched_barrier(0);
  issue_w(IC<1>{}, 1, IC<1>{});
  __builtin_amdgcn_sched_barrier(0);
  if constexpr (kZ) lds_barrier();  // the zero-point table, before the first decode reads it
#pragma unroll
  for (int i = 0; i < B_PER; ++i) commit(IC<0>{}, i);
  wait_vm_lgkm0<W_PER>();
  if (er < BM) e_sc[er] = er_sc;  // read after the K loop's barriers
  __builtin_amdgcn_s_barrier();
  int kt = 0;
  for (; kt + 3 < KT; kt += 2) {
    step(IC<0>{}, kt, IC<0>{});
    step(IC<1>{}, kt + 1, IC<0>{});
  }
  wide_steps<0, 3>([&](auto I) __attribute__((always_inline)) {
    constexpr int i = decltype(I)::value;
    step(IC<i % 2>{}, kt + i, IC<1>{});
  });
  // the empty loads of the last steps write LDS too: all landed before the epilogue reuses it
  wait_vm_lgkm0<0>();
  __builtin_amdgcn_s_barrier();

  const int64_t row0 = blk_row0 + (int64_t)wm * RB * 16;
  float e_rsc[RB][4];
  uint32_t e_valid = 0;
#pragma unroll
  for (int rb = 0; rb < RB; ++rb)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int lr = rb * 16 + 4 * (lane >> 4) + r;
      e_rsc[rb][r] = e_sc[wm * RB * 16 + lr];
      e_valid |= (row0 + lr < p.M ? 1u : 0u) << (rb * 4 + r);
    }
  constexpr int kScr = 16 * (NSB * 16 * 4 + 16);
  static_assert(kB / kScr * 2 >= NW && RB * 4 <= 32, "epilogue scratch, row mask");
  store_tile_scaled(p, acc, e_rsc, e_valid, row0, lane,
                    [&](int j, bool& ok) __attribute__((always_inline)) { return gstrip(wn * NSB + j, ok); },
                    (wave < kB / kScr ? sb0 : sb1) + (wave % (kB / kScr)) * kScr);
}

int launch_prefill_wide(const GemmArgs& p, int64_t rows, hipStream_t stream) {
  const int64_t ncols = p.silu ? p.N / 2 : p.N, colw = p.silu ? 128 : 256;
  const dim3 grid((unsigned)((ncols + colw - 1) / colw), (unsigned)((rows + 255) / 256));
  if (p.zeros)
    hipLaunchKernelGGL((gemm_wide_kernel<2, 4, 8, 4, kPAsym>), grid, dim3(512), 0, stream, p);
  else
    hipLaunchKernelGGL((gemm_wide_kernel<2, 4, 8, 4, kPSym>), grid, dim3(512), 0, stream, p);
  return hipGetLastError() == hipSuccess ? kOk : kErrHip;
}

}  // namespace w4a8
