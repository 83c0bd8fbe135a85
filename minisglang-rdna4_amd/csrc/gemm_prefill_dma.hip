// Large-M W4A8 GEMM (prefill band and grouped MoE GEMMs) with the activation tile copied straight
// from global memory into LDS by the buffer unit (buffer_load ... lds), three LDS stages deep (the 64 x 64 tile four).
//
// The math of the reference's wmma_tiled_tuned arm and of its grouped MoE GEMMs
// (python/minisgl/quant/kernels.py:1632, 1686-1734, 744-773): y[m,n] = s_m * sum_g scale[g,n] *
// sum_{k in g} e4m3(x[m,k]) w(n,k), f32 accumulation. Per (row block, strip, K step of 128): one
// 16x16x128 MFMA, or for groups of 64 and 32 four 16x16x32 ones (half the rate, but a group's partial
// must be scaled by itself: the full-rate MFMA with the other blocks masked out takes 2 or 4 times its
// cycles).
//
// How a K step's operands reach LDS:
//   A (BM x 128 fp8) and, for MXFP4, the fp4 weight strips and their E8M0 bytes are loaded by
//   LDS-DMA: one 1 KiB block per wave instruction, written in lane order, which is exactly the
//   MFMA operand order, so no VGPR holds them and no ds_write is issued;
//   int4 weights go through registers: each workgroup unpacks every strip once to the fp8 operand and
//   writes it to LDS, with its fp16 scales. Symmetric groups of 128+ are unpacked as q - 7.5 with one
//   table lookup and the half step taken back through the row sums; the other forms as e4m3(q - z),
//   which needs no row sums (decode_lut4). With zero points applied per accumulator instead (two FMAs
//   per element and a row-sum MFMA per row block) a call of M=1777 K=2560 N=9728 on row-major 256 x 128
//   tiles took 102 us, so 86. Groups of 32 on the kernel that masks the full-rate MFMA and loads operands
//   straight from global memory: M=2048 K=2816 N=2048 196 us a call, here 42.
// Each stage is its own __shared__ array and every stage index is a compile-time constant (the K
// loop is unrolled by the stages), so the compiler tells the stages apart: reading stage k does not
// wait for the DMAs in flight to the later ones. With three stages step k issues the loads of step
// k+2 (int4: between its MFMAs), computes step k, writes the int4 registers of step k+1, then waits
// for its own step-k+1 loads (a counted vmcnt, the loads of step k+2 stay in flight) and meets the
// other waves at one s_barrier; with four, everything is loaded one step earlier.
#include "prefill.h"

namespace w4a8 {

template <int I, int N, typename F>
__device__ __forceinline__ void for_stages(F f) {
  if constexpr (I < N) {
    f(IC<I>{});
    for_stages<I + 1, N>(f);
  }
}

template <int WM, int WN, int RB, int NSB, int NST, int MODE, bool AT>
__global__ void __launch_bounds__(WM * WN * 64) __attribute__((amdgpu_waves_per_eu(2, 2)))
gemm_dma_kernel(const GemmArgs p) {
  constexpr int T = WM * WN * 64, NW = WM * WN;
  constexpr int BM = WM * RB * 16, BN = WN * NSB * 16;
  constexpr int NSTRIP = BN / 16;
  constexpr bool kFp4 = MODE == kPE8M0;
  // groups per K tile, and the modes whose weights are decoded as e4m3(q - z) (see decode_lut4)
  constexpr int GPT = prefill_gpt(MODE);
  constexpr bool kLut = prefill_lut(MODE), kLutZ = prefill_lut_zeros(MODE);
  using S = LdsStage<BM, BN, MODE>;
  constexpr int A_PER = (BM / 8) / NW;                 // A 1 KiB blocks per wave per step
  static_assert(A_PER * NW == BM / 8, "A blocks / waves");
  constexpr int B_DMA = kFp4 ? NSTRIP / NW : 0;        // fp4 strips per wave per step
  constexpr int S_DMA = kFp4 ? NSTRIP / NW : 0;        // E8M0 strips per wave per step
  // E8M0 bytes: one 256-byte slot per strip (a wave's dword DMA covers 64 lanes x 4 bytes; lanes
  // 0-15 carry the strip's 64 bytes, the rest repeat them into the slot's unused tail)
  constexpr int kSE8 = NSTRIP * 256;
  // AT (p.a_tiled): A in operand order, and for symmetric int4 the row-sum seeds travel by LDS-DMA
  // (one dword per row, kSeedB bytes per stage) instead of four MFMAs per wave and step
  constexpr bool kSeedL = AT && MODE == kPSym;
  constexpr int kSeedOff = kFp4 ? S::kA + S::kB + kSE8 : S::kBytes;
  constexpr int kSeedB = kSeedL ? BM * 4 : 0;
  constexpr int kStage = kSeedOff + kSeedB;
  static_assert(!kFp4 || B_DMA * NW == NSTRIP, "fp4 strips / waves");
  constexpr int B_PER = kFp4 ? 0 : NSTRIP * 64 / T;    // int4 16-byte chunks per thread per step
  static_assert(kFp4 || B_PER * T == NSTRIP * 64, "int4 chunks / threads");
  // vector-memory operations every wave issues per step (all unconditional, so one count holds)
  constexpr int ZL = kLutZ ? (GPT > 1 ? 2 : 1) : 0;    // zero words per chunk: its one or two groups
  constexpr int NOPS = (kFp4 ? S_DMA + A_PER + B_DMA : A_PER + B_PER * (1 + ZL) + 1) + (kSeedL ? 1 : 0);

  // NST stages, each its own array; loads run D steps ahead
  constexpr int D = NST - 1;
  static_assert(NST == 3 || NST == 4, "stages");
  __shared__ __align__(16) unsigned char st0[kStage];
  __shared__ __align__(16) unsigned char st1[kStage];
  __shared__ __align__(16) unsigned char st2[kStage];
  __shared__ __align__(16) unsigned char st3[NST > 3 ? kStage : 16];
  auto stage = [&](auto I) __attribute__((always_inline)) -> unsigned char* {
    constexpr int i = decltype(I)::value;
    if constexpr (i == 0) return st0;
    else if constexpr (i == 1) return st1;
    else if constexpr (i == 2) return st2;
    else return st3;
  };

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave / WN, wn = wave % WN;
  int bx = (int)blockIdx.x, by = (int)blockIdx.y;
  int64_t expert = 0;
  if (p.sorted_ids) {
    // Grouped: tiles in XCD order. Workgroup i runs on XCD i % 8; each XCD takes a contiguous
    // range of the tiles that hold rows (row tiles below ntp, every column tile of each), so a
    // row tile's A rows and an expert's weight strips, read by the neighbouring tiles, stay in one
    // L2 (in grid order a row tile's column tiles and an expert's row tiles sat on different XCDs).
    // The grid is a multiple of 8 workgroups, so every XCD has the same number of slots.
    const int gx = (int)gridDim.x;
    const int i = by * gx + bx;
    const int used = ((*p.ntp) + BM - 1) / BM * gx;
    const int share = (used + 7) / 8;
    const int v = (i & 7) * share + (i >> 3);
    if ((i >> 3) >= share || v >= used) return;
    bx = v % gx;
    by = v / gx;
    expert = p.expert_ids[(uint32_t)(by * BM) / (uint32_t)p.bm];  // padded rows < 2^31
  }
  const int64_t blk_row0 = (int64_t)by * BM;
  const int N = (int)p.N, K = (int)p.K, KT = (int)p.KT;
  const int nstrips = N / kTileN;
  const int gshift = 31 - __builtin_clz((unsigned)(p.group >= kTileK ? p.group / kTileK : 1));

  // global strip of LDS strip s: wave wn computes LDS strips [wn*NSB, wn*NSB + NSB); with silu the
  // first half of each wave's strips are gate strips and the second half the matching up strips
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

  const uint4* wt = p.wt + (size_t)(expert * p.w_expert_tiles) * 64;
  constexpr int kEsz = kFp4 ? 1 : 2;
  const unsigned char* scales = reinterpret_cast<const unsigned char*>(p.scales) + (size_t)(expert * p.s_expert_stride) * kEsz;
  const int32_t* zeros = p.zeros ? p.zeros + expert * p.z_expert_stride : nullptr;
  const int ngroups = K >> (31 - __builtin_clz((unsigned)p.group));
  static_assert(GPT == 1 || !kFp4, "sub-tile groups are int4");
  const uint32_t w_bytes = (uint32_t)((size_t)nstrips * KT * kTileBytes);
  const uint32_t s_bytes = (uint32_t)((size_t)(kFp4 ? K / 32 : ngroups) * N * kEsz);
  const uint32_t z_bytes = zeros ? (uint32_t)((size_t)ngroups * (N / 8) * 4) : 0u;

  // ---- per-lane source offsets (fixed across K steps; the step adds a scalar offset)
  // A block b = wave + i*NW of a step is row block b/2, half b%2; lane l reads row (l & 15) of it,
  // bytes [64*half + 16*(l >> 4), +16) of the step's 128
  // AT: block b's 1 KiB sits whole in the tiled codes (row blocks past M read the last one)
  // kKTail: K may end inside a tile (formats with groups below 128 only; A in operand order has whole ones)
  constexpr bool kKTail = (GPT > 1 || kFp4) && !AT;
  constexpr int kABase = kKTail ? kABias : 0;
  uint32_t a_voff[A_PER];
  const int64_t nblk16 = (p.M + 15) / 16;
#pragma unroll
  for (int i = 0; i < A_PER; ++i) {
    const int b = wave + i * NW;
    if constexpr (AT) {
      int64_t rbg = blk_row0 / 16 + (b >> 1);
      rbg = rbg < nblk16 ? rbg : nblk16 - 1;
      a_voff[i] = (uint32_t)((rbg * KT * 2 + (b & 1)) * 1024 + lane * 16);
    } else {
      int64_t ar;
      const bool ok = lrow_source(p, blk_row0 + (b >> 1) * 16 + (lane & 15), ar);
      a_voff[i] = a_piece((uint32_t)((ok ? ar : 0) * p.ldx), b & 1, lane) + kABase;
    }
  }
  const int ktail = K - (KT - 1) * kTileK;
  const uint32_t back = a_back(wave & 1, lane, ktail);
  static_assert(NW % 2 == 0, "a wave's A blocks are all the same half");
  // seeds: wave w copies rows 64 (w % (BM / 64)) + lane of the tile (waves past BM / 64 copy the same
  // rows again, so every wave issues one DMA per step and one vmcnt count holds)
  constexpr int kSeedW = BM / 64 > 0 ? BM / 64 : 1;
  const uint32_t seed_bytes = kSeedL ? (uint32_t)((size_t)KT * p.seeds_ld * 4) : 0u;
  uint32_t seed_voff = 0;
  if constexpr (kSeedL) {
    int64_t sr = blk_row0 + 64 * (wave % kSeedW) + lane;
    sr = sr < p.seeds_ld ? sr : p.seeds_ld - 1;
    seed_voff = (uint32_t)(sr * 4);
  }
  // The epilogue's rows: one per thread, its source looked up in the same round trip as the A
  // rows' and its act scale loaded ahead of step 0's loads; both go to LDS at the end of the
  // prologue, so the epilogue starts with no load to wait for (grouped rows had three dependent
  // ones there: ntp, sorted id, act scale). LDS rather than registers: the int4 tiles already use
  // nearly every VGPR through the K loop.
  __shared__ float e_sc[BM];
  __shared__ int e_ok[BM];
  __shared__ uint4 zlut[kLutZ ? 16 : 1];
  if constexpr (kLutZ) {
    if (threadIdx.x < 16) zlut[threadIdx.x] = zero_point_lut((int)threadIdx.x);
  }
  const int er = (int)threadIdx.x;
  float er_sc = 0.f;
  bool er_ok = false;
  if (er < BM) {
    int64_t ar;
    er_ok = lrow_source(p, blk_row0 + er, ar);
    er_sc = p.act_scales[er_ok ? ar : 0];
  }
  // fp4: wave strip s = wave + i*NW; E8M0 dword of DMA lane m (< 16): 32-block m >> 2, channels
  // 4 * (m & 3) .. +3 (LDS byte (m >> 2) * 16 + channel = the MFMA lane whose scale it is)
  int b_gs[kFp4 ? B_DMA : 1];
  uint32_t e_voff[kFp4 ? S_DMA : 1];
  if constexpr (kFp4) {
#pragma unroll
    for (int i = 0; i < B_DMA; ++i) {
      bool ok;
      b_gs[i] = gstrip(wave + i * NW, ok);
      e_voff[i] = e8m0_word(lane, b_gs[i], N);
    }
  }
  // int4: chunk c = tid + i*T is lane c & 63 of strip c >> 6; scales 2 chunks of 16 B per strip,
  // zero words 8 B per strip (threads past the counts load duplicates of the last and write the
  // same bytes again)
  // kStripS: a chunk's strip (one wave's, so uniform) in the scalar offsets. Groups of 32 with zero points
  // hold the most per lane, and with the strips in lane registers too the 128 x 256 grouped tile spills 19
  // of them inside its K loop: MoE T=4096 679 -> 656 us, T=1024 274 -> 262. The other tiles spill none and
  // are up to 1% slower this way.
  constexpr bool kStripS = MODE == kPG32Z && BN == 256;
  int b_strip[kStripS ? B_PER : 1];
  uint32_t b_voff[kFp4 ? 1 : B_PER];
  constexpr int S_CHUNKS = NSTRIP * 2 * GPT;
  static_assert(kFp4 || S_CHUNKS <= T, "scale chunks / threads");
  const int sc_c = (int)threadIdx.x < S_CHUNKS ? (int)threadIdx.x : S_CHUNKS - 1;
  uint32_t s_voff = 0;
  uint32_t z_voff[kLutZ ? B_PER : 1];
  int z_sh[kLutZ ? B_PER : 1];
  if constexpr (!kFp4) {
#pragma unroll
    for (int i = 0; i < B_PER; ++i) {
      const int c = (int)threadIdx.x + i * T;
      bool ok;
      const int gs = gstrip(c >> 6, ok);
      if constexpr (kStripS) b_strip[i] = __builtin_amdgcn_readfirstlane(gs);
      b_voff[i] = (uint32_t)(((size_t)(kStripS ? 0 : gs) * KT * 64 + (c & 63)) * 16);
      if constexpr (kLutZ) {
        z_voff[i] = zero_word(lane, (kStripS ? 0 : gs * 16) + (lane & 15), GPT, N);
        z_sh[i] = 4 * (lane & 7);
      }
    }
    bool ok;
    const int sc_s = sc_c % (NSTRIP * 2), sc_g = sc_c / (NSTRIP * 2);
    s_voff = scale_piece(sc_g, gstrip(sc_s >> 1, ok), sc_s & 1, N);
  }

  // int4 register sets, one per stage index (two are live at a time)
  v4u rbw[NST][kFp4 ? 1 : B_PER];
  uint4 rsc[NST];
  uint32_t rzp[NST][kLutZ ? B_PER : 1][ZL > 0 ? ZL : 1];

  // loads of K step kt into stage I (DMA) / register set I (int4 weights, scales, zeros)
  // part: 1 = the A DMAs (and fp4 strips / E8M0 bytes), 2 = the int4 weight, scale and zero loads.
  // Tail: steps past the last read empty buffers (at the last step's offsets): those loads touch no
  // memory and nothing uses what they bring, so every step issues the same instructions and the one
  // vmcnt count holds to the end.
  auto issue = [&](auto I, int kt, int part, auto Tail) __attribute__((always_inline)) {
    constexpr int R = decltype(I)::value;
    unsigned char* st = stage(I);
    constexpr bool kRagged = kKTail && decltype(Tail)::value;  // the last tile is always loaded by a tail step
    const uint32_t live = decltype(Tail)::value ? (uint32_t)__builtin_amdgcn_readfirstlane(kt < KT ? -1 : 0) : 0xffffffffu;
    if constexpr (decltype(Tail)::value) kt = kt < KT ? kt : KT - 1;
    const BufRsrc rs_a = make_rsrc(p.xq - kABase, live);
    const BufRsrc rs_w = make_rsrc(wt, w_bytes & live);
    const BufRsrc rs_s = make_rsrc(scales, s_bytes & live);
    const BufRsrc rs_z = make_rsrc(zeros, z_bytes & live);
    const BufRsrc rs_seed = make_rsrc(p.seeds, seed_bytes & live);
    if constexpr (kFp4) {
#pragma unroll
      for (int i = 0; i < S_DMA; ++i) {  // scale rows past K: out of the buffer's range, so zeros
        const BufOffset o = row_step(e_voff[i], (uint32_t)__builtin_amdgcn_readfirstlane(kt * 4 * N), kRagged);
        lds_dma4(rs_s, st + S::kA + S::kB + (wave + i * NW) * 256, o.v, o.s);
      }
    }
    const uint32_t so_a = (uint32_t)__builtin_amdgcn_readfirstlane(AT ? kt * 2048 : kt * kTileK);
    if (part & 1) {
      const uint32_t last = kRagged ? (uint32_t)__builtin_amdgcn_readfirstlane(kt == KT - 1 ? -1 : 0) : 0u;
#pragma unroll
      for (int i = 0; i < A_PER; ++i)
        lds_dma16(rs_a, st + (wave + i * NW) * 1024, a_step(a_voff[i], back, last), so_a);
      if constexpr (kSeedL)
        lds_dma4(rs_seed, st + kSeedOff + (wave % kSeedW) * 256, seed_voff,
                 (uint32_t)__builtin_amdgcn_readfirstlane(kt * (int)p.seeds_ld * 4));
    }
    if constexpr (kFp4) {
#pragma unroll
      for (int i = 0; i < B_DMA; ++i)
        lds_dma16(rs_w, st + S::kA + (wave + i * NW) * 1024, (uint32_t)lane * 16,
                    (uint32_t)__builtin_amdgcn_readfirstlane((b_gs[i] * KT + kt) * kTileBytes));
    } else if (part & 2) {
      const uint32_t so_b = (uint32_t)__builtin_amdgcn_readfirstlane(kt * kTileBytes);
#pragma unroll
      for (int i = 0; i < B_PER; ++i)
        rbw[R][i] = bload128v(rs_w, b_voff[i], kStripS ? (uint32_t)__builtin_amdgcn_readfirstlane((b_strip[i] * KT + kt) * kTileBytes) : so_b);
      const int g = GPT > 1 ? kt * GPT : kt >> gshift;
      const BufOffset o = row_step(s_voff, (uint32_t)__builtin_amdgcn_readfirstlane(g * N * 2), kRagged);
      rsc[R] = bload128(rs_s, o.v, o.s);  // scale and zero rows past K: out of the buffers' ranges, so zeros
      if constexpr (kLutZ) {
#pragma unroll
        for (int i = 0; i < B_PER; ++i)
#pragma unroll
          for (int h = 0; h < ZL; ++h) {
            const uint32_t so_z = (uint32_t)__builtin_amdgcn_readfirstlane((g + h * (GPT / 2)) * (N / 8) * 4 + (kStripS ? b_strip[i] * 8 : 0));
            const BufOffset oz = row_step(z_voff[i], so_z, kRagged);
            rzp[R][i][h] = bload32(rs_z, oz.v, oz.s);
          }
      }
    }
  };
  // int4: unpack register set R into stage I
  auto commit = [&](auto I, auto R_) __attribute__((always_inline)) {
    if constexpr (!kFp4) {
      constexpr int R = decltype(R_)::value;
      unsigned char* st = stage(I);
      unsigned char* sb = st + S::kA;
#pragma unroll
      for (int i = 0; i < B_PER; ++i) {
        const int c = (int)threadIdx.x + i * T;
        const int s = c >> 6, l = c & 63;
        const uint4 w = make_uint4(rbw[R][i].x, rbw[R][i].y, rbw[R][i].z, rbw[R][i].w);
        v8i u;
        if constexpr (kLutZ) {
          const uint4 t0 = zlut[(rzp[R][i][0] >> z_sh[i]) & 15u];
          const uint4 t1 = ZL > 1 ? zlut[(rzp[R][i][ZL - 1] >> z_sh[i]) & 15u] : t0;
          u = unpack_tile_lut(w, t0, t1);
        } else if constexpr (kLut) {
          u = unpack_tile_lut(w, zero_point_lut(8), zero_point_lut(8));
        } else {
          u = unpack_tile_int4(w);
        }
        *reinterpret_cast<uint4*>(sb + ((s * 2 + 0) * 64 + l) * 16) = make_uint4(u[0], u[1], u[2], u[3]);
        *reinterpret_cast<uint4*>(sb + ((s * 2 + 1) * 64 + l) * 16) = make_uint4(u[4], u[5], u[6], u[7]);
      }
      *reinterpret_cast<uint4*>(st + S::kA + S::kB + sc_c * 16) = rsc[R];
    }
  };

  v4f acc[RB][NSB];
#pragma unroll
  for (int rb = 0; rb < RB; ++rb)
#pragma unroll
    for (int j = 0; j < NSB; ++j) acc[rb][j] = v4f{0.f, 0.f, 0.f, 0.f};
  const v4f zero4 = v4f{0.f, 0.f, 0.f, 0.f};

  // per-lane LDS offsets of this wave's operands within a stage; the empty asm keeps each in one
  // VGPR so every read is that VGPR plus an immediate
  // GPT > 1: 8-byte operands of the 16x16x32 MFMA, lane (row, q) holding K 8q.. of each 32: chunk
  // q / 2 of the 16-byte chunks, half q % 2
  const int lo = GPT > 1 ? (((lane >> 5) * 16 + (lane & 15)) * 16 + ((lane >> 4) & 1) * 8) : lane * 16;
  uint32_t oa = (uint32_t)(wm * RB * 2048 + lo);
  uint32_t ob = (uint32_t)(S::kA + wn * NSB * (kFp4 ? 1024 : 2048) + lo);
  uint32_t os = (uint32_t)(S::kA + S::kB + (kFp4 ? wn * NSB * 256 + lane : (wn * NSB * 16 + (lane & 15)) * 2));
  asm volatile("" : "+v"(oa), "+v"(ob), "+v"(os));

  // MFMA work of one K step from stage I (operands read one row block / strip ahead of their
  // MFMAs). mid(i) runs right after the MFMAs of int4 strip i (i = 0, 1) or MXFP4 row block i, so
  // its work (the loads of a later step, the unpack of the next step's weights) overlaps MFMAs in
  // flight. Waves of two row blocks and four strips have few MFMAs to hide it behind and wait on LDS instead:
  // there mid(0) fills the wait for the step's first operands (K=4096 N=6144 M=512 30.9 against 30.0
  // us, K=2816 N=2048 M=2048 in groups of 32 43.2 against 42.1; 256-row tiles equal or 1% slower).
  constexpr bool kMidFirst = RB <= 2 && NSB > 2;
  auto compute = [&](auto I, auto mid, int valid) __attribute__((always_inline)) {
    const unsigned char* st = stage(I);
    // valid: the tile's K (128 but for a ragged last one, whose operand bytes past it are cleared)
    const bool mlo = 16 * (lane >> 4) < valid, mhi = 64 + 16 * (lane >> 4) < valid;
    auto a_operand = [&](const unsigned char* at) __attribute__((always_inline)) {
      v8i a = lds_operand(at, 0);
      if constexpr (kKTail) {
#pragma unroll
        for (int i = 0; i < 8; ++i) a[i] = (i < 4 ? mlo : mhi) ? a[i] : 0;
      }
      return a;
    };
    if constexpr (kFp4) {
      uint4 braw[NSB];
      int sbyte[NSB];
#pragma unroll
      for (int j = 0; j < NSB; ++j) {
        braw[j] = *reinterpret_cast<const uint4*>(st + ob + j * 1024);
        sbyte[j] = (int)st[os + j * 256];
      }
      v8i a0 = a_operand(st + oa);
#pragma unroll
      for (int rb = 0; rb < RB; ++rb) {
        v8i a1;
        if (rb + 1 < RB) a1 = a_operand(st + oa + (rb + 1) * 2048);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int j = 0; j < NSB; ++j) acc[rb][j] = mfma_f8f4_sb(a0, fp4_operand(braw[j]), acc[rb][j], sbyte[j]);
        mid(rb);
        if (rb + 1 < RB) a0 = a1;
      }
    } else if constexpr (GPT > 1) {
      // the tile in 32-wide pieces, piece s at byte (s / 2) * 1024 + (s % 2) * 512 of the 16-row block
      constexpr int PPG = 4 / GPT;  // pieces per group
      long a[RB][4];
#pragma unroll
      for (int rb = 0; rb < RB; ++rb)
#pragma unroll
        for (int s = 0; s < 4; ++s)
          a[rb][s] = 32 * s < valid ? *reinterpret_cast<const long*>(st + oa + rb * 2048 + (s >> 1) * 1024 + (s & 1) * 512) : 0;
      long bn[4];
#pragma unroll
      for (int s = 0; s < 4; ++s) bn[s] = *reinterpret_cast<const long*>(st + ob + (s >> 1) * 1024 + (s & 1) * 512);
      float scn[GPT];
#pragma unroll
      for (int g = 0; g < GPT; ++g) scn[g] = f16_to_f32(*reinterpret_cast<const uint16_t*>(st + os + g * NSTRIP * 32));
      v4f cp[RB];
      float scp = 0.f;
      if constexpr (kMidFirst) {
        __builtin_amdgcn_sched_barrier(0);
        mid(0);
      }
#pragma unroll
      for (int j = 0; j < NSB; ++j) {
        long b[4];
        float sc[GPT];
#pragma unroll
        for (int s = 0; s < 4; ++s) b[s] = bn[s];
#pragma unroll
        for (int g = 0; g < GPT; ++g) sc[g] = scn[g];
        if (j + 1 < NSB) {
#pragma unroll
          for (int s = 0; s < 4; ++s)
            bn[s] = *reinterpret_cast<const long*>(st + ob + (j + 1) * 2048 + (s >> 1) * 1024 + (s & 1) * 512);
#pragma unroll
          for (int g = 0; g < GPT; ++g)
            scn[g] = f16_to_f32(*reinterpret_cast<const uint16_t*>(st + os + g * NSTRIP * 32 + (j + 1) * 32));
        }
#pragma unroll
        for (int g = 0; g < GPT; ++g) {
          // keeps one group's partials live at a time (and the one before it, below)
          __builtin_amdgcn_sched_barrier(0);
          v4f cj[RB];
#pragma unroll
          for (int rb = 0; rb < RB; ++rb) {
            cj[rb] = __builtin_amdgcn_mfma_f32_16x16x32_fp8_fp8(a[rb][g * PPG], b[g * PPG], zero4, 0, 0, 0);
            if constexpr (PPG == 2)
              cj[rb] = __builtin_amdgcn_mfma_f32_16x16x32_fp8_fp8(a[rb][g * PPG + 1], b[g * PPG + 1], cj[rb], 0, 0, 0);
          }
          if (g == GPT - 1 && j < 2 && (j > 0 || !kMidFirst)) mid(j);
          // the previous group's scale FMAs run between this group's MFMAs
          if (j > 0 || g > 0) {
            const int jp = g > 0 ? j : j - 1;
#pragma unroll
            for (int rb = 0; rb < RB; ++rb)
#pragma unroll
              for (int r = 0; r < 4; ++r) acc[rb][jp][r] += scp * cp[rb][r];
#pragma unroll
            for (int rb = 0; rb < RB; ++rb) {
              __builtin_amdgcn_sched_group_barrier(0x008, PPG, 0);
              __builtin_amdgcn_sched_group_barrier(0x002, 4, 0);
            }
          }
#pragma unroll
          for (int rb = 0; rb < RB; ++rb) cp[rb] = cj[rb];
          scp = sc[g];
        }
      }
#pragma unroll
      for (int rb = 0; rb < RB; ++rb)
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[rb][NSB - 1][r] += scp * cp[rb][r];
    } else {
      v8i a[RB];
#pragma unroll
      for (int rb = 0; rb < RB; ++rb) a[rb] = lds_operand(st + oa + rb * 2048, 0);
      v4f pre[RB];
#pragma unroll
      for (int rb = 0; rb < RB; ++rb) {  // symmetric: -R/2 undoes the codes' half step
        if constexpr (kLut)
          pre[rb] = zero4;
        else if constexpr (kSeedL)
          pre[rb] = *reinterpret_cast<const v4f*>(st + kSeedOff + (wm * RB * 16 + rb * 16 + 4 * (lane >> 4)) * 4);
        else
          pre[rb] = mfma_f8f8(a[rb], splat8(0xB0B0B0B0u), zero4);
      }
      v4f cp[RB];
      float scp = 0.f;
      v8i bn = lds_operand(st + ob, 0);
      float scn = f16_to_f32(*reinterpret_cast<const uint16_t*>(st + os));
      if constexpr (kMidFirst) {
        __builtin_amdgcn_sched_barrier(0);
        mid(0);
      }
#pragma unroll
      for (int j = 0; j <= NSB; ++j) {
        v4f cj[RB];
        float scj = 0.f;
        if (j < NSB) {
          const v8i b = bn;
          scj = scn;
          if (j + 1 < NSB) {
            bn = lds_operand(st + ob + (j + 1) * 2048, 0);
            scn = f16_to_f32(*reinterpret_cast<const uint16_t*>(st + os + (j + 1) * 32));
          }
          __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int rb = 0; rb < RB; ++rb) cj[rb] = mfma_f8f8(a[rb], b, pre[rb]);
          if (j < 2 && (j > 0 || !kMidFirst)) mid(j);
        }
        if (j > 0) {
#pragma unroll
          for (int rb = 0; rb < RB; ++rb)
#pragma unroll
            for (int r = 0; r < 4; ++r) acc[rb][j - 1][r] += scp * cp[rb][r];
          // issue the previous strip's scale FMAs between this strip's MFMAs (one MFMA, then four
          // VALU ops), so they run while the matrix pipe works instead of after it
          if (j < NSB) {
#pragma unroll
            for (int rb = 0; rb < RB; ++rb) {
              __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
              __builtin_amdgcn_sched_group_barrier(0x002, 4, 0);
            }
          }
        }
        if (j < NSB) {
#pragma unroll
          for (int rb = 0; rb < RB; ++rb) cp[rb] = cj[rb];
          scp = scj;
        }
      }
    }
  };

  // one pipelined step kt (stage C = kt % NST): loads of kt+D, MFMAs of kt, int4 registers of kt+1
  // to LDS, wait for kt+1's loads, barrier. The loads of kt+D are issued between the step's MFMAs
  // instead of ahead of them all (int4: the weight loads after the first strip's, ahead of the
  // unpack of kt+1's weights, and the A DMAs after the second's; MXFP4: all after the second row
  // block's): at the top of the step every wave's loads would meet in the address unit's queue
  // while the step's first MFMAs wait (1-4% on int4 and MXFP4 shapes from 2048 rows). The weight
  // registers go first because the unpack one step later waits on them, while the A DMAs are only
  // waited for at the end of the next step (weights first: int4 2-8% faster from 2048 rows, MoE T=4096 2%).
  auto step = [&](auto C, int kt, auto Tail) __attribute__((always_inline)) {
    if (decltype(Tail)::value && kt >= KT) return;
    constexpr int c = decltype(C)::value, n1 = (c + 1) % NST, nd = (c + D) % NST;
    static_assert(kFp4 || NSB >= 2, "int4 steps issue their loads after strips 0 and 1");
    const int valid = decltype(Tail)::value && kKTail && kt == KT - 1 ? ktail : kTileK;
    if constexpr (kFp4) {
      compute(C, [&](int rb) __attribute__((always_inline)) {
        // past the last step nothing is loaded (unlike int4 below, whose unpack the branch would hold
        // back, MXFP4 is 2% faster at M=1000 K=N=4096 with the branch than with empty loads)
        if (rb == 1 && (!decltype(Tail)::value || kt + D < KT)) issue(IC<nd>{}, kt + D, 3, Tail);
      }, valid);
    } else {
      compute(C, [&](int j) __attribute__((always_inline)) {
        if (j == 0) {
          issue(IC<nd>{}, kt + D, 2, Tail);
          if (!decltype(Tail)::value || kt + 1 < KT) commit(IC<n1>{}, IC<n1>{});
        } else {
          issue(IC<nd>{}, kt + D, 1, Tail);
        }
      }, valid);
    }
    __builtin_amdgcn_sched_barrier(0);
    if (kFp4 && decltype(Tail)::value && kt + D >= KT) wait_vm_lgkm0<0>();
    else wait_vm_lgkm0<NOPS * (D - 1)>();
    __builtin_amdgcn_s_barrier();
  };
  // prologue: steps 0 and 1 in flight, step 0 in LDS. The epilogue rows' loads above are older
  // than both, so the counted wait covers them; their LDS writes land before the first step's
  // barrier (its wait takes lgkmcnt to 0), long before the epilogue reads them.
  issue(IC<0>{}, 0, 3, IC<0>{});
  for_stages<1, D>([&](auto I) __attribute__((always_inline)) { issue(I, decltype(I)::value, 3, IC<1>{}); });
  if constexpr (kLutZ) lds_barrier();  // the zero-point table, before the first decode reads it
  commit(IC<0>{}, IC<0>{});
  wait_vm_lgkm0<NOPS * (D - 1)>();
  if (er < BM) {
    e_sc[er] = er_sc;
    e_ok[er] = er_ok ? 1 : 0;
  }
  __builtin_amdgcn_s_barrier();
  int kt = 0;
  for (; kt + NST - 1 + D + (kKTail ? 1 : 0) < KT; kt += NST)  // kKTail: loads of steps up to KT - 2 only
    for_stages<0, NST>([&](auto I) __attribute__((always_inline)) { step(I, kt + decltype(I)::value, IC<0>{}); });
  for_stages<0, NST - 1 + D + (kKTail ? 1 : 0)>([&](auto I) __attribute__((always_inline)) {
    constexpr int i = decltype(I)::value;
    step(IC<i % NST>{}, kt + i, IC<1>{});
  });
  // the empty loads of the last steps write LDS too: all landed before the epilogue reuses it
  wait_vm_lgkm0<0>();
  __builtin_amdgcn_s_barrier();

  // epilogue: lane holds rows 4*(lane>>4)+r of each row block, channel (lane & 15) of each strip
  const int64_t row0 = blk_row0 + (int64_t)wm * RB * 16;
  float e_rsc[RB][4];
  uint32_t e_valid = 0;
#pragma unroll
  for (int rb = 0; rb < RB; ++rb)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int lr = wm * RB * 16 + rb * 16 + 4 * (lane >> 4) + r;
      e_rsc[rb][r] = e_sc[lr];
      e_valid |= (e_ok[lr] ? 1u : 0u) << (rb * 4 + r);
    }
  // the stages are free: the last step's barrier followed every wave's reads and every DMA
  constexpr int kScr = 16 * (NSB * 16 * 4 + 16);  // one wave's row-major tile, f32 worst case
  constexpr int kWps = kStage / kScr;
  static_assert(3 * kWps >= NW && NOPS * (D - 1) < 64, "epilogue scratch, vmcnt");
  unsigned char* scr = (wave < kWps ? st0 : wave < 2 * kWps ? st1 : st2) + (wave % kWps) * kScr;
  store_tile_scaled(p, acc, e_rsc, e_valid, row0, lane,
                    [&](int j, bool& ok) __attribute__((always_inline)) { return gstrip(wn * NSB + j, ok); }, scr);
}

template <int WM, int WN, int RB, int NSB, int NST, int MODE, bool AT = false>
static int launch_dma_cfg_at(const GemmArgs& p, int64_t row_tiles, hipStream_t stream) {
  constexpr int BN = WN * NSB * 16;
  const int64_t ncols = p.silu ? p.N / 2 : p.N;
  const int64_t colw = p.silu ? BN / 2 : BN;
  const int64_t gx = (ncols + colw - 1) / colw;
  int64_t gy = row_tiles;
  if (p.sorted_ids)  // the grouped tile order needs a multiple of 8 workgroups
    while ((gx * gy) % 8) ++gy;
  const dim3 grid((unsigned)gx, (unsigned)gy);
  const dim3 block(WM * WN * 64);
  auto kern = gemm_dma_kernel<WM, WN, RB, NSB, NST, MODE, AT>;
  hipLaunchKernelGGL(kern, grid, block, 0, stream, p);
  return hipGetLastError() == hipSuccess ? kOk : kErrHip;
}

// int4; p.a_tiled takes the tiled-A instantiation (groups of 64 and 32 are row-major)
template <int WM, int WN, int RB, int NSB, int NST, bool AT>
static int launch_dma_int4(const GemmArgs& p, int mode, int64_t row_tiles, hipStream_t stream) {
  switch (mode) {
    case kPSym:
      if constexpr (AT) {
        if (p.a_tiled) return launch_dma_cfg_at<WM, WN, RB, NSB, NST, kPSym, true>(p, row_tiles, stream);
      }
      return launch_dma_cfg_at<WM, WN, RB, NSB, NST, kPSym>(p, row_tiles, stream);
    case kPAsym:
      if constexpr (AT) {
        if (p.a_tiled) return launch_dma_cfg_at<WM, WN, RB, NSB, NST, kPAsym, true>(p, row_tiles, stream);
      }
      return launch_dma_cfg_at<WM, WN, RB, NSB, NST, kPAsym>(p, row_tiles, stream);
    case kPG64: return launch_dma_cfg_at<WM, WN, RB, NSB, NST, kPG64>(p, row_tiles, stream);
    case kPG64Z: return launch_dma_cfg_at<WM, WN, RB, NSB, NST, kPG64Z>(p, row_tiles, stream);
    case kPG32: return launch_dma_cfg_at<WM, WN, RB, NSB, NST, kPG32>(p, row_tiles, stream);
    default: return launch_dma_cfg_at<WM, WN, RB, NSB, NST, kPG32Z>(p, row_tiles, stream);
  }
}
template <int WM, int WN, int RB, int NSB, int NST, bool AT>
static int launch_dma_mx(const GemmArgs& p, int64_t row_tiles, hipStream_t stream) {
  if constexpr (AT) {
    if (p.a_tiled) return launch_dma_cfg_at<WM, WN, RB, NSB, NST, kPE8M0, true>(p, row_tiles, stream);
  }
  return launch_dma_cfg_at<WM, WN, RB, NSB, NST, kPE8M0>(p, row_tiles, stream);
}

// grouped tiles: A rows gathered through the sorted ids, or (p.a_tiled, int4 in groups of 128+, A rows at
// their padded positions: gemm2) the padded rows' codes in operand order with their seeds
template <int WM, int WN, int RB, int NSB>
static int launch_dma_grouped(const GemmArgs& p, int mode, int64_t row_tiles, hipStream_t stream) {
  if (mode == kPE8M0) return launch_dma_mx<WM, WN, RB, NSB, 3, false>(p, row_tiles, stream);
  return launch_dma_int4<WM, WN, RB, NSB, 3, true>(p, mode, row_tiles, stream);
}

// Dense tile shapes (pick_tile) and what a K step of a full round of workgroups (one per CU) costs, relative to the
// format's largest tile. A wave of the smaller ones has fewer MFMAs behind each LDS operand and
// barrier, so their cost per output is higher; what they win is a grid that fills the 256 CUs. The two
// smallest fit a CU twice and are measured at up to 256 workgroups (a round of the 64 x 128 one is
// twice 256, at twice the cost). us per K step of a round, int4 symmetric: 1.26 / 1.02 / 0.78 / 0.54 /
// 0.46; MXFP4: 1.41 / 1.13 / 0.85 / 0.70 / 0.63 / 0.46 / 0.40. Zero points and groups of 64 and 32 raise
// all of a format's tiles alike (256 x 128: 1.29, 2.0 and 2.4).
static const DmaTile kInt4Tiles[] = {{256, 128, 1.0f}, {192, 128, 0.81f}, {128, 128, 0.64f}, {64, 128, 0.45f}, {64, 64, 0.38f}};
// with the activations in operand order also gemm_prefill_wide.hip's tile (2.08 us)
static const DmaTile kInt4TiledA[] = {{256, 128, 1.0f}, {192, 128, 0.81f}, {128, 128, 0.64f}, {64, 128, 0.45f},
                                      {64, 64, 0.38f}, {256, 256, 1.65f}};
static const DmaTile kMxTiles[] = {{256, 256, 1.0f}, {192, 256, 0.80f}, {128, 256, 0.60f}, {192, 128, 0.50f},
                                   {128, 128, 0.45f}, {64, 128, 0.33f}, {64, 64, 0.29f}};

// the tile that launch_prefill_dma gives a dense call, its activations in operand order or not
DmaTile prefill_tile(const GemmArgs& p, bool a_tiled) {
  if (p.wfmt == kE2M1) return kMxTiles[pick_tile(kMxTiles, p, p.M)];
  return a_tiled ? kInt4TiledA[pick_tile(kInt4TiledA, p, p.M)] : kInt4Tiles[pick_tile(kInt4Tiles, p, p.M)];
}

// int4 with groups of 32, 64 and 128+ and MXFP4, on 16-byte aligned rows; kErrUnsupported otherwise.
// bm_rows: rows per workgroup the caller requires (grouped: 64 or 128; 0 for dense).
int launch_prefill_dma(const GemmArgs& p, int64_t rows_to_cover, int bm_rows, hipStream_t stream) {
  int mode;
  if (p.wfmt == kInt4 && p.sfmt == kScaleF16 && p.group % kTileK == 0)
    mode = p.zeros ? kPAsym : kPSym;
  else if (p.wfmt == kInt4 && p.sfmt == kScaleF16 && p.group == 64)
    mode = p.zeros ? kPG64Z : kPG64;
  else if (p.wfmt == kInt4 && p.sfmt == kScaleF16 && p.group == 32)
    mode = p.zeros ? kPG32Z : kPG32;
  else if (p.wfmt == kE2M1 && p.sfmt == kScaleE8M0)
    mode = kPE8M0;
  else
    return kErrUnsupported;
  if (p.silu && (p.N / kTileN) % 2) return kErrUnsupported;
  // a K that ends inside its first tile has no tile before it for the chunks past K to read
  if (p.K % kTileK && (p.KT < 2 || p.a_tiled)) return kErrUnsupported;
  // grouped rows: a workgroup's rows must sit inside one align block (one expert)
  if (p.sorted_ids && bm_rows != 64 && bm_rows != 128) return kErrUnsupported;
  // 32-bit offsets within one matrix
  if ((int64_t)p.N * p.KT * 64 >= (int64_t)1 << 31) return kErrUnsupported;
  if (p.ldx % 16) return kErrUnsupported;  // A rows are read in 16-byte pieces, at 32-bit offsets
  if ((p.a_by_token ? p.num_slots / p.top_k : p.M) * p.ldx > (int64_t)0xffffffff - kABias) return kErrUnsupported;
  if (p.a_tiled && (p.sorted_ids ? ((mode != kPSym && mode != kPAsym) || p.a_by_token != 0)
                                 : (bm_rows != 0 || prefill_gpt(mode) > 1)))
    return kErrUnsupported;
  if (bm_rows == 64) return launch_dma_grouped<2, 4, 2, 2>(p, mode, (rows_to_cover + 63) / 64, stream);
  if (bm_rows == 128) return launch_dma_grouped<2, 4, 4, 4>(p, mode, (rows_to_cover + 127) / 128, stream);
  // Dense tiles (waves WM x WN, wave tile RB x NSB blocks of 16). The largest are those whose three
  // stages fit the 160 KiB of LDS and whose registers fit two waves per SIMD. MXFP4 keeps its weights
  // as fp4 in LDS and its accumulators are the only per-step state, so it takes 64 x 128 wave tiles
  // (256 x 256 per workgroup: a quarter less LDS read per MFMA than 64 x 64); int4 holds the unpacked
  // fp8 weights plus the partials of its per-group scaling and stays at 64 x 64. The 64 x 64 tile takes
  // four stages (two of its workgroups still fit a CU; AWQ M=100 K=4096 N=6144 22.9 -> 21.1 us, more
  // stages gained nothing).
  if (mode == kPE8M0) {
    const int t = pick_tile(kMxTiles, p, rows_to_cover);
    const int64_t rt = (rows_to_cover + kMxTiles[t].bm - 1) / kMxTiles[t].bm;
    switch (t) {
      case 0: return launch_dma_mx<4, 2, 4, 8, 3, true>(p, rt, stream);
      case 1: return launch_dma_mx<4, 2, 3, 8, 3, true>(p, rt, stream);
      case 2: return launch_dma_mx<4, 2, 2, 8, 3, true>(p, rt, stream);
      case 3: return launch_dma_mx<4, 2, 3, 4, 3, true>(p, rt, stream);
      case 4: return launch_dma_mx<4, 2, 2, 4, 3, true>(p, rt, stream);
      case 5: return launch_dma_mx<2, 4, 2, 2, 3, true>(p, rt, stream);
      default: return launch_dma_mx<2, 2, 2, 2, 4, true>(p, rt, stream);
    }
  }
  const int t = p.a_tiled ? pick_tile(kInt4TiledA, p, rows_to_cover) : pick_tile(kInt4Tiles, p, rows_to_cover);
  const int64_t rt = (rows_to_cover + kInt4TiledA[t].bm - 1) / kInt4TiledA[t].bm;
  switch (t) {
    case 0: return launch_dma_int4<4, 2, 4, 4, 3, true>(p, mode, rt, stream);
    case 1: return launch_dma_int4<4, 2, 3, 4, 3, true>(p, mode, rt, stream);
    case 2: return launch_dma_int4<4, 2, 2, 4, 3, true>(p, mode, rt, stream);
    case 3: return launch_dma_int4<2, 4, 2, 2, 3, true>(p, mode, rt, stream);
    case 4: return launch_dma_int4<2, 2, 2, 2, 4, true>(p, mode, rt, stream);
    default: return launch_prefill_wide(p, rows_to_cover, stream);
  }
}

// The LDS-staged kernels: NVFP4 on the fp16 MFMA, else the DMA-staged pipeline; kErrUnsupported for
// what neither takes (the per-wave kernel serves it).
int launch_prefill_staged(const GemmArgs& p, int64_t rows_to_cover, int bm_rows, hipStream_t stream) {
  const int rc = launch_prefill_nv(p, rows_to_cover, bm_rows, stream);
  return rc != kErrUnsupported ? rc : launch_prefill_dma(p, rows_to_cover, bm_rows, stream);
}

}  // namespace w4a8
