// MXFP4 / MXFP8 tile kernel with a deep operand ring, for problems of one round of tiles (gfx950, MI355X).
//
// What bounds these problems: with one workgroup or less per CU nothing covers a request's way to HBM or to the memory
// side cache (about 1 us, 2 under load) but the requests that the workgroup itself has in flight.  The five-slot ring of
// the tile kernel (mxfp4_gemm_tile.hip), which is sized for two workgroups per CU and for the matrix pipes, gives the
// second half of a K tile of B a lead of three quarters of a K tile, and its per-lane scale loads, one K tile ahead in
// the same in-order queue, no more: 0.72 us per K tile of a 128x128 tile, whose MFMAs take 0.2.  Here
//   * LDS is one ring of 3 (128x256, 256x128, 128x192) or 4 whole K tiles (a stream of B with few rows: 8 of 64x64), requested that
//     many ahead.  More of the small tiles than four only put requests in front of the first K tile, which the workgroup
//     issues before it can wait for it (64x64 with 8 -> 4, 64x128 with 6 -> 4; us by name: 1024 x 1024 x 1024 5.1 -> 4.6,
//     1024 x 1024 x 3840 8.3 -> 7.6, 512 x 2048 x 2048 7.2 -> 6.6, 64 x 14336 x 4096 12.7 -> 11.9; over 3000 random calls the
//     ones on these tiles take 0.94 of the time);
//   * the scales travel in the ring too (one 256-byte block per 32 rows and K tile, four bytes per lane), so that no
//     load that returns to a register stands in the queue in front of the operands; row-major scales of up to 31 K tiles
//     (the largest tiles: 5, 128x192: 15) are staged once per workgroup instead, and then no launch has to re-lay them
//     (186 x 4832 x 5888 17.0 -> 10.9 us, 644 x 5888 x 2304 17.1 -> 12.0);
//   * the tiles are small enough for the problem to reach most CUs without a split along K (64x64 up to 256 of them),
//     which saves the launch that adds the parts, and the parts.
// Measured (us per call through the C ABI, weights from HBM, bf16 C, scales resident unless said, the kernel that the library
// took before -> its choice of tile and parts here, both on one box):
//   1024 x 1024 x 1024 row-major scales, f32 C 7.9 -> 5.8    128 x 3840 x 4096 12.8 -> 9.4    387 x 2048 x 4096 15.8 -> 8.7
//   326 x 3584 x 5376 18.6 -> 12.6    512 x 8192 x 8192 31.3 -> 24.6    1813 x 2624 x 9728 39.5 -> 32.8
//   1000 x 7168 x 4096 22.7 -> 20.3    2048 x 4096 x 14336 66.5 -> 61.2    1 x 4096 x 6080 15.7 -> 8.1
//   727 x 4096 x 11008 row-major 43.0 -> 34.1
// MXFP8 (the tile kernels with their re-layout launch before -> now): 675 x 1760 x 11136 111 -> 37, 290 x 4608 x 7424
//   40.2 -> 23.4, 64 x 1856 x 2048 18.7 -> 7.7, 907 x 1024 x 2560 20.3 -> 9.4.
// 128x192 tiles lie between: 526 x 7424 x 3584 15.6 (on 256x128) -> 14.2, 256 x 24576 x 8192 37.9 -> 35.4; among random shapes that
// take them 0.93 of the time.  Tiles of an odd count of 32 columns (64x96 .. 128x224, the waves in two halves of K whose
// sums meet in LDS) were no faster than the even ones beside them, and are not built.
// Eight waves (two per SIMD) beat four on 128x128 by 1-4 % and on 128x256 by 3-9 %; 64x256 tiles and more than one round
// (two workgroups of the tile kernel share a CU there, and the persistent kernel streams across tiles) lost and are not
// built.  A time per K tile of 0.21-0.30 us at 64x64 up to 0.93 at 128x256 leaves the fixed part (launch, first K tile,
// C: 3.3-6.7 us) as what bounds short K.  On a full grid of the largest tiles it is the step: 2048 x 4096 x 14336 takes 65 us on
// random operands and 54 on zeros (256x128: 66 and 56; 61 and 51 on a faster card), 1000 x 7168 x 4096 22.5 and 17.2, so a fifth to a quarter
// is the matrix pipes' power limit.  What holds the rest is not established.  It is no limit of a CU's L1 or of what stands
// behind it: 67 lines of 128 bytes are under way and 0.185 arrive a cycle, where the same requests alone reach 144 and 0.42; no
// bank conflicts, MFMAs busy 46 % of the cycles (profiles/pmc_deep_ring_l1_requests.txt).
#ifndef WAVE_MXFP4_GEMM_DEEP_H_
#define WAVE_MXFP4_GEMM_DEEP_H_
#include <type_traits>

#include "mxfp4_tile_common.h"

namespace wave_mxfp4 {

namespace {

// How the scales reach a lane: a 256-byte block per 32 rows and K tile in MFMA32 order (one dword per lane) or in
// e8m0_shuffle order (two dwords and a byte permute), fetched into the ring beside the operands; or row-major, the
// rows of the workgroup's K range copied into LDS once.
enum DeepScales { kDeepNative = 0, kDeepShuffled = 1, kDeepRows = 2 };

template <int BM_, int BN_, int WAVES_M_, int WAVES_N_, int STAGES_>
struct DeepCfg {
  static constexpr int BM = BM_, BN = BN_, WAVES_M = WAVES_M_, WAVES_N = WAVES_N_, STAGES = STAGES_;
  static constexpr int NWAVES = WAVES_M * WAVES_N, NT = NWAVES * 64;
  static constexpr int WM = BM / WAVES_M, WN = BN / WAVES_N;  // per-wave tile
  static constexpr int MT_M = WM / 32, MT_N = WN / 32;        // 32x32 MFMA tiles per wave
  static constexpr int A_BYTES = BM * kTileKBytes, B_BYTES = BN * kTileKBytes;
  static constexpr int SB = (BM + BN) / 32;                   // 32-row scale blocks of a K tile
  static constexpr int A_LD = BM / 8 / NWAVES, B_LD = BN / 8 / NWAVES, S_LD = (SB + NWAVES - 1) / NWAVES;
  static constexpr int STAGE = A_BYTES + B_BYTES;
  static constexpr int RING = STAGES * STAGE, S_STAGE = SB * 256, S_RING = STAGES * S_STAGE;
  static_assert(BM % (8 * NWAVES) == 0 && BN % (8 * NWAVES) == 0 && NWAVES % 2 == 0, "operand tiles split over the waves' DMA");
  static_assert(WM % 32 == 0 && WN % 32 == 0 && STAGES >= 3 && RING + S_RING <= 160 * 1024, "wave tile; ring");
  static_assert(NWAVES * WM * (WN * 4 + 16) <= 160 * 1024, "C staging");
};
// The tile shapes by their index (kDeepShapes in mxfp4_api.hip): `f` on the configuration, `none` for any other index
template <class R, class F>
R with_deep_shape(int shape, R none, F f) {
  switch (shape) {
    case 0: return f(DeepCfg<64, 64, 2, 2, 4>{});
    case 1: return f(DeepCfg<64, 128, 2, 2, 4>{});
    case 2: return f(DeepCfg<128, 128, 2, 4, 4>{});
    case 3: return f(DeepCfg<128, 256, 2, 4, 3>{});
    case 4: return f(DeepCfg<256, 128, 4, 2, 3>{});
    case 8: return f(DeepCfg<128, 192, 4, 2, 3>{});
    default: return none;
  }
}
// ... and those that are built for MXFP8 operands (kDeepShapes8)
template <class R, class F>
R with_deep8_shape(int shape, R none, F f) {
  switch (shape) {
    case 0: return f(DeepCfg<64, 64, 2, 2, 4>{});
    case 2: return f(DeepCfg<128, 128, 2, 4, 4>{});
    case 4: return f(DeepCfg<256, 128, 4, 2, 3>{});
    default: return none;
  }
}
// K tiles of row-major scales a workgroup can stage behind the ring: `unit` bytes per row and K tile (8, MXFP8: 4), rows
// padded to an odd count of units (conflict-free reads).
template <class Cfg>
__host__ __device__ constexpr int rows_max_k_tiles(int unit) {
  const int units = (160 * 1024 - Cfg::RING) / ((Cfg::BM + Cfg::BN) * unit), odd = units - 1 + units % 2;
  return odd < 31 ? odd : 31;
}
static_assert(rows_max_k_tiles<DeepCfg<128, 192, 4, 2, 3>>(8) == 15 && rows_max_k_tiles<DeepCfg<128, 256, 2, 4, 3>>(8) == 5 &&
              rows_max_k_tiles<DeepCfg<256, 128, 4, 2, 3>>(8) == 5, "as the head of this file has it");

__host__ __device__ constexpr int rows_pitch(int nkt, int unit) { return (nkt + 1 - (nkt & 1)) * unit; }

// FMT / FMT_B: A's and B's element formats as in the tile kernel (4 = e2m1; 0 = e4m3, 1 = e5m2: a 128-byte K tile is 128
// elements, two 64-wide K steps of 32 bytes per lane, and four scale groups, half of a scale block; a 4-bit operand
// against an 8-bit one fills the lower four chunks of its LDS row).
template <class Cfg, int SC, int FMT, int FMT_B>
__device__ __forceinline__ void deep_body(const GemmParams &p) {
  constexpr bool FP8 = FMT != 4 || FMT_B != 4, A4 = FP8 && FMT == 4, B4 = FP8 && FMT_B == 4;
  constexpr int STEPS = FP8 ? 2 : 4, kUnit = FP8 ? 4 : 8;
  // (64 bits as one scalar: in front of a read of HIP's uint2 from LDS the compiler waits for every outstanding request,
  // and where a branch loads a vector it copies it, and so waits, before the next load; see the staging below)
  typedef typename std::conditional<FP8, uint32_t, uint64_t>::type RowUnit;
  static_assert(!FP8 || SC != kDeepShuffled, "MXFP8 scales: MFMA32 order or row-major");
  constexpr int BM = Cfg::BM, BN = Cfg::BN, MT_M = Cfg::MT_M, MT_N = Cfg::MT_N, S = Cfg::STAGES;
  constexpr int NWAVES = Cfg::NWAVES, A_LD = Cfg::A_LD, B_LD = Cfg::B_LD, S_LD = SC == kDeepRows ? 0 : Cfg::S_LD;
  constexpr int REQ = A_LD + B_LD + S_LD;  // requests of a wave per K tile
  extern __shared__ __attribute__((aligned(1024))) uint8_t smem[];
  uint8_t *const s_ring = smem + Cfg::RING;

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wave_m = wave / Cfg::WAVES_N, wave_n = wave % Cfg::WAVES_N;
  int tm, tn;
  if (!map_tile(blockIdx.x, p.tiles_m, p.tiles_n, tm, tn)) return;
  const int split = blockIdx.y;
  const int m0 = tm * BM, n0 = tn * BN;
  const int kt_begin = split * p.tiles_per_split;
  const int nkt = min(p.k_tiles, kt_begin + p.tiles_per_split) - kt_begin;
  if (nkt <= 0) return;
  const int kp = p.kp, kpa = A4 ? kp >> 1 : kp, kpb = B4 ? kp >> 1 : kp;

  // ---------------- requests ----------------
  // As in the tile kernel: instruction d of a wave fills LDS rows (d * NWAVES + wave) * 8 .. + 7, chunk c of row r at
  // position c ^ (r / 2) % 8.  Every descriptor ends with its tensor, so rows past M or N arrive as zeros, and a K tile
  // past the last one is requested from beyond the descriptor: the same count of requests, no memory access.
  const __amdgpu_buffer_rsrc_t a_rsrc = make_rsrc_n(p.a + (int64_t)m0 * kpa, rsrc_bytes(((int64_t)p.m - m0) * kpa));
  const __amdgpu_buffer_rsrc_t b_rsrc = make_rsrc_n(p.b + (int64_t)n0 * kpb, rsrc_bytes(((int64_t)p.n - n0) * kpb));
  const int ld_row0 = wave * 8 + (lane >> 3);
  const int ld_chunk = (lane & 7) ^ ((ld_row0 >> 1) & 7);
  int a_goff[A_LD], b_goff[B_LD];
#pragma unroll
  for (int d = 0; d < A_LD; ++d)
    a_goff[d] = A4 && ld_chunk >= 4 ? (int)0x80000000 : (ld_row0 + d * NWAVES * 8) * kpa + ld_chunk * 16;
#pragma unroll
  for (int d = 0; d < B_LD; ++d) {
    const int r = ld_row0 + d * NWAVES * 8;
    b_goff[d] = p.b_preshuffled ? (r >> 4) * 16 * kp + (r & 15) * 16 + (ld_chunk >> 1) * 512 + (ld_chunk & 1) * 256
                                : r * kpb + ld_chunk * 16;
    if (B4 && ld_chunk >= 4) b_goff[d] = (int)0x80000000;
  }
  const int a_kt_stride = A4 ? kTileKBytes / 2 : kTileKBytes;
  const int b_kt_stride = p.b_preshuffled ? 2048 : B4 ? kTileKBytes / 2 : kTileKBytes;
  // A partial last K tile (blocked scales only): A's chunks past the end of K are requested from beyond the descriptor
  // and arrive as zeros; whatever B's requests bring in from there is finite, and so are the padding scales.
  const int tail_chunks = SC == kDeepNative && !FP8 ? (p.k & (kTileK - 1)) >> 5 : 0;
  const int tail_lane = tail_chunks != 0 && ld_chunk >= tail_chunks ? (int)0x80000000 : 0;
  // scale blocks: request d of a wave fetches block (d * NWAVES + wave) % SB of the K tile, A's blocks first (a wave
  // beyond the count repeats another's request)
  const int64_t blk_row = (int64_t)(p.ksp >> 3) * 256;  // bytes of the blocks of 32 rows
  const uint8_t *as_base = p.a_scale + (int64_t)(m0 >> 5) * blk_row, *bs_base = p.b_scale + (int64_t)(n0 >> 5) * blk_row;
  const __amdgpu_buffer_rsrc_t as_rsrc = make_rsrc_n(as_base, rsrc_bytes((((int64_t)p.m + 31) / 32 - (m0 >> 5)) * blk_row));
  const __amdgpu_buffer_rsrc_t bs_rsrc = make_rsrc_n(bs_base, rsrc_bytes((((int64_t)p.n + 31) / 32 - (n0 >> 5)) * blk_row));

  // requests [q0, q1) of K tile j (counted from the split's first) into ring slot `slot`
  auto issue = [&](int j, int slot, auto q0_tag, auto q1_tag) {
    constexpr int Q0 = decltype(q0_tag)::value, Q1 = decltype(q1_tag)::value;
    const int kt = kt_begin + j;
    const bool live = j < nkt;
    const int a_soff = live ? kt * a_kt_stride : (int)0x80000000, b_soff = live ? kt * b_kt_stride : (int)0x80000000;
    const int tail = live && kt == p.k_tiles - 1 ? tail_lane : 0;
    uint8_t *a_dst = smem + slot * Cfg::STAGE, *b_dst = a_dst + Cfg::A_BYTES;
#pragma unroll
    for (int q = Q0; q < Q1; ++q) {
      if (q < A_LD) {
        __builtin_amdgcn_raw_ptr_buffer_load_lds(a_rsrc, WAVE_LDS_PTR(a_dst + (q * NWAVES + wave) * 1024), 16,
                                                 a_goff[q] | tail, a_soff, 0, 0);
      } else if (q < A_LD + B_LD) {
        const int d = q - A_LD;
        __builtin_amdgcn_raw_ptr_buffer_load_lds(b_rsrc, WAVE_LDS_PTR(b_dst + (d * NWAVES + wave) * 1024), 16, b_goff[d],
                                                 b_soff, 0, 0);
      } else {
        const int blk = ((q - A_LD - B_LD) * NWAVES + wave) % Cfg::SB;
        const bool is_a = blk < BM / 32;
        const int row = is_a ? blk : blk - BM / 32;
        const int soff = live ? (int)(row * blk_row) + (FP8 ? kt >> 1 : kt) * 256 : (int)0x80000000;
        uint8_t *dst = s_ring + slot * Cfg::S_STAGE + blk * 256;
        if (is_a)
          __builtin_amdgcn_raw_ptr_buffer_load_lds(as_rsrc, WAVE_LDS_PTR(dst), 4, lane * 4, soff, 0, 0);
        else
          __builtin_amdgcn_raw_ptr_buffer_load_lds(bs_rsrc, WAVE_LDS_PTR(dst), 4, lane * 4, soff, 0, 0);
      }
    }
  };
#define WAVE_Q(ph) std::integral_constant<int, REQ * (ph) / STEPS>{}  // first request of phase `ph`

  // ---------------- fragments and scales ----------------
  const int fr = lane & 31, fg = lane >> 5;
  typedef typename std::conditional<FP8 && !A4, v8i, v4i>::type FragA;
  typedef typename std::conditional<FP8 && !B4, v8i, v4i>::type FragB;
  // chunk of K step t: 2t + fg; an 8-bit lane's 32 bytes of step t are the chunks 4t + fg and 4t + 2 + fg
  uint32_t foff[4];
#pragma unroll
  for (int t = 0; t < 4; ++t) foff[t] = (uint32_t)(fr * kTileKBytes + (((t * 2 + fg) ^ ((fr >> 1) & 7)) << 4));
  const int a_fbase = wave_m * Cfg::WM * kTileKBytes, b_fbase = Cfg::A_BYTES + wave_n * Cfg::WN * kTileKBytes;
  auto read_one = [&](const uint8_t *base, int t, auto &frag) {
    if constexpr (sizeof(frag) == 32) {
      const v4i lo = *(const v4i *)(base + foff[2 * t]), hi = *(const v4i *)(base + foff[2 * t + 1]);
      frag = v8i{lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
    } else {
      frag = *(const v4i *)(base + foff[t]);
    }
  };
  auto read_frags = [&](int slot, int t, FragA(&fa)[MT_M], FragB(&fb)[MT_N]) {
    const uint8_t *base = smem + slot * Cfg::STAGE;
#pragma unroll
    for (int i = 0; i < MT_M; ++i) read_one(base + a_fbase + i * 32 * kTileKBytes, t, fa[i]);
#pragma unroll
    for (int j = 0; j < MT_N; ++j) read_one(base + b_fbase + j * 32 * kTileKBytes, t, fb[j]);
  };
  // row-major scales: row r of the staged rows (A's tile rows, then B's) holds kUnit bytes per K tile
  uint8_t *const rows = smem + Cfg::RING;
  const uint32_t pitch = (uint32_t)rows_pitch(nkt, kUnit);
  const uint32_t pick = fg ? 0x07050301u : 0x06040200u;
  auto lane_scale = [&](int slot, int j, int blk) -> uint32_t {
    if constexpr (SC == kDeepRows) {
      const RowUnit v = *(const RowUnit *)(rows + (uint32_t)(blk * 32 + fr) * pitch + j * kUnit);
      if constexpr (FP8) return __builtin_amdgcn_perm(0u, v, fg ? 0x0c0c0301u : 0x0c0c0200u);
      else return __builtin_amdgcn_perm((uint32_t)(v >> 32), (uint32_t)v, pick);
    } else if constexpr (SC == kDeepShuffled) {
      const uint8_t *b = s_ring + slot * Cfg::S_STAGE + blk * 256 + fg * 64 + (fr & 15) * 4;
      return __builtin_amdgcn_perm(*(const uint32_t *)(b + 128), *(const uint32_t *)b,
                                   0x06020400u + (uint32_t)(fr >> 4) * 0x01010101u);
    } else {
      const uint32_t v = *(const uint32_t *)(s_ring + slot * Cfg::S_STAGE + blk * 256 + lane * 4);
      return FP8 ? v >> (((kt_begin + j) & 1) * 16) : v;  // (the block's second K tile: its upper half)
    }
  };
  auto read_scales = [&](int slot, int j, uint32_t(&sa)[MT_M], uint32_t(&sb)[MT_N]) {
#pragma unroll
    for (int i = 0; i < MT_M; ++i) sa[i] = lane_scale(slot, j, wave_m * MT_M + i);
#pragma unroll
    for (int i = 0; i < MT_N; ++i) sb[i] = lane_scale(slot, j, BM / 32 + wave_n * MT_N + i);
  };

  v16f acc[MT_M][MT_N];
#pragma unroll
  for (int i = 0; i < MT_M; ++i)
#pragma unroll
    for (int j = 0; j < MT_N; ++j)
#pragma unroll
      for (int g = 0; g < 16; ++g) acc[i][j][g] = 0.f;
  uint32_t sc_a[MT_M], sc_b[MT_N], nsc_a[MT_M], nsc_b[MT_N];
  auto operand = [](const auto &f) {
    if constexpr (sizeof(f) == 32) return f;
    else return v8i{f.x, f.y, f.z, f.w, 0, 0, 0, 0};
  };
  auto mfma_block = [&](const FragA(&fa)[MT_M], const FragB(&fb)[MT_N], auto t_tag) {
    constexpr int T = decltype(t_tag)::value;
#pragma unroll
    for (int i = 0; i < MT_M; ++i)
#pragma unroll
      for (int j = 0; j < MT_N; ++j) {
        const v8i va = operand(fa[i]), vb = operand(fb[j]);
        acc[i][j] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(vb, va, acc[i][j], FMT_B, FMT, T, (int)sc_b[j], T,
                                                                    (int)sc_a[i]);
      }
  };
  typedef std::integral_constant<int, 0> T0;
  typedef std::integral_constant<int, 1> T1;
  typedef std::integral_constant<int, 2> T2;
  typedef std::integral_constant<int, 3> T3;
  // inside a phase: one MFMA, the next step's fragment reads, then MFMAs and the requests of share PH in turn
  auto order_phase = [&](auto ph_tag) {
    constexpr int PH = decltype(ph_tag)::value;
    constexpr int Q = MT_M * MT_N, NQ = REQ * (PH + 1) / STEPS - REQ * PH / STEPS;
    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
    __builtin_amdgcn_sched_group_barrier(0x100, MT_M * (int)(sizeof(FragA) / 16) + MT_N * (int)(sizeof(FragB) / 16), 0);
#pragma unroll
    for (int g = 0; g < NQ; ++g) {
      if (g + 1 < Q) __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);
    }
    if (Q > NQ + 1) __builtin_amdgcn_sched_group_barrier(0x008, Q - NQ - 1, 0);
  };

  // ---------------- main loop ----------------
  // K tile j is multiplied in four phases (MXFP8: two); its slot is free from the barrier in its last phase on, where the requests
  // of K tile j + S begin (a share there, the others in the first phases of K tile j + 1).  That barrier
  // publishes K tile j + 1: younger than its requests are those of K tiles j + 2 .. j + S - 1.
  FragA fa0[MT_M], fa1[MT_M];
  FragB fb0[MT_N], fb1[MT_N];
  constexpr int kIters = SC == kDeepRows ? ((BM > BN ? BM : BN) * rows_max_k_tiles<Cfg>(kUnit) + Cfg::NT - 1) / Cfg::NT : 1;
  RowUnit row_a[kIters], row_b[kIters];
  // unit `it` of this thread: K tile c of row r (the quotient is exact up to u * (nkt - 1) = 2^18)
  static_assert(kIters * Cfg::NT * 30 < 1 << 18, "units of the staged rows");
  const int per_row = SC == kDeepRows ? ((1 << 18) + nkt - 1) / nkt : 0;
  const int units = (BM > BN ? BM : BN) * nkt;
  auto row_unit = [&](int it, int &r, int &c) {
    const int u = it * Cfg::NT + (int)threadIdx.x;
    r = (u * per_row) >> 18;
    c = u - r * nkt;
  };
  if constexpr (SC == kDeepRows) {
    // All loads are in flight together, and stay so: the first round is not behind a branch and nothing is zeroed in front,
    // or the compiler joins the branches with copies and waits for each load before the next.  With that and without a
    // drain of the ring per K tile (the uint2 above): 1024 x 1024 x 3840, scales row-major, 10.0 -> 8.2 us, 1024 x 3840
    // x 3840 17.1 -> 14.0, 512 x 2048 x 2048 8.3 -> 7.3, 1000 x 7168 x 1280 13.2 -> 12.0.
    // (Rounds that the range does not need are left out whole: 1024 x 1024 x 1024 5.0 -> 4.75, 512 x 2048 x 2048 7.8 -> 7.15.)
#pragma unroll
    for (int it = 0; it < kIters; ++it) {
      if (it > 0 && it * Cfg::NT >= units) continue;
      int r, c;
      row_unit(it, r, c);
      if (it == 0 || r < BM)
        row_a[it] = *(const RowUnit *)(p.a_scale + (int64_t)min(m0 + min(r, BM - 1), p.m - 1) * p.ks + (kt_begin + c) * kUnit);
      if (it == 0 || r < BN)
        row_b[it] = *(const RowUnit *)(p.b_scale + (int64_t)min(n0 + min(r, BN - 1), p.n - 1) * p.ks + (kt_begin + c) * kUnit);
    }
  }
#pragma unroll
  for (int j = 0; j < S - 1; ++j) issue(j, j, WAVE_Q(0), WAVE_Q(STEPS));
  issue(S - 1, S - 1, WAVE_Q(0), WAVE_Q(1));
  if constexpr (SC == kDeepRows) {
#pragma unroll
    for (int it = 0; it < kIters; ++it) {
      if (it > 0 && it * Cfg::NT >= units) continue;
      int r, c;
      row_unit(it, r, c);
      if (r < BM) *(RowUnit *)(rows + (uint32_t)r * pitch + c * kUnit) = row_a[it];
      if (r < BN) *(RowUnit *)(rows + (uint32_t)(BM + r) * pitch + c * kUnit) = row_b[it];
    }
  }
  __builtin_amdgcn_s_waitcnt(waitcnt_vm_lgkm0((S - 2) * REQ + REQ / STEPS));
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  read_frags(0, 0, fa0, fb0);
  read_scales(0, 0, sc_a, sc_b);
  __builtin_amdgcn_sched_barrier(0);

  int slot = 0, slot_prev = S - 1;
  auto k_tile = [&](int j, auto next_tag) {
    constexpr bool NEXT = decltype(next_tag)::value;
    const int slot_next = slot + 1 == S ? 0 : slot + 1;
    const int jr = j + S - 1;
    read_frags(slot, 1, fa1, fb1);
    mfma_block(fa0, fb0, T0{});
    if (NEXT) issue(jr, slot_prev, WAVE_Q(1), WAVE_Q(2));
    order_phase(T1{});
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (!FP8) {
      read_frags(slot, 2, fa0, fb0);
      mfma_block(fa1, fb1, T1{});
      if (NEXT) issue(jr, slot_prev, WAVE_Q(2), WAVE_Q(3));
      order_phase(T2{});
      __builtin_amdgcn_sched_barrier(0);
      read_frags(slot, 3, fa1, fb1);
      mfma_block(fa0, fb0, T2{});
      if (NEXT) issue(jr, slot_prev, WAVE_Q(3), WAVE_Q(4));
      order_phase(T3{});
      __builtin_amdgcn_sched_barrier(0);
    }
    if (NEXT) {
      __builtin_amdgcn_s_waitcnt(waitcnt_vm_lgkm0((S - 2) * REQ));
      asm volatile("" ::: "memory");
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
      __builtin_amdgcn_sched_barrier(0);
      read_frags(slot_next, 0, fa0, fb0);
      read_scales(slot_next, j + 1, nsc_a, nsc_b);
    }
    mfma_block(fa1, fb1, std::integral_constant<int, STEPS - 1>{});
    if (NEXT) issue(j + S, slot, WAVE_Q(0), WAVE_Q(1));
    order_phase(T0{});
    __builtin_amdgcn_sched_barrier(0);
    if (NEXT) {
#pragma unroll
      for (int i = 0; i < MT_M; ++i) sc_a[i] = nsc_a[i];
#pragma unroll
      for (int i = 0; i < MT_N; ++i) sc_b[i] = nsc_b[i];
      slot_prev = slot;
      slot = slot_next;
    }
  };
  for (int j = 0; j < nkt - 1; ++j) k_tile(j, std::true_type{});
  k_tile(nkt - 1, std::false_type{});
#undef WAVE_Q

  // ---------------- C ----------------
  // acc[i][jn][4q + e]: row fr, column 8q + 4 fg + e of the 32x32 tile: every wave transposes its sub-tile through its
  // share of LDS and stores whole 16-byte pieces of rows (N is a multiple of 4, for bf16 of 8).
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt(waitcnt_vm_lgkm0(0));
  __builtin_amdgcn_s_barrier();  // every wave is done with the ring, and no request is on its way into it
  asm volatile("" ::: "memory");
  const bool to_partial = p.partial != nullptr;
  const int64_t ldc = p.n;
  const int wm0 = m0 + wave_m * Cfg::WM, wn0 = n0 + wave_n * Cfg::WN;
  if (!to_partial && p.out_bf16) {
    constexpr int ROWB = Cfg::WN * 2 + 8, LPR = Cfg::WN * 2 / 16;
    typedef __bf16 bf4 __attribute__((ext_vector_type(4)));
    uint8_t *stage = smem + wave * (Cfg::WM * (Cfg::WN * 4 + 16));
#pragma unroll
    for (int i = 0; i < MT_M; ++i)
#pragma unroll
      for (int jn = 0; jn < MT_N; ++jn)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const bf4 h = {(__bf16)acc[i][jn][4 * q], (__bf16)acc[i][jn][4 * q + 1], (__bf16)acc[i][jn][4 * q + 2],
                         (__bf16)acc[i][jn][4 * q + 3]};
          *(bf4 *)(stage + (i * 32 + fr) * ROWB + (jn * 32 + q * 8 + fg * 4) * 2) = h;
        }
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(waitcnt_vm_lgkm0(63));
#pragma unroll
    for (int u0 = 0; u0 < Cfg::WM * LPR; u0 += 64) {  // (64 pieces of 16 bytes at a time, WM being whole 32 rows)
      const int r = (u0 + lane) / LPR, lc = u0 + lane - r * LPR, m = wm0 + r, n = wn0 + lc * 8;
      const v4i v = *(const v4i *)(stage + r * ROWB + lc * 16);
      if (m < p.m && n < p.n) *(v4i *)((__bf16 *)p.c + (int64_t)m * ldc + n) = v;
    }
  } else {
    constexpr int ROWB = Cfg::WN * 4 + 16, LPR = Cfg::WN * 4 / 16;
    uint8_t *stage = smem + wave * (Cfg::WM * ROWB);
#pragma unroll
    for (int i = 0; i < MT_M; ++i)
#pragma unroll
      for (int jn = 0; jn < MT_N; ++jn)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const v4f v = {acc[i][jn][4 * q], acc[i][jn][4 * q + 1], acc[i][jn][4 * q + 2], acc[i][jn][4 * q + 3]};
          *(v4f *)(stage + (i * 32 + fr) * ROWB + (jn * 32 + q * 8 + fg * 4) * 4) = v;
        }
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(waitcnt_vm_lgkm0(63));
    float *cbase = to_partial ? p.partial + (int64_t)split * p.m * ldc : (float *)p.c;
#pragma unroll
    for (int u0 = 0; u0 < Cfg::WM * LPR; u0 += 64) {
      const int r = (u0 + lane) / LPR, lc = u0 + lane - r * LPR, m = wm0 + r, n = wn0 + lc * 4;
      const v4f v = *(const v4f *)(stage + r * ROWB + lc * 16);
      if (m < p.m && n < p.n) *(v4f *)(cbase + (int64_t)m * ldc + n) = v;
    }
  }
}

template <class Cfg, int SC, int FMT, int FMT_B>
__global__ void __launch_bounds__(Cfg::NT, 1) deep_gemm_kernel(const GemmParams p) {
  deep_body<Cfg, SC, FMT, FMT_B>(p);
}

template <class Cfg, int SC, int FMT = 4, int FMT_B = FMT>
hipError_t launch_deep_cfg(GemmParams p, hipStream_t stream) {
  constexpr int kUnit = FMT == 4 && FMT_B == 4 ? 8 : 4;
  constexpr int kStaging = Cfg::NWAVES * Cfg::WM * (Cfg::WN * 4 + 16);
  constexpr int kScales = SC == kDeepRows ? (Cfg::BM + Cfg::BN) * rows_pitch(rows_max_k_tiles<Cfg>(kUnit), kUnit) : Cfg::S_RING;
  constexpr int kMax = Cfg::RING + kScales > kStaging ? Cfg::RING + kScales : kStaging;
  if constexpr (kMax > 160 * 1024) {
    return hipErrorInvalidValue;
  } else {
    static LdsAttrOnce once;
    const hipError_t e = allow_dynamic_lds(once, (const void *)deep_gemm_kernel<Cfg, SC, FMT, FMT_B>, kMax);
    if (e != hipSuccess) return e;
    p.tiles_m = (p.m + Cfg::BM - 1) / Cfg::BM;
    p.tiles_n = (p.n + Cfg::BN - 1) / Cfg::BN;
    const int per_xcd = (p.tiles_m * p.tiles_n + kNumXcd - 1) / kNumXcd;
    deep_gemm_kernel<Cfg, SC, FMT, FMT_B><<<dim3(per_xcd * kNumXcd, p.splits, 1), dim3(Cfg::NT), kMax, stream>>>(p);
    return hipGetLastError();
  }
}

}  // namespace
}  // namespace wave_mxfp4
#endif  // WAVE_MXFP4_GEMM_DEEP_H_
