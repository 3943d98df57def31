// Mid-sized block-FP8 GEMM for gfx950: the LDS-tiled FP8-MFMA GEMM on tiles of
// 64 or 128 weight rows x 32 .. 128 tokens, for shapes whose 256 x 256 tiles
// (gk_fp8_prefill.hip) would leave most of the 256 CUs idle.
//
// Same arithmetic and order as the 256 x 256 kernel: per 128-K group one
// v_mfma_f32_16x16x128_f8f6f4 per 16 x 16 block, multiplied by sa[m, g] *
// sw[n / 128, g] and added in fp32, groups in ascending order -- so the result
// bits do not depend on which of the two kernels runs, nor on the tile.
//
// Measured on MI355X (us of the GEMM launch, launches back to back; 256 x 256
// tiles -> here): M = 300, N = 6144, K = 4096 45.3 -> 15.6; M = 128, same weights
// 44.3 -> 11.1; M = 256, N = K = 4096 45.0 -> 11.3; M = 1024, N = K = 4096 47.1 ->
// 25.2.  Bound: the LDS port (128 bytes a cycle).  A 128 x 64 group reads 64 KB of
// fragments and writes 24 KB of copies, 700 of the 1000 cycles that it takes; its
// MFMAs take 256.  Four waves of larger wave tiles read less but lose more latency
// (18.2 -> 21.6 us).
//
// Structure (one workgroup = 8 waves, 4 along N x 2 along M; a wave holds
// 16 NA weight rows x 16 MB tokens):
//   * Stage = U 128-K groups (two a barrier where one workgroup has the CU: 13.9
//     -> 13.0 us at M = 128, N = 6144, K = 4096): BN x 128 weight bytes and BM x
//     128 activation bytes of each, and the token scales, copied global -> LDS by
//     buffer loads with the LDS bit.  NS stages in a ring, filled NS - 1 steps
//     ahead: a step is short, so the copies of several steps have to be in flight
//     to cover the memory latency.
//   * A wave issues the same number of copies in every step (wave 0 also the
//     token scales; pieces past the last are copied twice, steps past the last
//     re-read the last group into a stage that is no longer read), so the step's
//     own copies are done when at most NS - 2 steps' are outstanding.  One bare
//     barrier a step.
//   * LDS chunk order and inline-asm fragment reads as in the 256 x 256 kernel.

#include <mutex>
#include <utility>

#include "gk_fp8_lds.h"

namespace gk {

namespace {

// s_waitcnt vmcnt(n) alone (expcnt and lgkmcnt at their maxima).
constexpr int vmcnt_imm(int n) { return 0x0F70 | (n & 15) | ((n >> 4) << 14); }

template <int OFF>
__device__ inline float lds_read_f32(uint32_t base) {
  float r;
  asm volatile("ds_read_b32 %0, %1 offset:%2" : "=v"(r) : "v"(base), "n"(OFF));
  return r;
}

// The reads of one group's fragments and scales have arrived (LATER reads issued after them may be in flight);
// the wait is tied to the registers read into.
template <int NA, int MB, bool CH, int LATER>
__device__ inline void tile_wait(v8i (&a)[NA], v8i (&b)[MB], float (&s)[MB]) {
  asm volatile("s_waitcnt lgkmcnt(%2)" : "+v"(a[0]), "+v"(b[0]) : "n"(LATER));
#pragma unroll
  for (int i = 1; i < NA; ++i) asm volatile("" : "+v"(a[i]));
#pragma unroll
  for (int j = 1; j < MB; ++j) asm volatile("" : "+v"(b[j]));
  if (!CH) {
#pragma unroll
    for (int j = 0; j < MB; ++j) asm volatile("" : "+v"(s[j]));
  }
}

// A tile: WN x WM waves (along N x along M) of 16 NA weight rows x 16 MB tokens; U groups per step, NS stages.
template <int WN_, int WM_, int NA_, int MB_, int U_, int NS_>
struct Tile {
  static constexpr int WN = WN_, WM = WM_, NA = NA_, MB = MB_, U = U_, NS = NS_;
  static constexpr int kWaves = WN * WM, BN = 16 * NA * WN, BM = 16 * MB * WM;
  // LDS of one stage: U groups of both operand tiles, and their token scales (one 1 KB piece)
  static constexpr int kStage = U * (BN + BM) * 128 + 1024;
  static_assert(NS * kStage <= 160 * 1024, "the stages fit the LDS");
};

template <typename T, bool HALF, bool CH, bool WPACK>
__device__ __forceinline__ void gemm_tile_body(
    const uint8_t* __restrict__ qa, const float* __restrict__ sa, const uint8_t* __restrict__ w,
    const float* __restrict__ sw, const float* __restrict__ bias, uint16_t* __restrict__ y, int64_t ldy, int M, int N,
    int K, int G, int Mpad, int64_t ldq, int gs, float* __restrict__ yp, int64_t ldyp, int accum) {
  constexpr int NA = T::NA, MB = T::MB, U = T::U, NS = T::NS, BN = T::BN, BM = T::BM;
  constexpr int kStage = T::kStage, kWBytes = BN * 128, kGBytes = (BN + BM) * 128;
  constexpr int kWP = BN / 8, kAP = BM / 8;  // 1 KB pieces (8 rows) of the two tiles of one group
  constexpr int kWL = kWP / T::kWaves, kAL = (kAP + T::kWaves - 1) / T::kWaves;
  constexpr int kLoads = U * (kWL + kAL);  // copies per wave and step (wave 0: and the token scales)
  static_assert(kWP % T::kWaves == 0 && 128 % BN == 0, "a workgroup's rows lie in one 128-row scale block");
  static_assert(U * BM <= 256, "a step's token scales are one 1 KB piece");
  static_assert((NS - 2) * (kLoads + 1) < 64, "the step's wait fits vmcnt");
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wn = wave % T::WN, wm = wave / T::WN;
  // Tile order: workgroup b runs on XCD b % 8; each XCD takes a contiguous
  // eighth of the tiles, row tiles of one weight panel first, so a panel is
  // fetched into one XCD's L2 once.
  const int tiles_m = (M + BM - 1) / BM, tiles = static_cast<int>(gridDim.x);
  const int b = static_cast<int>(blockIdx.x), xcd = b & 7, tq = tiles >> 3, tr = tiles & 7;
  const int l = xcd * tq + min(xcd, tr) + (b >> 3);
  const int n0 = (l / tiles_m) * BN, m0 = (l % tiles_m) * BM;

  // Copies.  Lane -> row lane / 8 of the piece, slot lane % 8, which holds chunk slot ^ key(row).
  const int lr = lane >> 3, ls = lane & 7;
  const uint32_t lane16 = static_cast<uint32_t>(lane) * 16u;
  const uint8_t* wbase = w + static_cast<int64_t>(n0) * (WPACK ? static_cast<int64_t>(gs) * 128 : K);
  const uint8_t* abase = CH ? qa + static_cast<int64_t>(m0) * ldq : qa + static_cast<int64_t>(m0) * 128;
  const __amdgpu_buffer_rsrc_t wrsrc =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(wbase), 0, -1, kBufferWord3);
  const __amdgpu_buffer_rsrc_t arsrc =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(abase), 0, -1, kBufferWord3);
  const __amdgpu_buffer_rsrc_t srsrc =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(CH ? sw : sa), 0, -1, kBufferWord3);
  int apc[kAL];                   // this wave's activation pieces
  uint32_t woff[kWL], aoff[kAL];  // per-lane byte offsets (rows past the last re-read it)
#pragma unroll
  for (int i = 0; i < kWL; ++i) {
    const int p = wave * kWL + i, r = 8 * p + lr;
    // packed: piece p is half p % 2 of 16-row block p / 2
    woff[i] = WPACK ? static_cast<uint32_t>(min(p >> 1, ((N + 15) >> 4) - 1 - (n0 >> 4))) * static_cast<uint32_t>(gs) * 2048u +
                          static_cast<uint32_t>(p & 1) * 1024u + lane16
                    : static_cast<uint32_t>(min(r, N - 1 - n0)) * static_cast<uint32_t>(K) +
                          static_cast<uint32_t>((ls ^ lds_key(r)) << 4);
  }
#pragma unroll
  for (int i = 0; i < kAL; ++i) {
    apc[i] = min(wave * kAL + i, kAP - 1);
    const int r = 8 * apc[i] + lr;
    aoff[i] = static_cast<uint32_t>(min(r, M - 1 - m0)) * static_cast<uint32_t>(CH ? ldq : 128) +
              static_cast<uint32_t>((ls ^ lds_key(r)) << 4);
  }
  // Token scales: lane -> four tokens of group lane / (BM / 4); the lanes past the last group re-read it.
  const int su = min(lane / (BM / 4), U - 1);
  const uint32_t stok = static_cast<uint32_t>(m0 + 4 * (lane % (BM / 4))) * 4u;
  auto issue = [&](int g0, int st) {  // groups g0 .. g0 + U - 1 (past the last: it again) into stage st
    uint8_t* base = smem + st * kStage;
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const uint32_t g = static_cast<uint32_t>(min(g0 + u, G - 1));
#pragma unroll
      for (int i = 0; i < kWL; ++i)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(wrsrc, lds_ptr(base + u * kGBytes + (wave * kWL + i) * 1024), 16,
                                                 woff[i], g * (WPACK ? 2048u : 128u), 0, 0);
#pragma unroll
      for (int i = 0; i < kAL; ++i)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(arsrc, lds_ptr(base + u * kGBytes + kWBytes + apc[i] * 1024), 16,
                                                 aoff[i], g * (CH ? 128u : static_cast<uint32_t>(Mpad) * 128u), 0, 0);
    }
    if (!CH && wave == 0)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(
          srsrc, lds_ptr(base + U * kGBytes), 16,
          static_cast<uint32_t>(min(g0 + su, G - 1)) * static_cast<uint32_t>(Mpad) * 4u + stok, 0, 0, 0);
  };

  // Fragment addresses within a stage (operand layout: lane -> row lane % 16, K bytes [32 (lane / 16), +32)).
  const int fr = lane & 15, fq = lane >> 4, kf = lds_key(fr);
  const uint32_t xo0 = static_cast<uint32_t>(((2 * fq) ^ kf) << 4), xo1 = static_cast<uint32_t>(((2 * fq + 1) ^ kf) << 4);
  const uint32_t lbase = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(smem));
  const uint32_t arow = WPACK ? static_cast<uint32_t>(wn * NA) * 2048u + lane16
                              : static_cast<uint32_t>(wn * 16 * NA + fr) * 128u;
  const uint32_t wo0 = lbase + arow + (WPACK ? 0u : xo0), wo1 = lbase + arow + (WPACK ? 1024u : xo1);
  const uint32_t bo = lbase + kWBytes + static_cast<uint32_t>(wm * 16 * MB + fr) * 128u;
  const uint32_t so = lbase + U * kGBytes + static_cast<uint32_t>(wm * 16 * MB + fr) * 4u;
  const float* swp = sw + static_cast<int64_t>(n0 >> 7) * gs;

  v4f acc[NA][MB];
#pragma unroll
  for (int i = 0; i < NA; ++i)
#pragma unroll
    for (int j = 0; j < MB; ++j) acc[i][j] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
  const int nb = n0 + wn * 16 * NA + 4 * fq, mb = m0 + wm * 16 * MB + fr;  // output (mb + 16 j, nb + 16 i + r)
  if (accum) {
#pragma unroll
    for (int j = 0; j < MB; ++j)
#pragma unroll
      for (int i = 0; i < NA; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (mb + 16 * j < M && nb + 16 * i + r < N)
            acc[i][j][r] = yp[static_cast<int64_t>(mb + 16 * j) * ldyp + nb + 16 * i + r];
  }
  // Weight scales of 64 groups, one per lane: a step takes its groups' by
  // readlane.  (A scalar load per step puts its latency into the step, and its
  // wait drains the fragment reads in flight: both count in lgkmcnt.)
  float swv = CH ? 0.0f : swp[min(lane, G - 1)];
  asm volatile("" : "+v"(swv));
  __builtin_amdgcn_s_waitcnt(vmcnt_imm(0));  // from here on only the copies are counted

#pragma unroll
  for (int s = 0; s < NS - 1; ++s) issue(min(U * s, G - 1), s);
  int st = 0;
  // One step of kGroups groups from g on (a template: the last step of an odd
  // G takes one group, in code of its own, so no branch lies between a
  // fragment read and its wait, where register copies would read too early).
  auto step = [&](auto nc, int g) {
    constexpr int kGroups = decltype(nc)::value, kBlocks = kGroups * NA * MB, kAhead = 3;
    constexpr int kReads = 2 * (NA + MB) + (CH ? 0 : MB);  // LDS reads of one group
    // this wave's copies of the step are done (those of the NS - 2 steps after it may be in flight) ...
    if (!CH && wave == 0)
      __builtin_amdgcn_s_waitcnt(vmcnt_imm((NS - 2) * (kLoads + 1)));
    else
      __builtin_amdgcn_s_waitcnt(vmcnt_imm((NS - 2) * kLoads));
    __builtin_amdgcn_s_barrier();  // ... and every wave's; every wave has read its fragments of the step before
    const uint32_t sb = static_cast<uint32_t>(st) * kStage;
    const uint32_t A0 = wo0 + sb, A1 = wo1 + sb, B0 = bo + xo0 + sb, B1 = bo + xo1 + sb, S = so + sb;
    v8i fa[kGroups][NA], fb[kGroups][MB];
    float sv[kGroups][MB];
    unroll_each([&](auto uc) {
      constexpr int u = decltype(uc)::value;
      if (!CH) {
        unroll_each([&](auto jc) {
          constexpr int j = decltype(jc)::value;
          sv[u][j] = lds_read_f32<u * BM * 4 + 64 * j>(S);
        }, std::make_integer_sequence<int, MB>{});
      }
      unroll_each([&](auto ic) {
        constexpr int i = decltype(ic)::value;
        fa[u][i] = lds_frag_at<u * kGBytes + i * 2048>(A0, A1);
      }, std::make_integer_sequence<int, NA>{});
      unroll_each([&](auto jc) {
        constexpr int j = decltype(jc)::value;
        fb[u][j] = lds_frag_at<u * kGBytes + j * 2048>(B0, B1);
      }, std::make_integer_sequence<int, MB>{});
    }, std::make_integer_sequence<int, kGroups>{});
    issue(min(g + U * (NS - 1), G - 1), st == 0 ? NS - 1 : st - 1);
    st = st == NS - 1 ? 0 : st + 1;
    __builtin_amdgcn_sched_barrier(0);
    // Blocks in order (group, token block, weight block); the MFMA of a block is issued kAhead blocks before its
    // promotion, so a wave does not wait for the MFMA it has just issued.
    v4f t[kAhead + 1];
    float f[kGroups][MB];
    unroll_each([&](auto kc) {
      constexpr int k = decltype(kc)::value;
      if constexpr (k < kBlocks) {
        constexpr int u = k / (NA * MB), j = k / NA % MB, i = k % NA;
        if constexpr (k % (NA * MB) == 0) {
          constexpr int kLater = (kGroups - 1 - u) * kReads;
          tile_wait<NA, MB, CH, (kLater < 15 ? kLater : 15)>(fa[u], fb[u], sv[u]);
          if (HALF) {
#pragma unroll
            for (int h = 0; h < NA; ++h) fa[u][h] = half_codes(fa[u][h]);
          }
          if (!CH) {
            // native_half doubles the weight scales (block_fp8_oracle.py:35); x2 is exact
            const float ws = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(swv), (g + u) & 63));
#pragma unroll
            for (int h = 0; h < MB; ++h) f[u][h] = sv[u][h] * (HALF ? 2.0f * ws : ws);
          }
        }
        if (CH) acc[i][j] = mfma_f8_acc(fa[u][i], fb[u][j], acc[i][j]);
        else t[k % (kAhead + 1)] = mfma_f8(fa[u][i], fb[u][j]);
      }
      if constexpr (!CH && k >= kAhead) {
        constexpr int q = k - kAhead, u = q / (NA * MB), j = q / NA % MB, i = q % NA;
        promote4(acc[i][j], t[q % (kAhead + 1)], f[u][j]);
      }
      __builtin_amdgcn_sched_barrier(0);
    }, std::make_integer_sequence<int, kBlocks + (CH ? 0 : kAhead)>{});
  };
  auto next_scales = [&](int g) {
    if (!CH && g > 0 && (g & 63) == 0) {
      swv = swp[min(g + lane, G - 1)];
      asm volatile("" : "+v"(swv));
      __builtin_amdgcn_s_waitcnt(vmcnt_imm(0));
    }
  };
  int g = 0;
  for (; g + U <= G; g += U) {
    next_scales(g);
    step(std::integral_constant<int, U>{}, g);
  }
  if (U > 1 && g < G) {
    next_scales(g);
    step(std::integral_constant<int, 1>{}, g);
  }
  __builtin_amdgcn_s_waitcnt(0);  // the re-read copies still in flight write LDS

#pragma unroll
  for (int j = 0; j < MB; ++j) {
    const int m = mb + 16 * j;
    if (m >= M) continue;
    const float sam = CH ? sa[m] : 0.0f;
#pragma unroll
    for (int i = 0; i < NA; ++i) {
      const int n = nb + 16 * i;
      if (CH) {
        store_channel_tile(y, ldy, sw, bias, N, m, n, sam, acc[i][j]);
      } else if (yp) {
        float* dst = yp + static_cast<int64_t>(m) * ldyp + n;
        if (n + 3 < N && (reinterpret_cast<uintptr_t>(dst) & 15) == 0) {
          *reinterpret_cast<v4f*>(dst) = acc[i][j];
        } else {
#pragma unroll
          for (int r = 0; r < 4; ++r)
            if (n + r < N) dst[r] = acc[i][j][r];
        }
      } else {
        store_tile(y, ldy, bias, M, N, m, n, acc[i][j]);
      }
    }
  }
}

template <typename T, bool HALF, bool CH, bool WPACK>
__global__ __launch_bounds__(64 * T::kWaves) void gemm_tile_kernel(
    const uint8_t* __restrict__ qa, const float* __restrict__ sa, const uint8_t* __restrict__ w,
    const float* __restrict__ sw, const float* __restrict__ bias, uint16_t* __restrict__ y, int64_t ldy, int M, int N,
    int K, int G, int Mpad, int64_t ldq, int gs, float* __restrict__ yp, int64_t ldyp, int accum) {
  gemm_tile_body<T, HALF, CH, WPACK>(qa, sa, w, sw, bias, y, ldy, M, N, K, G, Mpad, ldq, gs, yp, ldyp, accum);
}

// The dynamic LDS of a tile is above the default limit: raised once per device and kernel.
constexpr int kMaxDevices = 64;

template <typename T, bool HALF, bool CH, bool WPACK>
hipError_t tile_lds_limit() {
  static std::once_flag once[kMaxDevices];
  static hipError_t err[kMaxDevices];
  int dev = 0;
  const hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  if (dev < 0 || dev >= kMaxDevices) return hipErrorInvalidDevice;
  std::call_once(once[dev], [dev] {
    err[dev] = hipFuncSetAttribute(reinterpret_cast<const void*>(&gemm_tile_kernel<T, HALF, CH, WPACK>),
                                   hipFuncAttributeMaxDynamicSharedMemorySize, T::NS * T::kStage);
  });
  return err[dev];
}

template <typename T, bool HALF, bool CH, bool WPACK>
hipError_t tile_launch(const GemmArgs& a, hipStream_t stream) {
  const hipError_t e = tile_lds_limit<T, HALF, CH, WPACK>();
  if (e != hipSuccess) return e;
  const unsigned tiles = static_cast<unsigned>((a.M + T::BM - 1) / T::BM) *
                         static_cast<unsigned>((a.N + T::BN - 1) / T::BN);
  gemm_tile_kernel<T, HALF, CH, WPACK><<<tiles, 64 * T::kWaves, T::NS * T::kStage, stream>>>(
      a.qa, a.sa, a.w, a.sw, a.bias, a.y, a.ldy, a.M, a.N, a.K, a.G, a.Mpad, a.ldq, a.gstride(), a.yp, a.ldyp,
      a.accumulate ? 1 : 0);
  return hipGetLastError();
}

template <typename T>
hipError_t tile_dispatch(const GemmArgs& a, hipStream_t stream) {
  if (a.channel) return tile_launch<T, false, true, false>(a, stream);
  if (a.wpack) return a.half_w ? tile_launch<T, true, false, true>(a, stream) : tile_launch<T, false, false, true>(a, stream);
  return a.half_w ? tile_launch<T, true, false, false>(a, stream) : tile_launch<T, false, false, false>(a, stream);
}

}  // namespace

hipError_t launch_gemm_tiles(const GemmArgs& a, TileId tile, hipStream_t stream) {
  switch (tile) {
    case kTile64x32: return tile_dispatch<Tile<4, 2, 1, 1, 2, 5>>(a, stream);
    case kTile64x64: return tile_dispatch<Tile<4, 2, 1, 2, 2, 4>>(a, stream);
    case kTile128x64: return tile_dispatch<Tile<4, 2, 2, 2, 2, 3>>(a, stream);
    case kTile128x64Two: return tile_dispatch<Tile<4, 2, 2, 2, 1, 3>>(a, stream);
    case kTile128x128: return tile_dispatch<Tile<4, 2, 2, 4, 1, 4>>(a, stream);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace gk
