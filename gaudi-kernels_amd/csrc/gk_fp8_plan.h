// Decode-variant shape planning: plain C++ (no HIP), shared by the kernels'
// dispatch (gk_fp8_gemm.hip), the C-ABI layer (gk_fp8_abi.hip) and a host test
// that checks every planned shape against the instantiated list.
#pragma once

namespace gk {

// Decode variant shape: NW waves per workgroup (splitting K), R 16-row weight
// tiles per workgroup, U groups per load step, MT 16-token column tiles.
struct DecodeShape {
  int nw, r, u, mt;
};

// Instantiated decode shapes (NW, R, U, MT).  GK_DECODE_SHAPES1: the
// per-channel decode (plan_decode_shape at MT = 1, no step fitting);
// GK_DECODE_SHAPES_T1: every MT = 1 shape (fit_group_step and
// fused_quant_shape halve U); GK_DECODE_SHAPES4: the shapes planned at MT = 4,
// which also run three tiles (launched_shape); GK_DECODE_SHAPES: all.
#define GK_DECODE_SHAPES1(X) X(2, 2, 4, 1) X(8, 2, 2, 1) X(8, 2, 4, 1) X(8, 1, 2, 1) X(16, 1, 2, 1)
#define GK_DECODE_SHAPES_T1(X) GK_DECODE_SHAPES1(X) \
  X(2, 2, 2, 1) X(2, 2, 1, 1) X(8, 2, 1, 1) X(8, 1, 1, 1) X(16, 1, 1, 1)
#define GK_DECODE_SHAPES4(X, MT) X(2, 2, 1, MT) X(8, 2, 1, MT) X(8, 1, 1, MT) X(16, 1, 1, MT)
#define GK_DECODE_SHAPES(X) GK_DECODE_SHAPES_T1(X)                                             \
  X(2, 2, 2, 2) X(2, 2, 1, 2) X(8, 2, 1, 2) X(8, 2, 2, 2) X(8, 1, 1, 2) X(16, 1, 1, 2)         \
  GK_DECODE_SHAPES4(X, 3) GK_DECODE_SHAPES4(X, 4)

constexpr int decode_key(int nw, int r, int u, int mt) { return ((nw * 10 + r) * 10 + u) * 10 + mt; }

// Membership in the three lists above (list 1, T1 or all).
inline bool decode_shape_listed(const DecodeShape& d, int list) {
  const int key = decode_key(d.nw, d.r, d.u, d.mt);
  int n = 0;
  int keys[32];
#define GK_KEY(NW, R, U, MT) keys[n++] = decode_key(NW, R, U, MT);
  if (list == 1) {
    GK_DECODE_SHAPES1(GK_KEY)
  } else if (list == 2) {
    GK_DECODE_SHAPES_T1(GK_KEY)
  } else {
    GK_DECODE_SHAPES(GK_KEY)
  }
#undef GK_KEY
  for (int i = 0; i < n; ++i)
    if (keys[i] == key) return true;
  return false;
}

inline DecodeShape plan_decode_shape(int N, int G, bool packed_weights, int mt) {
  // R: 16-row tiles per workgroup.  Every workgroup reads the activations of
  // its K range once, so larger R cuts activation traffic, but the workgroup
  // count (tiles / R) must stay near or above the 256 CUs.  NW: waves
  // splitting K (the partials are summed in wave order, so NW fixes the
  // result bits; both weight layouts use the same NW for every N and give
  // identical results).  U: groups per load step, divided by the token tiles
  // mt (each group's activation fragments grow with mt).  Measured on MI355X
  // at M = 16 for N x K = 28672 x 4096, 6144 x 4096, 4096 x 14336; the packed
  // layout (no LDS transpose) gains from the deeper step at N = 6144.
  (void)G;
  const int tiles = (N + 15) / 16;
  DecodeShape d;
  if (tiles >= 1536) d = DecodeShape{2, 2, 4, 1};
  else if (tiles >= 384) d = packed_weights ? DecodeShape{8, 2, 4, 1} : DecodeShape{8, 2, 2, 1};
  else if (tiles >= 256) d = DecodeShape{8, 1, 2, 1};
  else d = DecodeShape{16, 1, 2, 1};
  d.mt = mt;
  d.u = d.u / mt > 0 ? d.u / mt : 1;
  return d;
}

inline DecodeShape fit_group_step(DecodeShape d, int G) {
  // A wave's last load step is padded with repeats of its last group (loaded
  // again, multiplied, and scaled by zero), so U is halved until it divides
  // every wave's group count (G/NW rounded either way).  Measured on MI355X:
  // 7168 x 7168 (7 groups a wave) 10.9 -> 10.0 us at M = 16 with U = 1,
  // 8192 x 2048 (2 a wave) 6.5 -> 5.0 us with U = 2.  NW, and so the result
  // bits, is unchanged.
  const int lo = G / d.nw, hi = (G + d.nw - 1) / d.nw;
  while (d.u > 1 && (lo == 0 || lo % d.u != 0 || hi % d.u != 0)) d.u /= 2;
  return d;
}

inline DecodeShape launched_shape(DecodeShape d, int M) {
  // 33 .. 48 tokens leave the fourth tile of the 64-row layout empty: three tiles read and multiply a quarter less
  // (every workgroup reads all tiles; the activations' L2 reads and the weights' HBM reads add up in a CU).  The same
  // bits.  M = 40, N = 4096, K = 14336: 21.4 -> 18.3 us (kernel trace).
  if (d.mt == 4 && M <= 48) d.mt = 3;
  return d;
}

inline DecodeShape fused_quant_shape(DecodeShape d, int G) {
  // With the quantizer fused, a load step also quantizes its U groups, and a
  // padded step repeats that work for nothing.  U divides every wave's group
  // count: 4 only where each wave has exactly 4 groups, else 2 where both
  // counts are even, else 1.  More, shorter steps also keep the quantizer's
  // arithmetic beside the weight fetch.  Measured on MI355X at M = 1, 8, 16
  // for nine N x K shapes; NW (and so the result bits) is unchanged.
  const int lo = G / d.nw, hi = (G + d.nw - 1) / d.nw;
  d.u = (lo == 4 && hi == 4 && d.u == 4) ? 4 : (lo % 2 == 0 && hi % 2 == 0 && lo > 0) ? 2 : 1;
  return d;
}

// Dense 256 x 256 GEMM tile order (gk_fp8_prefill.hip).  Workgroup bid of a
// launch (or column range) of tiles_m x tiles_nn tiles and kparts K parts runs
// on XCD bid % 8 of the GPU.  With a multiple of 8 tiles and one K part, XCD
// x takes the x-th eighth of the tiles in super-block order: 4 weight panels
// (tn) by all row tiles (tm), row tile by row tile -- so the CUs of one XCD
// share few weight panels and activation row tiles in its L2.  Returns
// tn * 65536 + tm; a bijection on the tiles for every grid (plan_check.cpp).
// constexpr: callable from device code.
constexpr int dense_tile_of(int bid, int tiles_m, int tiles_nn, int kparts) {
  const int tiles = tiles_m * tiles_nn;
  const int l = (tiles % 8 == 0 && kparts == 1) ? (bid % 8) * (tiles / 8) + bid / 8 : bid;
  const int sb = l / (4 * tiles_m);
  const int left = tiles_nn - sb * 4;
  const int wsb = left < 4 ? left : 4;
  const int rem = l - sb * 4 * tiles_m;
  return (sb * 4 + rem % wsb) * 65536 + rem / wsb;
}

// Columns [0, n_wide) in 256-wide weight tiles and the rest in 192-wide tiles,
// when that fills the CUs better than 256-wide tiles alone: a GEMM whose
// 256 x 256 tiles need more than one round over the CUs otherwise leaves CUs
// idle in its last round (M = 4096, N = 7168: 448 tiles on 256 CUs = 1.75
// rounds, run as 256 + 256 tiles of 256 and 192 columns).  Work is counted in
// rounds, a 192-wide tile taking 0.8 of a 256-wide one (it keeps the activation
// traffic of the full tile).  Returns N (no split) when nothing gains; *rounds
// is the estimate of what is returned.
inline int prefill_wide_columns(int Mpad, int N, int cus, double* rounds_out = nullptr) {
  const long long tiles_m = Mpad / 256;
  const int nt = static_cast<int>((N + 255LL) / 256);
  auto rounds = [cus](long long tiles) { return static_cast<double>((tiles + cus - 1) / cus); };
  double best = cus > 0 ? rounds(tiles_m * nt) : 1.0;
  int best_wide = N;
  if (cus > 0 && tiles_m * nt > cus) {
    for (int a = 1; a < nt; ++a) {
      const int n2 = N - 256 * a;
      const double est = rounds(tiles_m * a) + 0.8 * rounds(tiles_m * ((n2 + 191LL) / 192)) + 0.02;
      if (est < best - 1e-9) {
        best = est;
        best_wide = 256 * a;
      }
    }
  }
  if (rounds_out) *rounds_out = best;
  return best_wide;
}

// Tile of the LDS-tiled FP8 GEMM (weight rows x tokens).  kTile128x64Two keeps
// the LDS of two workgroups on a CU (shorter stages), the others use it whole.
enum TileId { kTile64x32 = 0, kTile64x64, kTile128x64, kTile128x64Two, kTile128x128, kTile256 };

// What a group of 128 K costs: E4M3 codes with block scales, the same with the
// half-range conversion of every weight fragment, per-token / per-channel (no
// promotion).
enum TileForm { kFormOcp = 0, kFormHalf, kFormChannel };

// Estimated us of one round over the CUs: round + G (group + busy f) + loose,
// f the share of the CUs that the rounds fill, busy_more in the place of busy
// when there is more than one round, loose only where the output rows take no
// wide stores (16 bytes for the 256 x 256 tile, 8 for the others).
struct TileCost {
  double round, group, busy, busy_more, loose;
};

// Which tile: the least estimated time.  The costs are fitted to 3587 measured
// calls on MI355X (all tiles at 65 <= M <= 16384, 256 <= N <= 32768, 256 <= K <=
// 14336, odd N among them; bits are the same for every tile).  Over these the
// chosen tile takes 1.010 (half range 1.001, per-channel 1.007) times the best
// one's time; one set of costs for all three forms, counted in groups alone,
// took 1.016, 1.005 and 1.035 and was up to 15% slower than 256 x 256 tiles where
// it chose others (half range M = 700, N = 6144, K = 14336 308 us against 293;
// M = 4096, N = K = 2048 33.0 against 29.6).
// M = 300, N = 6144, K = 4096: 45.3 us in 48 tiles of 256 x 256, 15.6 us in 240
// tiles of 128 x 64; M = 1024, N = K = 4096: 47.1 and 25.2 us (128 x 128); M =
// 1024, N = 28672: 106 us in 256 x 256 tiles, 162 us in 128 x 128 ones (us of the
// launch, launches back to back).
inline TileId plan_tile(int M, int Mpad, int N, int cus, int G = 32, TileForm form = kFormOcp, bool rows16 = true,
                        bool rows8 = true) {
  if (cus <= 0) return kTile256;
  static constexpr TileCost kCosts[3][6] = {
      {{2.9, 0.205, 0, 0, 0.3}, {3.05, 0.24, 0, 0, 0.6}, {3.75, 0.335, 0, 0, 0.85},
       {2.4, 0.30, 0, 0.018, 1.25}, {4.55, 0.53, 0.113, 0.26, 2.75}, {10.4, 1.11, 0.49, 0.49, 7.1}},
      {{2.7, 0.56, 0, 0, 0.3}, {2.9, 0.615, 0, 0, 0.6}, {3.8, 1.055, 0, 0, 0.8},
       {2.4, 0.925, 0, 0, 0.9}, {4.8, 1.235, 0.075, 0.15, 1.8}, {8.3, 2.53, 0.395, 0.395, 6.9}},
      {{2.95, 0.135, 0, 0, 0.4}, {3.5, 0.175, 0, 0, 0.6}, {4.7, 0.28, 0, 0, 1.05},
       {3.0, 0.294, 0, 0, 1.07}, {7.7, 0.355, 0.158, 0.145, 2.5}, {8.9, 1.0, 0.4, 0.4, 27.0}}};
  // Weights past the 256 MB last-level cache come from HBM in every call; fewer tokens a tile, more fetches of a panel.
  static constexpr double kCold[6] = {1.3, 1.3, 1.3, 1.3, 1.15, 1.05};
  const bool cold = static_cast<long long>(N) * G * 128 > (1LL << 28);
  auto cost = [&](TileId t, double rounds, double tiles, bool wide) {
    const TileCost& c = kCosts[form][t];
    const double f = tiles / cus / rounds;
    const double us = rounds * (c.round + G * (c.group + (rounds > 1.0 ? c.busy_more : c.busy) * f) + (wide ? 0.0 : c.loose));
    return cold ? us * kCold[t] : us;
  };
  double rounds256 = 0.0;
  prefill_wide_columns(Mpad, N, cus, &rounds256);
  const double tiles256 = static_cast<double>(Mpad / 256) * ((N + 255LL) / 256);
  double best = cost(kTile256, rounds256, tiles256 < cus ? tiles256 : cus, rows16);
  TileId id = kTile256;
  auto offer = [&](TileId t, long long bn, long long bm) {
    const long long tiles = ((M + bm - 1) / bm) * ((N + bn - 1) / bn);
    if (tiles > cus && t == kTile128x64) t = kTile128x64Two;  // two workgroups a CU
    const double us = cost(t, static_cast<double>((tiles + cus - 1) / cus), static_cast<double>(tiles), rows8);
    if (us < best) {
      best = us;
      id = t;
    }
  };
  offer(kTile128x128, 128, 128);
  offer(kTile128x64, 128, 64);
  offer(kTile64x64, 64, 64);
  offer(kTile64x32, 64, 32);
  return id;
}

}  // namespace gk
