// bf16 expert products over few rows per batch: C[b] (R x N) = epi(A[b] (R x Kd) . Bt[b]^T + bias[b]), and the
// choice between the tiles of this kernel, of gemm_bf16_mid.h and of gemm_bf16_stream.h.
//
// What bounds them.  With a few dozen rows per expert the 128 x 256 and 256 x 256 tiles
// of gemm_bf16.h make a handful of workgroups that each walk all of k: the second product over one
// image (8 experts x 52 rows x 768 x 3072) was 24 tiles on 256 CUs and 86 us, for 38 MB of weights
// that take 6 us to read.  Small tiles fill the chip; what they cost is operand bytes per flop, and
// a CU takes those at 55 - 80 GB/s (requests of whole 128-byte lines; fragments loaded straight into
// registers, 64 bytes per row, moved at half of that and were dropped: 20 instead of 13 us on the
// first product of the same layer).  Each shape therefore wants the largest tile that still
// occupies every CU, and the tile is chosen from a table of measured constants (RowsTile below).
//
// gemm_bf16_rows_kernel: tiles of 32 x 32 to 32 x 128, one workgroup of 4 waves each; no launch plan (a workgroup past
// its batch's count leaves after one scalar load).  Operands go global memory -> LDS by DMA, 8 rows x 128 bytes per
// request, into a ring of S stages of 64 KT k; the 16-byte pieces of a row are XOR-swizzled so that fragment
// reads meet no bank conflict; fragments of stage t + 1 are read while stage t is multiplied; one
// barrier per stage.  The smallest take 128 k per stage (KT = 2): with one row block per wave a
// stage's MFMAs are shorter than the barrier and the LDS latency around them (second product of one
// 196-token image, 32 x 32 tiles: 13.2 us with KT = 1, 9.6 with KT = 2).
#ifndef VMOE_GEMM_BF16_ROWS_H_
#define VMOE_GEMM_BF16_ROWS_H_
#include "gemm_bf16.h"
#include "gemm_bf16_mid.h"
#include "gemm_bf16_stream.h"

namespace vmoe {

template <int BM_, int BN_, int WM_, int WN_, int STAGES_, int KT_>
struct RowsCfg {
  static constexpr int BM = BM_, BN = BN_, WM = WM_, WN = WN_, S = STAGES_, KT = KT_;
  static constexpr int kWaves = WM * WN, kThreads = 64 * kWaves;
  static constexpr int TM = BM / WM, TN = BN / WN;             // wave tile
  static constexpr int FM = TM / 16, FN = TN / 16;
  static constexpr int kHalfBytes = (BM + BN) * 128;           // 64 k of both operands
  static constexpr int kStageBytes = KT * kHalfBytes, BK = 64 * KT;
  static constexpr int kAIssues = BM / 8 / kWaves, kBIssues = BN / 8 / kWaves;
  static constexpr int kIssues = KT * (kAIssues + kBIssues);          // DMA requests per wave and k tile
  static constexpr int kOutLd = TN + 8;
  static constexpr size_t kOutBytes = (size_t)kWaves * TM * kOutLd * sizeof(bf16_t);
  static constexpr size_t kLdsBytes = (size_t)S * kStageBytes > kOutBytes ? (size_t)S * kStageBytes : kOutBytes;
  static_assert(BM % (8 * kWaves) == 0 && BN % (8 * kWaves) == 0, "whole requests per wave");
  static_assert(S >= 2 && S * kIssues < 64, "vmcnt is a 6-bit counter");
};

// Tiles that a launch may take (VMOE_ROW_TILES counts them, kStreamTiles and kMoreTiles on behind each other), and
// what the choice between them is made from.  A workgroup's round takes fix (+ gelu) microseconds and step1 per
// 64 k, step2 where two of them share the CU; a launch cannot beat its bytes at tbs TB/s nor its flops
// at pflops.  Fitted to 230 random shapes, both products (1 - 128 experts, 24 - 50 000 rows, widths 192 - 1 024,
// weights from memory): rms 6 - 12 % per tile.  The kernel that the choice takes, the tile-walking and the large ones
// among them, is on average 4 - 5 % above the fastest of all tiles where experts are full (230 random layers) and 7 %
// (first product) and 13 % (second) where they are partly filled (310).  The tiles below 64 x 64 are
// gemm_bf16_rows_kernel's, the others gemm_bf16_mid_kernel's.
struct RowsTile {
  int bm, bn, per_cu;
  double fix, step1, step2, gelu, tbs, pflops;
};
constexpr RowsTile kRowsTiles[] = {
    {32, 32, 2, 1.41, 0.13, 0.19, 0, 4.2, 0.33},    {64, 32, 2, 1.55, 0.19, 0.30, 0, 4.2, 0.43},
    {32, 64, 2, 1.33, 0.21, 0.31, 0.1, 4.2, 0.63},  {64, 64, 2, 1.05, 0.30, 0.37, 0.6, 4.0, 0.51},
    {32, 128, 2, 1.14, 0.35, 0.55, 0.5, 4.3, 2.5},  {64, 128, 2, 1.20, 0.41, 0.62, 0.8, 4.4, 0.86},
    {96, 64, 2, 1.00, 0.36, 0.50, 1.0, 4.5, 0.56},  {128, 128, 1, 1.61, 0.50, 0, 2.1, 4.4, 0.79}};
constexpr int kNumRowsTiles = sizeof(kRowsTiles) / sizeof(kRowsTiles[0]);
constexpr RowsTile kMoreTiles[] = {
    {96, 128, 2, 0.75, 0.60, 0.88, 1.7, 4.5, 0.91}, {128, 128, 2, 1.09, 0.65, 0.97, 2.1, 4.5, 0.92},
    {128, 192, 1, 2.13, 0.69, 0, 2.7, 4.5, 0.89},   {256, 192, 1, 2.46, 1.11, 0, 4.6, 3.5, 0.89}};
constexpr int kNumMoreTiles = sizeof(kMoreTiles) / sizeof(kMoreTiles[0]);
// The large tiles in the same terms: the first product's (gemm_bf16_mixed_kernel, and gemm_bf16_kernel where k is no
// multiple of 64), and the second one's eight waves on 256 and on 192 columns.
constexpr RowsTile kFirstProductTile = {128, 256, 2, 2.98, 1.12, 1.66, 2.2, 4.3, 2.5};
constexpr RowsTile kFirstProductK32Tile = {128, 256, 2, 1.28, 1.45, 2.25, 0.8, 4.3, 2.5};
constexpr RowsTile kEightWavesTile = {256, 256, 1, 8.00, 1.23, 0, 0, 5.6, 1.87};
constexpr RowsTile kNarrowTile = {256, 192, 1, 3.69, 0.87, 0, 0, 4.2, 1.34};

// How a launch's tiles are dealt to the dies, whose rounds count: one by one (kDealTiles), all row tiles of a (batch,
// column tile) pair to one die (kDealPairs: a launch of two pairs runs on two dies), or all column tiles of a row tile
// (kDealRows: launch plans.  35 row tiles of seven column tiles each are 245 tiles for 256 CUs, and 35 for the 32 of a
// die: 5 experts x 800 rows x 832 x 3 328, second product, on 128 x 128: 60.6 us, on 64 x 128 35.9).
enum TileDeal { kDealTiles, kDealPairs, kDealRows };

// Time in microseconds of a product on tiles of this kind.
inline double product_us(const RowsTile& t, int batch, int R, int N, int Kd, bool gelu, TileDeal deal) {
  const double row_tiles = (R + t.bm - 1) / t.bm, tiles_n = (N + t.bn - 1) / t.bn;
  const double on_die = deal == kDealPairs  ? std::ceil(batch * tiles_n / kNumXcd) * row_tiles
                        : deal == kDealRows ? std::ceil(batch * row_tiles / kNumXcd) * tiles_n
                                            : std::ceil(batch * tiles_n * row_tiles / kNumXcd);
  const double full = (double)kCusPerXcd * t.per_cu;
  const double fix = t.fix + (gelu ? t.gelu : 0);
  const int nk = (Kd + 63) / 64;
  const double one = fix + nk * t.step1, two = 1.35 * fix + nk * t.step2;
  const double rounds = std::floor(on_die / full), rest = on_die - rounds * full;
  const double busy = rounds * (t.per_cu == 2 ? two : one) + (rest > kCusPerXcd ? two : rest > 0 ? one : 0);
  const double weights = (double)batch * N * Kd, memory = 2e-6 * (weights + (double)batch * R * (Kd + N)) / t.tbs;
  const double matrix = 2e-9 * weights * R / t.pflops;
  // (their 4-norm.  A layer's calls estimate every tile of both products several times: with pow() that was
  // 11 us of the host's 60 on one image.)
  const double b2 = busy * busy, m2 = memory * memory, f2 = matrix * matrix;
  return 2 + std::sqrt(std::sqrt(b2 * b2 + m2 * m2 + f2 * f2));
}

// The same for a launch whose live rows (partly: some of all) are counted on the device: the mean over full, 70 % full and 40 % full
// experts.  On 80 random ragged layers, 23 % to all of their rows live, the choice by this mean takes 6 514 us for the
// 160 products, by the time of full experts 6 566 and 39 % too long at worst instead of 18 %, on the best tile of each 6 113.
inline double launch_us(const RowsTile& t, int batch, int R, int N, int Kd, bool gelu, TileDeal deal, bool partly) {
  const double us = product_us(t, batch, R, N, Kd, gelu, deal);
  if (!partly) return us;
  return (us + product_us(t, batch, (int)std::ceil(0.7 * R), N, Kd, gelu, deal) +
          product_us(t, batch, (int)std::ceil(0.4 * R), N, Kd, gelu, deal)) / 3;
}

// The tiles of gemm_bf16_stream_kernel, and what the choice
// is made from: a CU takes its tiles one after the other at step_us per 64 k, with the GELU's or the plain
// epilogue behind each, and the launch cannot beat its weights at w_tbs plus its rows, once per column
// tile, at a_tbs.  Fitted to 106 random shapes (4 - 128 experts, 12 - 128 rows, widths 384 - 4096; either product):
// rms 5 % and less per tile, 30 % at worst.
struct StreamTile {
  int bm, bn;
  double step_us, gelu_us, plain_us, fix_us, lat_us, w_tbs, a_tbs;
};
constexpr StreamTile kStreamTiles[] = {
    {64, 192, 0.57, 3.8, 4.0, 2.0, 3.4, 8.5, 8.0},   {64, 256, 0.73, 4.1, 2.7, 2.0, 2.0, 7.3, 8.0},
    {128, 128, 0.58, 3.3, 2.9, 3.0, 7.0, 9.0, 20.0}, {128, 256, 0.93, 6.1, 4.1, 2.0, 5.0, 6.9, 63.0},
    {128, 192, 0.77, 4.7, 3.4, 2.0, 6.4, 9.0, 19.3}};
constexpr int kNumStreamTiles = sizeof(kStreamTiles) / sizeof(kStreamTiles[0]);

// f(StreamCfg of tile i).
template <typename F>
inline auto with_stream_tile(int i, F&& f) {
  switch (i) {
    case 0: return f(StreamCfg<64, 192, 4, 2, 3, 5>{});
    case 1: return f(StreamCfg<64, 256, 1, 8, 3, 4>{});
    case 2: return f(StreamCfg<128, 128, 2, 4, 3, 6>{});
    case 3: return f(StreamCfg<128, 256, 2, 4, 3, 3>{});
    default: return f(StreamCfg<128, 192, 4, 2, 3, 4>{});
  }
}

inline bool stream_tile_ok(int i, int batch, int R, int Kd, bool ragged) {
  return i >= 0 && i < kNumStreamTiles && with_stream_tile(i, [&](auto cfg) {
    return stream_gemm_ok<decltype(cfg)>(batch, R, Kd, ragged);
  });
}

// Time of tile i of kStreamTiles, 1e30 where the kernel does not take the product.  (Below 24 rows most of a tile is
// padding and the 32-row tiles win.)
inline double stream_us(int i, int batch, int R, int N, int Kd, bool ragged, bool gelu) {
  if (R < 24 || !stream_tile_ok(i, batch, R, Kd, ragged)) return 1e30;
  const StreamTile& s = kStreamTiles[i];
  const double units = (double)batch * ((N + s.bn - 1) / s.bn);
  const double rounds = std::ceil(std::ceil(units / kNumXcd) / kCusPerXcd);
  const double busy = s.fix_us + rounds * ((Kd + 63) / 64 * s.step_us + (gelu ? s.gelu_us : s.plain_us));
  const double memory = s.lat_us + 2e-6 * Kd * ((double)batch * N / s.w_tbs + units * s.bm / s.a_tbs);
  return std::sqrt(std::sqrt(busy * busy * busy * busy + memory * memory * memory * memory));
}

constexpr int kFirstMoreTile = kNumRowsTiles + kNumStreamTiles;
inline bool is_mid_tile(int i) {
  return i == 3 || (i >= 5 && i < kNumRowsTiles) || (i >= kFirstMoreTile && i < kFirstMoreTile + kNumMoreTiles);
}
// f(MidCfg of tile i).
template <typename F>
inline auto with_mid_tile(int i, F&& f) {
  switch (i) {
    case 3: return f(MidCfg<64, 64, 2, 2, 2, 2, 2>{});
    case 5: return f(MidCfg<64, 128, 2, 2, 3, 2, 1>{});
    case 6: return f(MidCfg<96, 64, 2, 2, 2, 2, 2>{});
    case 7: return f(MidCfg<128, 128, 2, 4, 4, 1, 1>{});
    case kFirstMoreTile: return f(MidCfg<96, 128, 2, 2, 2, 2, 1>{});
    case kFirstMoreTile + 1: return f(MidCfg<128, 128, 2, 2, 2, 2, 1>{});
    case kFirstMoreTile + 2: return f(MidCfg<128, 192, 4, 2, 3, 1, 1>{});
    default: return f(MidCfg<256, 192, 4, 2, 2, 1, 1>{});
  }
}

// Whether a ragged launch of a tile of gemm_bf16_mid.h has a plan: with two row tiles per die and more.  Below that
// (batch, column tile) pairs go round the dies, which is as even.
inline bool mid_tile_planned(int batch, int R, int bm) { return (long long)batch * ((R + bm - 1) / bm) >= 2 * kNumXcd; }

// Whether the kernel takes the operands: whole 16-byte pieces, 31-bit byte offsets inside a batch.
inline bool rows_gemm_ok(int R, int N, int Kd, long long items) {
  const uint64_t lim = 1ull << 31;
  return N % 8 == 0 && Kd % 8 == 0 && (uint64_t)R * Kd * 2 < lim && (uint64_t)N * Kd * 2 < lim &&
         (uint64_t)items * Kd * 2 < lim;
}

// The tile that should run the product in less than `us` microseconds, the time of the large tiles, or -1.
// (ragged: the rows' counts stand on the device; partly: and may be fewer than all; walkers: whether kStreamTiles are
// among the tiles)
inline int best_tile(int batch, int R, int N, int Kd, long long items, bool ragged, bool partly, bool gelu, double us,
                     bool walkers = true) {
  int best = -1;
  auto take = [&](int i, double t) {
    if (t < us) { us = t; best = i; }
  };
  const bool mid_ok = mid_gemm_ok(batch, R, N, Kd, items);
  auto take_tile = [&](int i, const RowsTile& t) {
    const bool mid = is_mid_tile(i);
    if (!mid || mid_ok)
      take(i, launch_us(t, batch, R, N, Kd, gelu,
                        !mid || (ragged && !mid_tile_planned(batch, R, t.bm)) ? kDealPairs : ragged ? kDealRows : kDealTiles, partly));
  };
  for (int i = 0; i < kNumRowsTiles; ++i) take_tile(i, kRowsTiles[i]);
  for (int i = 0; i < kNumMoreTiles; ++i) take_tile(kFirstMoreTile + i, kMoreTiles[i]);
  // (8 % ahead: no tile walker where another kernel is as good)
  for (int i = 0; walkers && i < kNumStreamTiles; ++i) take(kNumRowsTiles + i, 1.08 * stream_us(i, batch, R, N, Kd, ragged, gelu));
  return best;
}

// `guard`: the plan of the other product of the call, where that one has a plan: a launch whose
// plan was not written for this geometry runs nothing, and neither does this one.
template <typename Cfg, int EPI>
__global__ __launch_bounds__(Cfg::kThreads, 2) void gemm_bf16_rows_kernel(
    const bf16_t* __restrict__ A, const bf16_t* __restrict__ Bt, const bf16_t* __restrict__ bias,
    bf16_t* __restrict__ C, int R, int N, int Kd, int tiles_m, int tiles_n, int batch,
    const int32_t* __restrict__ rows, const int32_t* __restrict__ a_rows, int a_items,
    PlanRef guard, int32_t* __restrict__ clear, int clear_count, int32_t* __restrict__ status) {
#if defined(__HIP_DEVICE_COMPILE__)
  constexpr int FM = Cfg::FM, FN = Cfg::FN, S = Cfg::S, L = Cfg::kIssues, W = Cfg::kWaves, KS = 2 * Cfg::KT;
  extern __shared__ __align__(1024) unsigned char smem[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / Cfg::WN, wn = wave % Cfg::WN;
  if (blockIdx.x == 0) begin_call(clear, clear_count, status, tid, Cfg::kThreads);
  if (guard.entries != nullptr && guard.entries[guard.blocks].y != guard.tag) {
    if (blockIdx.x == 0 && tid == 0 && status != nullptr) status[kStatusPlanMismatches] += 1;
    return;
  }
  // (batch, column tile) pairs go round the dies; the row tiles of a pair follow each other on
  // one die, so its weights come from memory once.
  const int xcd = blockIdx.x % kNumXcd, idx = blockIdx.x / kNumXcd;
  const int pair = idx / tiles_m * kNumXcd + xcd, tile_m = idx % tiles_m;
  if (pair >= batch * tiles_n) return;
  const int b = pair / tiles_n, tile_n = pair - b * tiles_n;
  const int row0 = tile_m * Cfg::BM, col0 = tile_n * Cfg::BN;
  int live = R;
  if (rows != nullptr) {
    live = min(rows[b], R);
    if (row0 >= live) return;
  }
  // Requests: lane l of a request fetches a 16-byte piece of row l / 8; the piece is the one
  // that the XOR swizzle (row / 2) % 8 puts at position l % 8 of the row in LDS.
  const int lrow = lane >> 3;
  const int piece = (lane & 7) ^ ((wave * 4 + (lrow >> 1)) & 7);
  uint32_t a_off[Cfg::kAIssues], b_off[Cfg::kBIssues];
#pragma unroll
  for (int i = 0; i < Cfg::kBIssues; ++i)
    b_off[i] = (uint32_t)min(col0 + (i * W + wave) * 8 + lrow, N - 1) * (uint32_t)Kd * 2u + piece * 16u;
#pragma unroll
  for (int i = 0; i < Cfg::kAIssues; ++i) {
    int r = min(row0 + (i * W + wave) * 8 + lrow, live - 1);
    if (a_rows != nullptr) {
      r = a_rows[(size_t)b * R + r];
      r = (unsigned)r < (unsigned)a_items ? r : 0;
    }
    a_off[i] = (uint32_t)r * (uint32_t)Kd * 2u + piece * 16u;
  }
  // Addresses past an operand's end (k past Kd in its last row) read as zero, as long as the scalar
  // offset itself lies inside the operand: the range check is num_records - offset, unsigned.  A second
  // half of the last stage may start past Kd, which one row (or a few short ones) may all be: it takes
  // the row's first half again, and its fragments are cleared like every k past Kd.
  const bf16_t* Ab = a_rows != nullptr ? A : A + (size_t)b * R * Kd;
  const uint32_t a_bytes = (uint32_t)(a_rows != nullptr ? a_items : R) * (uint32_t)Kd * 2u;
  const __amdgpu_buffer_rsrc_t a_rsrc =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16_t*>(Ab), 0, (int)a_bytes, 0x00020000);
  const __amdgpu_buffer_rsrc_t b_rsrc = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<bf16_t*>(Bt + (size_t)b * N * Kd), 0, (int)((uint32_t)N * (uint32_t)Kd * 2u), 0x00020000);
  auto request = [&](int stage, int kt) {
#pragma unroll
    for (int h = 0; h < Cfg::KT; ++h) {
      unsigned char* s = smem + stage * Cfg::kStageBytes + h * Cfg::kHalfBytes;
      const int half = kt * Cfg::KT + h, k_bytes = Cfg::KT == 1 || half * 64 < Kd ? half * 128 : 0;
#pragma unroll
      for (int i = 0; i < Cfg::kBIssues; ++i)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(
            b_rsrc, (lds_ptr_t)(s + Cfg::BM * 128 + (i * W + wave) * 1024), 16, b_off[i], k_bytes, 0, 0);
#pragma unroll
      for (int i = 0; i < Cfg::kAIssues; ++i)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(a_rsrc, (lds_ptr_t)(s + (i * W + wave) * 1024), 16,
                                                 a_off[i], k_bytes, 0, 0);
    }
  };

  const int r16 = lane & 15, q = lane >> 4;
  uint2 bias_pk[FN];
#pragma unroll
  for (int j = 0; j < FN; ++j) {
    bias_pk[j] = make_uint2(0, 0);
    if (bias != nullptr)
      __builtin_memcpy(&bias_pk[j], bias + (size_t)b * N + min(col0 + wn * Cfg::TN + j * 16 + q * 4, N - 4), 8);
  }
  floatx4 acc[FM][FN];
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j) acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};

  // v_mfma_f32_16x16x32_bf16: a lane supplies 8 consecutive k of one row (row = lane % 16, k from
  // (lane / 16) * 8).  The fragment reads are written as instructions: a read that the compiler
  // can see waits for every request in flight.
  typedef float frag_t __attribute__((ext_vector_type(4)));
  const uint32_t lds0 = (uint32_t)reinterpret_cast<uintptr_t>((lds_ptr_t)smem);
  const uint32_t a_row = lds0 + (wm * Cfg::TM + r16) * 128;
  const uint32_t b_row = lds0 + Cfg::BM * 128 + (wn * Cfg::TN + r16) * 128;
  const uint32_t pos[2] = {(uint32_t)((q ^ (r16 >> 1)) * 16), (uint32_t)(((4 + q) ^ (r16 >> 1)) * 16)};
  frag_t fa[2][KS][FM], fb[2][KS][FN];
  auto read_frags = [&](const int u, int stage) {
    const uint32_t s = stage * Cfg::kStageBytes;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
#pragma unroll
      for (int j = 0; j < FN; ++j)
        asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(fb[u][ks][j]) : "v"(b_row + s + pos[ks & 1]), "n"(j * 2048 + (ks >> 1) * Cfg::kHalfBytes));
#pragma unroll
      for (int i = 0; i < FM; ++i)
        asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(fa[u][ks][i]) : "v"(a_row + s + pos[ks & 1]), "n"(i * 2048 + (ks >> 1) * Cfg::kHalfBytes));
    }
  };
  const int nk = (Kd + Cfg::BK - 1) / Cfg::BK;
  // Iteration t: the wave's fragments of k tile t have arrived and its requests of t + 1 have
  // landed; barrier (everyone's have, and everyone has read stage t % S); requests of t + S into
  // that stage; fragment reads of t + 1; MFMAs of t.
  auto step = [&](const int u, int t, int stage) {
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
#pragma unroll
      for (int j = 0; j < FN; ++j) asm volatile("" : "+v"(fb[u][ks][j]));
#pragma unroll
      for (int i = 0; i < FM; ++i) asm volatile("" : "+v"(fa[u][ks][i]));
    }
    if (t + 1 < nk) {
      if (nk - 2 - t >= S - 2) wait_vmcnt<(S - 2) * L>();     // k tiles requested behind t + 1
      else wait_vmcnt<0>();
      raw_barrier();
      if (t + S < nk) request(stage, t + S);
      read_frags(1 - u, stage + 1 == S ? 0 : stage + 1);
    } else if (Kd % Cfg::BK != 0) {           // the last k tile ends inside: k past Kd counts as zero
#pragma unroll
      for (int ks = 0; ks < KS; ++ks)
        if (t * Cfg::BK + ks * 32 + q * 8 >= Kd) {
#pragma unroll
          for (int j = 0; j < FN; ++j) fb[u][ks][j] = frag_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int i = 0; i < FM; ++i) fa[u][ks][i] = frag_t{0.f, 0.f, 0.f, 0.f};
        }
    }
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
#pragma unroll
      for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              __builtin_bit_cast(bf16x8, fb[u][ks][j]), __builtin_bit_cast(bf16x8, fa[u][ks][i]),
              acc[i][j], 0, 0, 0);
  };
  static_for<S>([&](auto s) {
    if (s < nk) request(s, s);
  });
  if (nk >= S) wait_vmcnt<(S - 1) * L>();
  else wait_vmcnt<0>();
  raw_barrier();
  read_frags(0, 0);
  int stage = 0;
  for (int t = 0; t < nk; t += 2) {
    step(0, t, stage);
    stage = stage + 1 == S ? 0 : stage + 1;
    if (t + 1 < nk) {
      step(1, t + 1, stage);
      stage = stage + 1 == S ? 0 : stage + 1;
    }
  }
  __syncthreads();       // every wave has its last fragments: the ring is free for the output
  mfma_result_fence();
  // acc[i][j]: row i * 16 + lane % 16, columns j * 16 + (lane / 16) * 4 .. +3 of the wave tile, which
  // passes through a wave-private LDS region and leaves as 16-byte row-contiguous pieces.
  bf16_t* so = reinterpret_cast<bf16_t*>(smem) + (size_t)wave * Cfg::TM * Cfg::kOutLd;
  auto put = [&](auto has_bias) {
    constexpr bool kHasBias = decltype(has_bias)::value;
#pragma unroll
    for (int j = 0; j < FN; ++j)
#pragma unroll
      for (int i = 0; i < FM; ++i) {
        const uint32_t p0 = epilogue_pair<EPI, kHasBias>(acc[i][j][0], acc[i][j][1], bf_lo(bias_pk[j].x), bf_hi(bias_pk[j].x));
        const uint32_t p1 = epilogue_pair<EPI, kHasBias>(acc[i][j][2], acc[i][j][3], bf_lo(bias_pk[j].y), bf_hi(bias_pk[j].y));
        *reinterpret_cast<uint2*>(so + (i * 16 + r16) * Cfg::kOutLd + j * 16 + q * 4) = make_uint2(p0, p1);
      }
  };
  if (bias != nullptr) put(std::true_type{});
  else put(std::false_type{});
  constexpr int kPieces = Cfg::TN / 8, kPasses = (Cfg::TM * kPieces + 63) / 64;
  bf16_t* Cb = C + (size_t)b * R * N;
#pragma unroll
  for (int p = 0; p < kPasses; ++p) {
    const int id = p * 64 + lane, r = id / kPieces, c = (id % kPieces) * 8;
    const int row = row0 + wm * Cfg::TM + r, col = col0 + wn * Cfg::TN + c;
    if (r < Cfg::TM && row < live && col < N)
      *reinterpret_cast<uint4*>(Cb + (size_t)row * N + col) =
          *reinterpret_cast<const uint4*>(so + r * Cfg::kOutLd + c);
  }
#endif
}

template <typename Cfg, int EPI>
int launch_rows_tile(const bf16_t* A, const bf16_t* Bt, const bf16_t* bias, bf16_t* C, int batch, int R,
                     int N, int Kd, hipStream_t stream, const int32_t* rows, const int32_t* a_rows,
                     int a_items, PlanRef guard, int32_t* clear, int clear_count, int32_t* status) {
  const int tiles_m = (R + Cfg::BM - 1) / Cfg::BM, tiles_n = (N + Cfg::BN - 1) / Cfg::BN;
  const long long pairs = (long long)batch * tiles_n;
  const long long blocks = (pairs + kNumXcd - 1) / kNumXcd * kNumXcd * tiles_m;
  if (blocks > 0x7fffffffLL || pairs > 0x7ffffff0LL) return VMOE_E_OVERFLOW;
  auto kern = gemm_bf16_rows_kernel<Cfg, EPI>;
  hipError_t e = allow_dynamic_lds(reinterpret_cast<const void*>(kern), Cfg::kLdsBytes);
  if (e != hipSuccess) return (int)e;
  hipLaunchKernelGGL(kern, dim3((unsigned)blocks), dim3(Cfg::kThreads), Cfg::kLdsBytes, stream, A, Bt,
                     bias, C, R, N, Kd, tiles_m, tiles_n, batch, rows, a_rows, a_items, guard, clear,
                     clear_count, status);
  return launch_status();
}

// `tile`: index into kRowsTiles, behind them into kStreamTiles, behind those into kMoreTiles.  `plan`: the launch
// plan of a ragged product on a tile of gemm_bf16_mid_kernel, or none.
template <int EPI>
int launch_gemm_bf16_rows(int tile, const bf16_t* A, const bf16_t* Bt, const bf16_t* bias, bf16_t* C,
                          int batch, int R, int N, int Kd, hipStream_t stream, const int32_t* rows, const int4* plan,
                          const int32_t* a_rows, int a_items, PlanRef guard, int32_t* clear,
                          int clear_count, int32_t* status) {
  auto run = [&](auto cfg) {
    return launch_rows_tile<decltype(cfg), EPI>(A, Bt, bias, C, batch, R, N, Kd, stream, rows, a_rows,
                                                a_items, guard, clear, clear_count, status);
  };
  if (is_mid_tile(tile))
    return with_mid_tile(tile, [&](auto cfg) {
      return launch_mid_tile<decltype(cfg), EPI>(A, Bt, bias, C, batch, R, N, Kd, stream, rows, plan, a_rows,
                                                 a_items, guard, clear, clear_count, status);
    });
  if constexpr (EPI == kEpiBiasOnce) {
    if (tile >= kNumRowsTiles) return VMOE_E_UNSUPPORTED;      // (dense layers leave the tile walkers to the MLPs)
  } else if (tile >= kNumRowsTiles)
    return with_stream_tile(tile - kNumRowsTiles, [&](auto cfg) {
      return launch_gemm_bf16_stream<decltype(cfg), EPI>(A, Bt, bias, C, batch, R, N, Kd, stream, rows, a_rows,
                                                         a_items, guard, clear, clear_count, status);
    });
  switch (tile) {
    case 0: return run(RowsCfg<32, 32, 2, 2, 4, 2>{});
    case 1: return run(RowsCfg<64, 32, 2, 2, 3, 2>{});
    case 2: return run(RowsCfg<32, 64, 2, 2, 3, 2>{});
    case 4: return run(RowsCfg<32, 128, 1, 4, 4, 1>{});
  }
  return VMOE_E_UNSUPPORTED;
}

}  // namespace vmoe
#endif  // VMOE_GEMM_BF16_ROWS_H_
