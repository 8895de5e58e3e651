// float32 expert products (vmoe/nn/vit_moe.py:38-45 on float32 parameters) on the bfloat16 matrix
// cores: every operand value is taken apart into three bfloat16 values whose sum it is exactly (Henry, Tang and
// Heinecke, "Leveraging the bfloat16 artificial intelligence datatype for higher-precision computations", 2019).
//
// C[b] = epilogue(A[b] (R x Kd) . B[b] (Kd x N) + bias[b]); B in the reference's (in, out) order.
//
// v = hi + mid + lo, each rounded to nearest from what the ones before it leave: 8 + 8 + 8 bits hold
// a float32 significand.  Of the nine products six are taken (lo.hi, hi.lo, mid.mid, mid.hi, hi.mid,
// hi.hi, in this order, float32 accumulators); the three left out add up to 2^-24 of |a||b| at most (split3), the
// rounding of a float32 product.  One instruction adds 32 products to a sum in place of two, so there
// are fewer roundings along k than on v_mfma_f32_32x32x2_f32: against 64 bits the MLPs of eleven
// shapes (D 384 .. 832, M 1 408 .. 3 328, 22 .. 9 216 rows) are off by 6.8e-7 .. 1.0e-6 in place of 8.1e-7 ..
// 1.2e-6 (2-norm), 15 % less on each.  Values below 2^-110 lose low bits to the exponent range (absolute
// error below 2^-134); an infinite operand, or one that rounds to infinity, leaves inf - inf or inf * 0
// in the cross terms, and sums that come out infinite or NaN are taken again in float32.
//
// Why: a float32 MFMA does 256 flops a clock and CU, a bfloat16 one 4 096: 683 after six products.
// 9 216 rows, 768 x 3 072 (both products): 359 and 379 us (115 TFLOP/s, 0.74 of the float32 peak) on
// float32 MFMAs with operands by LDS-DMA, 240 and 229 (185) here; 51 experts x ~330 rows x 896 x 1 984: 589 and
// 611 to 398 and 406; 8 x 392 x 512 x 2 048: 81 and 79 to 50 and 51; 23 x 22 x 576 x 2 304: 38 and 48 to
// 26 and 26.  The large shapes run at 1.1 PFLOP/s of bfloat16 MFMAs, which is where the
// bfloat16 products of this library stand at the chip's power limit.
//
// Structure.  A k tile is fetched into registers (16-byte loads, one k tile ahead), split there and
// written to LDS as three planes of rows of BK bfloat16, 16-byte pieces XOR-swizzled by row / 2; B is
// transposed on the way (a thread holds 4 k x 4 columns; the columns of a group of 32 are written in
// 8 x 4 order, so that eight lanes with neighbouring column quads write neighbouring rows: no bank
// conflicts).  Splitting costs 5.5 VALU instructions per value, 0.46 of a 128 x 128 tile's MFMA time:
// it hides only behind another workgroup's MFMAs, so the LDS holds one stage and two (128 x 128) or
// four workgroups share a CU, and a wave that splits goes first (s_setprio: 4 - 8 % on the large shapes).
// Measured and not kept: two LDS stages with the split between the MFMAs of the same wave
// (128 x 256 tiles, eight waves: 250 and 228 us on the 9 216 rows); three 128 x 128 workgroups per CU
// (spills, 320); k tiles two or four ahead (no change).
// KG groups of four waves in a workgroup take consecutive runs of k tiles, each through its own LDS,
// and add their sums in group order: launches of few tiles are as long as one tile's chain of k tiles.  Two or four
// groups of the larger tiles take turns at splitting and multiplying.
// The tile comes from the sizes of the call (kSplitTiles), so the order of an output's sums does too: the same item
// through the same weights can differ in its last bits between calls over different numbers of rows or experts
// (not between dense, ragged and gathered calls of one size), as bfloat16 MLPs can.
// Workgroups -> tiles: the live tiles of all batches (row counts are read by every workgroup) are
// numbered batch-major, column panel by column panel, and cut into eight equal runs, one per XCD, so that
// the row tiles that share a column panel of weights run on one die at the same time.
#pragma once
#include <cmath>

#include "gemm_bf16.h"

namespace vmoe {

typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef f32x4_t f32x4_any_t __attribute__((aligned(4)));    // weights come at any float address
typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));

// The tanh GELU by tanhf, off from 64 bits by 3.8e-8 (2-norm, normal inputs), where kEpiBiasGeluTanh takes the
// hardware's exp2 and reciprocal, 4.7e-8.  (A form of its own: a branch in the epilogue cost the other 3 %.)
constexpr int kEpiBiasGeluTanhf = 3;

template <int BM_, int BN_, int WM_, int WN_, int BK_, int WGS_, int KG_>
struct SplitCfg {
  static constexpr int BM = BM_, BN = BN_, BK = BK_, WM = WM_, WN = WN_, kWgs = WGS_;
  static constexpr int KG = KG_, kWaves = WM * WN, kGroup = 64 * kWaves, kThreads = KG * kGroup;
  static constexpr int TM = BM / WM, TN = BN / WN, FM = TM / 16, FN = TN / 16;
  static constexpr int kQuads = BK / 4;                         // 4-wide k pieces of a k tile
  static constexpr int AI = BM * kQuads / kGroup;             // float4 of A per thread and k tile
  static constexpr int BU = (BN / 4) * kQuads / kGroup;       // 4 x 4 blocks of B per thread and k tile
  static constexpr int kRowBytes = BK * 2, kSwz = BK / 8 - 1;
  static constexpr int kAPlane = BM * kRowBytes, kBPlane = BN * kRowBytes;
  static constexpr int kStage = 3 * (kAPlane + kBPlane);
  static constexpr int kOutStride = TN + 4;                     // floats per staged output row
  static constexpr int kSumBytes = KG > 1 ? FM * FN * 16 * kGroup : 0, kOutBytes = kWaves * 16 * kOutStride * 4;
  static constexpr int kPiece = kStage > kOutBytes ? (kStage > kSumBytes ? kStage : kSumBytes)
                                                   : (kOutBytes > kSumBytes ? kOutBytes : kSumBytes);
  static constexpr int kLds = KG * kPiece;
  static constexpr bool kTurns = KG > 2 || (KG == 2 && BM * BN >= 64 * 128);      // groups take turns (see below)
  static_assert(AI >= 1 && BU >= 1, "tile");
};

template <int EPI, typename Cfg>
__global__ __launch_bounds__(Cfg::kThreads, Cfg::kWgs * Cfg::kThreads / 256) void gemm_f32_split_kernel(
    const float* __restrict__ A, const float* __restrict__ B, const float* __restrict__ bias,
    float* __restrict__ C, int batch, int R, int N, int Kd, int tiles_n,
    const int32_t* __restrict__ rows, const int32_t* __restrict__ a_rows, int a_items) {
  extern __shared__ __align__(1024) unsigned char smem[];
  constexpr int BM = Cfg::BM, BN = Cfg::BN, BK = Cfg::BK, FM = Cfg::FM, FN = Cfg::FN;
  const int lane = threadIdx.x & 63;
  const int group = __builtin_amdgcn_readfirstlane(threadIdx.x / Cfg::kGroup);
  const int tid = threadIdx.x - group * Cfg::kGroup;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  unsigned char* const piece = smem + group * Cfg::kPiece;

  // Workgroup -> tile (see above).
  int b, tile_m, tile_n, live = R;
  {
    const int xcd = blockIdx.x & 7, slot = blockIdx.x >> 3;
    if (rows == nullptr) {
      const int tiles_m = (R + BM - 1) / BM, per_batch = tiles_m * tiles_n, total = batch * per_batch;
      const int per_xcd = (total + 7) >> 3, id = xcd * per_xcd + slot;
      if (slot >= per_xcd || id >= total) return;
      b = id / per_batch;
      const int rem = id - b * per_batch;
      tile_n = rem / tiles_m;
      tile_m = rem - tile_n * tiles_m;
    } else {
      int total = 0;
      for (int e0 = 0; e0 < batch; e0 += 64) {
        int t = e0 + lane < batch ? (max(min(rows[e0 + lane], R), 0) + BM - 1) / BM * tiles_n : 0;
        for (int o = 32; o > 0; o >>= 1) t += __shfl_xor(t, o, kWave);
        total += t;
      }
      const int per_xcd = (total + 7) >> 3;
      int id = xcd * per_xcd + slot;
      if (slot >= per_xcd || id >= total) return;
      b = 0;
      for (int e0 = 0; e0 < batch; e0 += 64) {
        const int n = e0 + lane < batch ? max(min(rows[e0 + lane], R), 0) : 0;
        int incl = (n + BM - 1) / BM * tiles_n;
        for (int o = 1; o < 64; o <<= 1) {
          const int up = __shfl_up(incl, o, kWave);
          if (lane >= o) incl += up;
        }
        const uint64_t past = __ballot(incl > id);
        if (past != 0) {
          const int l = __builtin_ctzll(past);
          b = e0 + l;
          live = __shfl(n, l, kWave);
          if (l > 0) id -= __shfl(incl, l - 1, kWave);
          break;
        }
        id -= __shfl(incl, 63, kWave);
      }
      b = __builtin_amdgcn_readfirstlane(b);
      live = __builtin_amdgcn_readfirstlane(live);
      id = __builtin_amdgcn_readfirstlane(id);
      const int tiles_m = (live + BM - 1) / BM;
      tile_n = id / tiles_m;
      tile_m = id - tile_n * tiles_m;
    }
  }
  const int row0 = tile_m * BM, col0 = tile_n * BN;
  const int wm = wave / Cfg::WN, wn = wave - wm * Cfg::WN;
  const int r16 = lane & 15, q = lane >> 4;

  // What a thread stages of a k tile.
  constexpr int KQ = Cfg::kQuads;
  const int akq = tid % KQ;
  const float* a_base = a_rows != nullptr ? A : A + ((size_t)b * R + row0) * Kd;
  uint32_t a_off[Cfg::AI];
  uint32_t a_lds[Cfg::AI];
#pragma unroll
  for (int i = 0; i < Cfg::AI; ++i) {
    const int r = i * (Cfg::kGroup / KQ) + tid / KQ;
    int arow = min(r, live - 1 - row0);
    if (a_rows != nullptr) {
      arow = a_rows[(size_t)b * R + row0 + arow];
      arow = (unsigned)arow < (unsigned)a_items ? arow : 0;
    }
    a_off[i] = (uint32_t)arow * (uint32_t)Kd + akq * 4;
    a_lds[i] = r * Cfg::kRowBytes + (((akq >> 1) ^ ((r >> 1) & Cfg::kSwz)) << 4) + (akq & 1) * 8;
  }
  // B: lanes of a wave take 8 neighbouring column quads x 8 k quads
  constexpr int NG = BN / 32;                      // groups of 32 columns
  int b_nq[Cfg::BU], b_kq[Cfg::BU];
#pragma unroll
  for (int i = 0; i < Cfg::BU; ++i) {
    const int u = i * Cfg::kWaves + wave;                      // (column group, k octet of quads)
    b_nq[i] = (u % NG) * 8 + (lane & 7);
    b_kq[i] = (u / NG) * 8 + (lane >> 3);
  }
  const float* Bb = B + (size_t)b * Kd * N;

  f32x4_t ra[Cfg::AI], rb[Cfg::BU][4];
  auto fetch = [&](int kt) {
    const int k0 = kt * BK;
    const bool tail = k0 + BK > Kd;
#pragma unroll
    for (int i = 0; i < Cfg::AI; ++i) {
      if (!tail || k0 + akq * 4 < Kd)
        ra[i] = *reinterpret_cast<const f32x4_t*>(a_base + a_off[i] + k0);
      else
        ra[i] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
    }
#pragma unroll
    for (int i = 0; i < Cfg::BU; ++i) {
      const int n = min(col0 + b_nq[i] * 4, N - 4);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        int k = k0 + b_kq[i] * 4 + j;
        if (tail) k = min(k, Kd - 1);
        rb[i][j] = *reinterpret_cast<const f32x4_any_t*>(Bb + (size_t)k * N + n);
      }
    }
  };
  // Units of a thread's staging: AI pieces of A rows, then BU x 4 pieces of B columns.
  constexpr int kUnits = Cfg::AI + Cfg::BU * 4;
  auto stage_unit = [&](const int unit) {
    f32x4_t v;
    uint32_t at, plane;
    if (unit < Cfg::AI) {
      v = ra[unit];
      at = a_lds[unit];
      plane = Cfg::kAPlane;
    } else {
      const int i = (unit - Cfg::AI) >> 2, j = (unit - Cfg::AI) & 3;
      v = (f32x4_t){rb[i][0][j], rb[i][1][j], rb[i][2][j], rb[i][3][j]};
      // LDS row of column n: columns of a group of 32 transposed 8 x 4, so that the eight
      // lanes that hold neighbouring quads write neighbouring rows
      const int r = (b_nq[i] >> 3) * 32 + j * 8 + (lane & 7);
      at = 3 * Cfg::kAPlane + r * Cfg::kRowBytes + (((b_kq[i] >> 1) ^ ((r >> 1) & Cfg::kSwz)) << 4) + (b_kq[i] & 1) * 8;
      plane = Cfg::kBPlane;
    }
    u32x2_t p[3];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      uint32_t hi, mid, lo;
      split3(v[2 * h], v[2 * h + 1], hi, mid, lo);
      p[0][h] = hi; p[1][h] = mid; p[2][h] = lo;
    }
#pragma unroll
    for (int t = 0; t < 3; ++t) *reinterpret_cast<u32x2_t*>(piece + t * plane + at) = p[t];
  };
  f32x4_t acc[FM][FN];
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j) acc[i][j] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
  const int wrow0 = wm * Cfg::TM, wcol0 = wn * Cfg::TN;
  const int blocks = min(FM, (live - row0 - wrow0 + 15) >> 4);     // live 16-row blocks of the wave
  auto multiply = [&]() {
    constexpr int kCols = BK / 32 * FN;
    bf16x8 fa[3][FM], fb[2][3];
    auto read_a = [&](const int ks) {
#pragma unroll
      for (int i = 0; i < FM; ++i) {
        const int r = wrow0 + i * 16 + r16;
        const uint32_t at = r * Cfg::kRowBytes + (((ks * 4 + q) ^ ((r >> 1) & Cfg::kSwz)) << 4);
#pragma unroll
        for (int t = 0; t < 3; ++t) fa[t][i] = *reinterpret_cast<const bf16x8*>(piece + t * Cfg::kAPlane + at);
      }
    };
    auto read_b = [&](const int c) {
      const int ks = c / FN, j = c % FN, r = wcol0 + j * 16 + r16;
      const uint32_t at = 3 * Cfg::kAPlane + r * Cfg::kRowBytes + (((ks * 4 + q) ^ ((r >> 1) & Cfg::kSwz)) << 4);
#pragma unroll
      for (int t = 0; t < 3; ++t) fb[c & 1][t] = *reinterpret_cast<const bf16x8*>(piece + t * Cfg::kBPlane + at);
    };
    read_b(0);
#pragma unroll
    for (int c = 0; c < kCols; ++c) {
      const int j = c % FN;
      if (j == 0) read_a(c / FN);
      if (c + 1 < kCols) read_b(c + 1);
      constexpr int ta[6] = {2, 0, 1, 1, 0, 0}, tb[6] = {0, 2, 1, 0, 1, 0};
#pragma unroll
      for (int t = 0; t < 6; ++t)
#pragma unroll
        for (int i = 0; i < FM; ++i)
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fa[ta[t]][i], fb[c & 1][tb[t]], acc[i][j], 0, 0, 0);
    }
  };

  // A group's k tiles are consecutive; where they do not divide evenly the last group's run past
  // the end, where fetch() finds zeros.
  const int nk = ((Kd + BK - 1) / BK + Cfg::KG - 1) / Cfg::KG, kt0 = group * nk;
  // Turns: between two barriers every other group splits and the rest multiply.  (In step, all of a SIMD's waves want
  // its vector instructions first and its matrix core then: 8 x 392 rows x 2 048 x 512 on 64 x 128 tiles and two
  // groups 61 -> 54 us.  The smaller two-group tiles, four workgroups of which share a CU, lose 0 - 7 %; tiles
  // without groups fall out of step by themselves, and lost as two tiles of one workgroup: 50 -> 53, 235 -> 252.)
  fetch(kt0);
  if (Cfg::kTurns && (group & 1)) raw_barrier();
  for (int s = 0; s < nk; ++s) {
    if (!Cfg::kTurns && s > 0) raw_barrier();      // every wave has read the k tile before
    __builtin_amdgcn_s_setprio(2);
#pragma unroll
    for (int u = 0; u < kUnits; ++u) stage_unit(u);
    if (s + 1 < nk) fetch(kt0 + s + 1);
    wait_lgkmcnt0();
    __builtin_amdgcn_s_setprio(0);
    raw_barrier();
    if (blocks > 0) multiply();
    if (Cfg::kTurns) raw_barrier();
  }
  if (Cfg::kTurns && !(group & 1)) raw_barrier();
  mfma_result_fence();
  if (!Cfg::kTurns) raw_barrier();               // the operands' LDS is free
  if constexpr (Cfg::KG > 1) {
    f32x4_t* sums = reinterpret_cast<f32x4_t*>(piece);
    if (group > 0) {
#pragma unroll
      for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j) sums[(i * FN + j) * Cfg::kGroup + tid] = acc[i][j];
    }
    wait_lgkmcnt0();
    raw_barrier();
    if (group > 0) return;
#pragma unroll 1
    for (int g = 1; g < Cfg::KG; ++g)
#pragma unroll
      for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j)
          acc[i][j] += reinterpret_cast<const f32x4_t*>(smem + g * Cfg::kPiece)[(i * FN + j) * Cfg::kGroup + tid];
  }

  // Epilogue, 16 rows at a time through a wave-private piece of LDS.
  float* st = reinterpret_cast<float*>(smem) + wave * 16 * Cfg::kOutStride;
  constexpr int LPR = Cfg::TN / 4, RPI = 64 / LPR;    // lanes per row, rows per instruction
  const int ocol = col0 + wcol0 + (lane % LPR) * 4, orow = lane / LPR;
  const bool col_ok = ocol < N;
  f32x4_t bv = {0.f, 0.f, 0.f, 0.f};
  if (bias != nullptr && col_ok) {
#pragma unroll
    for (int t = 0; t < 4; ++t) bv[t] = bias[(size_t)b * N + ocol + t];
  }
  float* Cb = C + (size_t)b * R * N;
#pragma unroll
  for (int i = 0; i < FM; ++i) {
    if (i >= blocks) break;
#pragma unroll
    for (int j = 0; j < FN; ++j) {
      const int p = j * 16 + r16;
      const int n = (p & ~31) + (p & 7) * 4 + ((p >> 3) & 3);
#pragma unroll
      for (int v = 0; v < 4; ++v) st[(q * 4 + v) * Cfg::kOutStride + n] = acc[i][j][v];
    }
    wait_lgkmcnt0();
#pragma unroll
    for (int s = 0; s < 16 / RPI; ++s) {
      const int row = row0 + wrow0 + i * 16 + s * RPI + orow;
      f32x4_t o = *reinterpret_cast<const f32x4_t*>(st + (s * RPI + orow) * Cfg::kOutStride + (lane % LPR) * 4);
      if (row < live && col_ok) {
        const float chk = (o[0] - o[0]) + (o[1] - o[1]) + (o[2] - o[2]) + (o[3] - o[3]);
        if (__builtin_expect(!(chk == 0.f), 0)) {
          const float* ap = A + ((size_t)b * R + row) * Kd;
          if (a_rows != nullptr) {
            const int item = a_rows[(size_t)b * R + row];
            ap = A + (size_t)((unsigned)item < (unsigned)a_items ? item : 0) * Kd;
          }
          f32x4_t s4 = {0.f, 0.f, 0.f, 0.f};
          for (int k = 0; k < Kd; ++k) {
            const f32x4_t bk = *reinterpret_cast<const f32x4_any_t*>(Bb + (size_t)k * N + ocol);
            const float av = ap[k];
#pragma unroll
            for (int t = 0; t < 4; ++t) s4[t] = fmaf(av, bk[t], s4[t]);
          }
#pragma unroll
          for (int t = 0; t < 4; ++t)
            if (!(o[t] - o[t] == 0.f)) o[t] = s4[t];
        }
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          o[t] += bv[t];
          if (EPI == kEpiBiasGeluTanh) o[t] = gelu_tanh_fast(o[t]);
          if (EPI == kEpiBiasGeluTanhf) o[t] = gelu_tanh(o[t]);
          if (EPI == kEpiBiasGeluErf) o[t] = gelu_erf(o[t]);
        }
        *reinterpret_cast<f32x4_t*>(Cb + (size_t)row * N + ocol) = o;
      }
    }
    wait_lgkmcnt0();
  }
}

template <int EPI, typename Cfg>
int launch_gemm_f32_split_tile(const float* A, const float* B, const float* bias, float* C, int batch,
                               int R, int N, int Kd, hipStream_t stream, const int32_t* rows,
                               const int32_t* a_rows, int a_items) {
  const int tiles_m = (R + Cfg::BM - 1) / Cfg::BM, tiles_n = (N + Cfg::BN - 1) / Cfg::BN;
  const long long total = (long long)batch * tiles_m * tiles_n;
  if (total > 0x0fffffffLL) return VMOE_E_OVERFLOW;
  auto kern = gemm_f32_split_kernel<EPI, Cfg>;
  hipError_t e = allow_dynamic_lds(reinterpret_cast<const void*>(kern), Cfg::kLds);
  if (e != hipSuccess) return (int)e;
  hipLaunchKernelGGL(kern, dim3((unsigned)((total + 7) / 8 * 8)), dim3(Cfg::kThreads), Cfg::kLds, stream, A, B,
                     bias, C, batch, R, N, Kd, tiles_n, rows, a_rows, a_items);
  return launch_status();
}

// Tiles, with what they cost: a 32-wide step of k takes `work` us of a CU's time per tile, `latency` us alone on a
// CU, a tile `fix` us besides.  A launch is taken to last the 4-norm of one tile's chain and the fullest CU's work.
// Tiles per CU count as halfway between whole ones and even ones; four groups along k fill a CU, and are for launches
// of a tile per CU at most (with two rounds of them the others win, and constants fitted to both miss by 12 %).
// How many of the R rows are live stands on the device, and a dense call keeps the order of sums of a ragged
// one of its shape, so the tile may not depend on it.  Tiles whose groups take turns are taken where they are 5 %
// ahead of the best of the others for all rows and for 35 % of them together: their time is the chain's, which fewer
// rows do not shorten (18 experts of up to 88 rows, 393 in all, 2560 to 640: 53 us on four groups, 37 on 32 x 64).
// Fitted to 90 random shapes (1 - 64 experts, 16 - 9 000 rows, widths 192 - 4 096), every tile on both products, rms
// 6 - 10 % per tile; chosen on them and on 80 ragged ones, a quarter to all of their rows live.  Before groups took
// turns and before there were four of them the 180 products with all rows took 12 827 us and take 12 385 (5 % in the
// geometric mean; 11 792 on the best tile of each), the 160 ragged ones 12 620 and 12 177 (4 %; 11 030).
struct SplitTile {
  int bm, bn;
  double work, latency, fix;
  bool turns, fills_cu;
};
constexpr SplitTile kSplitTiles[] = {
    {128, 128, 1.09, 1.61, 2.7, false, false},   // two workgroups per CU
    {64, 128, 0.59, 1.14, 2.0, false, false},    // four
    {64, 128, 0.68, 0.47, 2.0, true, false},     // two groups of waves along k
    {32, 128, 0.42, 0.88, 1.0, false, false},
    {32, 128, 0.42, 0.57, 1.6, false, false},    // two groups
    {32, 64, 0.25, 0.29, 1.0, false, false},     // two groups
    {96, 128, 0.77, 1.39, 3.7, false, false},    // two workgroups per CU
    {64, 128, 0.48, 0.49, 4.1, true, true},      // four groups
    {32, 64, 0.10, 0.28, 1.6, true, true},       // four groups
};
constexpr int kNumSplitTiles = sizeof(kSplitTiles) / sizeof(kSplitTiles[0]);

inline int best_split_tile(int batch, int R, int N, int Kd) {
  const double steps = (Kd + 31) / 32;
  auto tiles_per_cu = [&](const SplitTile& t, int rows) {
    return (double)batch * ((rows + t.bm - 1) / t.bm) * ((N + t.bn - 1) / t.bn) / (kCusPerXcd * kNumXcd);
  };
  auto time = [&](const SplitTile& t, int rows) {
    const double per_cu = tiles_per_cu(t, rows);
    const double tiles = t.fills_cu ? 1.0 : std::max(1.0, 0.5 * (std::ceil(per_cu) + per_cu + 0.3));
    const double chain = steps * t.latency, busy = tiles * (steps * t.work + t.fix);
    return std::sqrt(std::sqrt(chain * chain * chain * chain + busy * busy * busy * busy));
  };
  int best = 0;
  double best_us = 1e30;
  for (int i = 0; i < kNumSplitTiles; ++i) {
    if (kSplitTiles[i].turns) continue;
    const double us = time(kSplitTiles[i], R);
    if (us < best_us) { best_us = us; best = i; }
  }
  const int few_rows = std::max(1, (int)(0.35 * R));
  best_us = 0.95 * (best_us + time(kSplitTiles[best], few_rows));
  for (int i = 0; i < kNumSplitTiles; ++i) {
    const SplitTile& t = kSplitTiles[i];
    if (!t.turns || (t.fills_cu && tiles_per_cu(t, R) > 1)) continue;
    const double us = time(t, R) + time(t, few_rows);
    if (us < best_us) { best_us = us; best = i; }
  }
  return best;
}

template <int EPI>
int launch_gemm_f32_split(int tile, const float* A, const float* B, const float* bias, float* C, int batch,
                          int R, int N, int Kd, hipStream_t stream, const int32_t* rows,
                          const int32_t* a_rows, int a_items) {
  auto run = [&](auto cfg) {
    return launch_gemm_f32_split_tile<EPI, decltype(cfg)>(A, B, bias, C, batch, R, N, Kd, stream, rows, a_rows, a_items);
  };
  switch (tile) {
    case 0: return run(SplitCfg<128, 128, 2, 2, 32, 2, 1>{});
    case 1: return run(SplitCfg<64, 128, 2, 2, 32, 4, 1>{});
    case 2: return run(SplitCfg<64, 128, 2, 2, 32, 2, 2>{});
    case 3: return run(SplitCfg<32, 128, 1, 4, 32, 4, 1>{});
    case 4: return run(SplitCfg<32, 128, 1, 4, 32, 2, 2>{});
    case 5: return run(SplitCfg<32, 64, 2, 2, 64, 2, 2>{});
    case 7: return run(SplitCfg<64, 128, 2, 2, 32, 1, 4>{});
    case 8: return run(SplitCfg<32, 64, 2, 2, 64, 1, 4>{});
    default: return run(SplitCfg<96, 128, 2, 2, 32, 2, 1>{});
  }
}

}  // namespace vmoe
