// bf16 expert products of a few hundred to a few thousand rows: C[b] (R x N) = epi(A[b] (R x Kd) . Bt[b]^T + bias[b]).
//
// What bounds them.  A launch of this size is one or two rounds of tiles: its time is a start (launch, row
// numbers, the first k tiles' trip to memory: 4 - 5 us), the chain of k tiles of one CU's tiles, and an
// epilogue.  Inside the chain a 128 x 128 x 64 step takes 0.46 - 0.6 us where its MFMAs take 0.21: fragment reads
// and DMA writes share the LDS (96 KB of its 128 bytes a clock), and every step ends in a barrier.  So what pays
// is a tile that makes whole rounds of the 256 CUs, more than one wave per SIMD (two workgroups per CU, or
// eight waves in one: 27 us where four waves on 128 x 128 took 36 over 1 568 rows x 768 x 3072), and a chain in
// which the fragment reads of one half of a k tile run under the MFMAs of the other.
//
// Operands go global memory -> LDS by DMA, 8 rows x 128 bytes per request, into a ring of S stages of 64 KT k,
// XOR-swizzled as in gemm_bf16_rows.h.  The output leaves straight from registers (v_permlane16_swap, as in
// gemm_bf16_stream.h).  Tiles are dealt to the dies: dense launches as eight runs of one list, which come out even;
// ragged ones from a launch plan (whole row tiles to a die) or, over less than two row tiles per die or many (batch,
// column tile) pairs, those pairs round the dies.  Sums run over k in the order of the other bfloat16 kernels: same bits.
#ifndef VMOE_GEMM_BF16_MID_H_
#define VMOE_GEMM_BF16_MID_H_
#include "gemm_bf16.h"

namespace vmoe {

template <int BM_, int BN_, int WM_, int WN_, int STAGES_, int PER_CU_, int KT_>
struct MidCfg {
  static constexpr int BM = BM_, BN = BN_, WM = WM_, WN = WN_, S = STAGES_, KT = KT_, BK = 64 * KT;
  static constexpr int kBlocksPerCu = PER_CU_;
  static constexpr int kWaves = WM * WN, kThreads = 64 * kWaves;
  static constexpr int TM = BM / WM, TN = BN / WN;             // wave tile
  static constexpr int FM = TM / 16, FN = TN / 16;
  static constexpr int kABytes = BM * 128, kHalfBytes = (BM + BN) * 128;    // 64 k of the rows, of both operands
  static constexpr int kStageBytes = KT * kHalfBytes;
  static constexpr int LA = BM / 8 / kWaves, LB = BN / 8 / kWaves;
  static constexpr int kIssues = KT * (LA + LB);               // DMA requests per wave and stage
  static constexpr size_t kLdsBytes = (size_t)S * kStageBytes;
  static_assert(BM % (8 * kWaves) == 0 && BN % (8 * kWaves) == 0 && kWaves % 2 == 0, "whole requests per wave");
  static_assert(TM % 16 == 0 && FN % 2 == 0, "column blocks leave in pairs");
  static_assert(S >= 2 && S * kIssues < 64, "vmcnt is a 6-bit counter");
  static_assert(kLdsBytes * PER_CU_ <= 160 * 1024, "LDS budget");
};

// Whether the kernel takes the operands: whole 16-byte pieces, 31-bit byte offsets inside a batch.
inline bool mid_gemm_ok(int batch, int R, int N, int Kd, long long items) {
  const uint64_t lim = 1ull << 31;
  return N % 8 == 0 && Kd % 8 == 0 && (uint64_t)R * Kd * 2 < lim && (uint64_t)N * Kd * 2 < lim &&
         (uint64_t)R * N * 2 < lim && (uint64_t)items * Kd * 2 < lim &&
         (uint64_t)batch * ((R + 63) / 64) * ((N + 63) / 64) < 0x7ffff000ull;
}

// `plan_ref`: the launch's own plan, or none.  `guard`: the plan of the other product of the call, where that one
// has a plan: a launch whose plan was not written for this geometry runs nothing, and neither does this one.
// per_die: tiles of a die (dense launches without a plan); 0: pairs go round the dies.
template <typename Cfg, int EPI>
__global__ __launch_bounds__(Cfg::kThreads, Cfg::kBlocksPerCu * Cfg::kWaves / 4) void gemm_bf16_mid_kernel(
    const bf16_t* __restrict__ A, const bf16_t* __restrict__ Bt, const bf16_t* __restrict__ bias,
    bf16_t* __restrict__ C, int R, int N, int Kd, int tiles_m, int tiles_n, int batch, int per_die,
    const int32_t* __restrict__ rows, PlanRef plan_ref, const int32_t* __restrict__ a_rows, int a_items,
    PlanRef guard, int32_t* __restrict__ clear, int clear_count, int32_t* __restrict__ status) {
#if defined(__HIP_DEVICE_COMPILE__)
  constexpr int FM = Cfg::FM, FN = Cfg::FN, S = Cfg::S, L = Cfg::kIssues, W = Cfg::kWaves, H = 2 * Cfg::KT;
  extern __shared__ __align__(1024) unsigned char smem[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / Cfg::WN, wn = wave % Cfg::WN;
  if (blockIdx.x == 0) begin_call(clear, clear_count, status, tid, Cfg::kThreads);
  if (guard.entries != nullptr && guard.entries[guard.blocks].y != guard.tag) {
    if (blockIdx.x == 0 && tid == 0 && status != nullptr) status[kStatusPlanMismatches] += 1;
    return;
  }
  int b, tile_m, tile_n, live = R;
  if (plan_ref.entries != nullptr) {
    int4 mine;
    if (!read_plan(plan_ref, status, tid, mine)) return;
    if (mine.x < 0) return;
    b = mine.x;
    tile_m = mine.y;
    tile_n = mine.z;
    live = mine.w;
  } else {
    const int xcd = blockIdx.x % kNumXcd, idx = blockIdx.x / kNumXcd;
    int pair;
    if (per_die > 0) {
      const int tile = xcd * per_die + idx;
      pair = tile / tiles_m;
      tile_m = tile - pair * tiles_m;
    } else {
      pair = idx / tiles_m * kNumXcd + xcd;
      tile_m = idx % tiles_m;
    }
    if (pair >= batch * tiles_n) return;
    b = pair / tiles_n;
    tile_n = pair - b * tiles_n;
    if (rows != nullptr) {
      live = min(rows[b], R);
      if (tile_m * Cfg::BM >= live) return;
    }
  }
  const int row0 = tile_m * Cfg::BM, col0 = tile_n * Cfg::BN;
  // Requests: lane l of a request fetches a 16-byte piece of row l / 8; the piece is the one
  // that the XOR swizzle (row / 2) % 8 puts at position l % 8 of the row in LDS.
  const int lrow = lane >> 3;
  const int piece = (lane & 7) ^ ((wave * 4 + (lrow >> 1)) & 7);
  uint32_t a_off[Cfg::LA], b_off[Cfg::LB];
#pragma unroll
  for (int i = 0; i < Cfg::LB; ++i)
    b_off[i] = (uint32_t)min(col0 + (i * W + wave) * 8 + lrow, N - 1) * (uint32_t)Kd * 2u + piece * 16u;
#pragma unroll
  for (int i = 0; i < Cfg::LA; ++i) {
    int r = min(row0 + (i * W + wave) * 8 + lrow, live - 1);
    if (a_rows != nullptr) {
      r = a_rows[(size_t)b * R + r];
      r = (unsigned)r < (unsigned)a_items ? r : 0;
    }
    a_off[i] = (uint32_t)r * (uint32_t)Kd * 2u + piece * 16u;
  }
  auto uniform = [](bf16_t* p) {                 // (the same in every lane; said explicitly)
    const uint64_t bits = reinterpret_cast<uint64_t>(p);
    return reinterpret_cast<bf16_t*>(
        ((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(bits >> 32)) << 32) |
        (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)bits));
  };
  // Addresses past an operand's end (k past Kd in its last row) read as zero, as long as the scalar
  // offset itself lies inside the operand.  A second half of the last stage may start past Kd, which one row
  // (or a few short ones) may all be: it takes the row's first half again, and its fragments are
  // cleared like every k past Kd.
  const bf16_t* Ab = a_rows != nullptr ? A : A + (size_t)b * R * Kd;
  const uint32_t a_bytes = (uint32_t)(a_rows != nullptr ? a_items : R) * (uint32_t)Kd * 2u;
  const __amdgpu_buffer_rsrc_t a_rsrc =
      __builtin_amdgcn_make_buffer_rsrc(uniform(const_cast<bf16_t*>(Ab)), 0, (int)a_bytes, 0x00020000);
  const __amdgpu_buffer_rsrc_t b_rsrc = __builtin_amdgcn_make_buffer_rsrc(
      uniform(const_cast<bf16_t*>(Bt + (size_t)b * N * Kd)), 0, (int)((uint32_t)N * (uint32_t)Kd * 2u), 0x00020000);
  auto request = [&](int slot, int kt) {
#pragma unroll
    for (int h = 0; h < Cfg::KT; ++h) {
      unsigned char* s = smem + slot * Cfg::kStageBytes + h * Cfg::kHalfBytes;
      const int half = kt * Cfg::KT + h, k_bytes = Cfg::KT == 1 || half * 64 < Kd ? half * 128 : 0;
#pragma unroll
      for (int i = 0; i < Cfg::LB; ++i)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(
            b_rsrc, (lds_ptr_t)(s + Cfg::kABytes + (i * W + wave) * 1024), 16, b_off[i], k_bytes, 0, 0);
#pragma unroll
      for (int i = 0; i < Cfg::LA; ++i)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(a_rsrc, (lds_ptr_t)(s + (i * W + wave) * 1024), 16, a_off[i],
                                                 k_bytes, 0, 0);
    }
  };

  const int r16 = lane & 15, q = lane >> 4;
  uint2 bias_pk[FN];
#pragma unroll
  for (int j = 0; j < FN; ++j) {
    bias_pk[j] = make_uint2(0x80008000u, 0x80008000u);     // no bias: x + -0 is x, -0 among them
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
  const uint32_t b_row = lds0 + Cfg::kABytes + (wn * Cfg::TN + r16) * 128;
  const uint32_t pos[2] = {(uint32_t)((q ^ (r16 >> 1)) * 16), (uint32_t)(((4 + q) ^ (r16 >> 1)) * 16)};
  frag_t fa[2][FM], fb[2][FN];         // of two consecutive 32-wide parts of a stage
  auto read_frags = [&](const int h, int slot) {
    const uint32_t at = slot * Cfg::kStageBytes + (h >> 1) * Cfg::kHalfBytes + pos[h & 1];
#pragma unroll
    for (int j = 0; j < FN; ++j)
      asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(fb[h & 1][j]) : "v"(b_row + at), "n"(j * 2048));
#pragma unroll
    for (int i = 0; i < FM; ++i)
      asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(fa[h & 1][i]) : "v"(a_row + at), "n"(i * 2048));
  };
  const int nk = (Kd + Cfg::BK - 1) / Cfg::BK;
  auto arrived = [&](const int h, int t) {
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
    for (int j = 0; j < FN; ++j) asm volatile("" : "+v"(fb[h & 1][j]));
#pragma unroll
    for (int i = 0; i < FM; ++i) asm volatile("" : "+v"(fa[h & 1][i]));
    if (Kd % Cfg::BK != 0 && t + 1 == nk && t * Cfg::BK + h * 32 + q * 8 >= Kd) {   // k past Kd counts as zero
#pragma unroll
      for (int j = 0; j < FN; ++j) fb[h & 1][j] = frag_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int i = 0; i < FM; ++i) fa[h & 1][i] = frag_t{0.f, 0.f, 0.f, 0.f};
    }
  };
  auto multiply = [&](const int u) {
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
      for (int j = 0; j < FN; ++j)
        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
            __builtin_bit_cast(bf16x8, fb[u][j]), __builtin_bit_cast(bf16x8, fa[u][i]), acc[i][j], 0, 0, 0);
  };
  // Step t: the fragment reads of every part of stage t but its first run under the MFMAs of the part before.
  // With the last part's fragments here, the wave's requests of t + 1 have landed; barrier (everyone's
  // have, and everyone has read stage t); requests of t + S into that stage; fragment reads of t + 1.
  int slot = 0;
  auto step = [&](int t) {
    const int next = slot + 1 == S ? 0 : slot + 1;
#pragma unroll
    for (int h = 0; h < H; ++h) {
      arrived(h, t);
      if (h + 1 < H) {
        read_frags(h + 1, slot);
      } else if (t + 1 < nk) {
        if (nk - 2 - t >= S - 2) wait_vmcnt<(S - 2) * L>();     // stages requested behind t + 1
        else wait_vmcnt<0>();
        raw_barrier();
        if (t + S < nk) request(slot, t + S);
        read_frags(0, next);
      }
      multiply(h & 1);
    }
    slot = next;
  };
  static_for<S>([&](auto s) {
    if (s < nk) request(s, s);
  });
  if (nk >= S) wait_vmcnt<(S - 1) * L>();
  else wait_vmcnt<0>();
  raw_barrier();
  read_frags(0, 0);
  for (int t = 0; t < nk; ++t) step(t);
  mfma_result_fence();

  // acc[i][j][v] = C[row i * 16 + lane % 16][column j * 16 + (lane / 16) * 4 + v].  Column blocks leave in
  // pairs, eight consecutive columns of a row per lane; rows and columns past the edge leave through the
  // range check.
  const __amdgpu_buffer_rsrc_t c_rsrc =
      __builtin_amdgcn_make_buffer_rsrc(uniform(C + (size_t)b * R * N), 0, R * N * 2, 0x00020000);
  const int wrow0 = row0 + wm * Cfg::TM, wcol0 = col0 + wn * Cfg::TN;
  const int lane_col = (q & 1) * 16 + (q >> 1) * 8;       // inside a pair of column blocks
  const uint32_t lane_off = (uint32_t)(r16 * N + lane_col) * 2u;
  typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
#pragma unroll
  for (int jp = 0; jp < FN / 2; ++jp)
#pragma unroll
    for (int i = 0; i < FM; ++i) {
      uint32_t p[2][2];
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        const int j = 2 * jp + t;
        p[t][0] = epilogue_pair<EPI, true>(acc[i][j][0], acc[i][j][1], bf_lo(bias_pk[j].x), bf_hi(bias_pk[j].x));
        p[t][1] = epilogue_pair<EPI, true>(acc[i][j][2], acc[i][j][3], bf_lo(bias_pk[j].y), bf_hi(bias_pk[j].y));
      }
      const auto x = __builtin_amdgcn_permlane16_swap(p[0][0], p[1][0], false, false);
      const auto y = __builtin_amdgcn_permlane16_swap(p[0][1], p[1][1], false, false);
      const u32x4_t v = {x[0], y[0], x[1], y[1]};
      const int col_s = wcol0 + jp * 32;
      const bool ok = r16 < live - (wrow0 + i * 16) && lane_col + 8 <= N - col_s;
      const uint32_t at = lane_off + (uint32_t)((wrow0 + i * 16) * N + col_s) * 2u;
      __builtin_amdgcn_raw_buffer_store_b128(v, c_rsrc, ok ? at : 0x80000000u, 0, 0);
      store_data_guard();
    }
#endif
}

// `plan`, if given, was written for tile_geometry(Cfg::BM, Cfg::BN, Cfg::kBlocksPerCu, ...).
template <typename Cfg, int EPI>
int launch_mid_tile(const bf16_t* A, const bf16_t* Bt, const bf16_t* bias, bf16_t* C, int batch, int R, int N,
                    int Kd, hipStream_t stream, const int32_t* rows, const int4* plan, const int32_t* a_rows,
                    int a_items, PlanRef guard, int32_t* clear, int clear_count, int32_t* status) {
  const GemmGeom g = tile_geometry(Cfg::BM, Cfg::BN, Cfg::kBlocksPerCu, batch, R, N);
  const int per_die = rows == nullptr ? g.tiles_per_xcd : 0;
  const long long pairs = (long long)batch * g.tiles_n;
  const long long blocks = kNumXcd * (plan != nullptr ? g.ragged_slots
                                      : per_die > 0   ? g.tiles_per_xcd
                                                      : (pairs + kNumXcd - 1) / kNumXcd * g.tiles_m);
  if (blocks > 0x7fffffffLL || g.tiles > 0x7ffffff0LL) return VMOE_E_OVERFLOW;
  auto kern = gemm_bf16_mid_kernel<Cfg, EPI>;
  hipError_t e = allow_dynamic_lds(reinterpret_cast<const void*>(kern), Cfg::kLdsBytes);
  if (e != hipSuccess) return (int)e;
  hipLaunchKernelGGL(kern, dim3((unsigned)blocks), dim3(Cfg::kThreads), Cfg::kLdsBytes, stream, A, Bt, bias, C, R,
                     N, Kd, g.tiles_m, g.tiles_n, batch, per_die, rows, plan_ref_of(g, plan, Cfg::BM, batch, R),
                     a_rows, a_items, guard, clear, clear_count, status);
  return launch_status();
}

}  // namespace vmoe
#endif  // VMOE_GEMM_BF16_MID_H_
