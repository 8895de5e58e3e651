// bf16 expert products over at most BM rows per batch, where the weights are what has to be moved:
//   C[b] (R x N) = epi(A[b] (R x Kd) . Bt[b]^T + bias[b]),  R <= BM.
//
// What bounds them.  Every weight is multiplied with one tile of rows, so a product cannot be done before
// its weights have come from memory, and a load-only kernel of the same requests moves 151 MB in 25 us
// and 604 MB in 88 (6.1 and 6.8 TB/s, 32 KB per CU on their way are enough).  The kernels with a workgroup per
// tile took 41 and 145 - 152: a workgroup starts with empty hands (its plan or row list, then the first k
// tiles: two trips to memory), and leaves the CU without requests again while it rounds, applies the
// GELU and stores.
//
// One workgroup of eight waves per CU walks a run of (batch, column tile) units: a die takes a
// contiguous part of them, its 32 CUs neighbouring units, so that a batch's rows are read through one L2.
// Operands go global memory -> LDS by DMA, 8 rows x 128 bytes per request, XOR-swizzled as in gemm_bf16_rows.h.
// Rows and weights have rings of their own, of SA and SB stages of 64 k, and waves that fill them (a
// wave's requests complete in order: one that asked for both would wait for its weights whenever it
// waits for rows).  The rings are never drained: the last steps of a tile request the next tile's first stages,
// which are on their way while the epilogue runs.  Whatever would make a wave wait for all its requests in
// between is fetched as part of the same stream: the bias of the tile and the row numbers of the next one go
// to LDS by DMA a tile ahead, and the output leaves straight from registers (v_permlane16_swap, as in
// gemm_bf16_w8.h), its stores counted by the waits that follow.  Weights are read once and leave no copy
// in the caches (non-temporal requests: 133 us without, 123 with).  The hidden layer leaves the same way
// (the second product of 64 experts x 64 rows: 65 us behind cached stores, 54 - 57 behind these).
//
// Measured (768 x 3072, first and second product): 128 experts x 128 rows 149 + 143 -> 142 + 123 us, 64 x 64:
// 62 + 74 -> 59 + 53, 32 x 100: 42 + 44 -> 37 + 39.  Rows that hit L2 and weights that miss it add up: 402 MB
// at 26 TB/s and 604 MB at 6.2 are 113 us of the 123 (128 x 192 tiles; the first product writes 100 MB
// beside its 604, which is copy rate with or without its GELU), so wide tiles win where they
// fill the chip's rounds; deeper rings do not (128 x 128: 135 us with four stages, 137 with six of the weights).
#ifndef VMOE_GEMM_BF16_STREAM_H_
#define VMOE_GEMM_BF16_STREAM_H_
#include "gemm_bf16.h"

namespace vmoe {

template <int BM_, int BN_, int WM_, int WN_, int SA_, int SB_>
struct StreamCfg {
  static constexpr int BM = BM_, BN = BN_, WM = WM_, WN = WN_, SA = SA_, SB = SB_;
  static constexpr int kWaves = 8, kThreads = 512;
  static constexpr int TM = BM / WM, TN = BN / WN;             // wave tile
  static constexpr int FM = TM / 16, FN = TN / 16;
  static constexpr int kABytes = BM * 128, kBBytes = BN * 128; // 64 k of either operand
  static constexpr int LA = BM / 32, LB = BN / 32;             // DMA requests per stage of a wave of either half
  static constexpr int kStores = FM * FN / 2;                  // per wave and tile
  static constexpr int kMaxBatch = 1024;                       // counts of a ragged launch in LDS
  static constexpr int kBAt = SA * kABytes;
  static constexpr int kBiasAt = kBAt + SB * kBBytes;          // per wave: 256 bytes of the tile's bias ...
  static constexpr int kIndexAt = kBiasAt + kWaves * 256;      // ... and 64 row numbers of the next tile's rows
  static constexpr int kRowsAt = kIndexAt + kWaves / 2 * 256;
  static constexpr size_t kLdsBytes = kRowsAt + kMaxBatch * 2;
  static_assert(WM * WN == kWaves && BM % 32 == 0 && BN % 32 == 0 && LA <= 8, "whole requests per wave");
  static_assert(FN % 2 == 0 && TN <= 128, "column blocks leave in pairs; one bias request per wave");
  static_assert(SA >= 3 && SB >= 3 && SA <= SB && SB * LB + kStores < 64, "vmcnt is a 6-bit counter");
  static_assert(BM <= 0xffff && kLdsBytes <= 160 * 1024, "LDS budget; counts of 16 bits");
};

// Whether the kernel takes the product: k tiles enough that what is requested at a tile's start has landed
// before it is used S stages ahead of the tile's end.
template <typename Cfg>
inline bool stream_gemm_ok(int batch, int R, int Kd, bool ragged) {
  return R <= Cfg::BM && (Kd + 63) / 64 >= 2 * Cfg::SB - 2 && (!ragged || batch <= Cfg::kMaxBatch);
}

// The operands' conditions are those of gemm_bf16_rows_kernel (rows_gemm_ok), `guard` as there.
template <typename Cfg, int EPI>
__global__ __launch_bounds__(512, 1) void gemm_bf16_stream_kernel(
    const bf16_t* __restrict__ A, const bf16_t* __restrict__ Bt, const bf16_t* __restrict__ bias,
    bf16_t* __restrict__ C, int R, int N, int Kd, int tiles_n, int units, int units_per_die, int batch,
    const int32_t* __restrict__ rows, const int32_t* __restrict__ a_rows, int a_items,
    PlanRef guard, int32_t* __restrict__ clear, int clear_count, int32_t* __restrict__ status) {
#if defined(__HIP_DEVICE_COMPILE__)
  constexpr int FM = Cfg::FM, FN = Cfg::FN, SA = Cfg::SA, SB = Cfg::SB, LA = Cfg::LA, LB = Cfg::LB;
  extern __shared__ __align__(1024) unsigned char smem[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / Cfg::WN, wn = wave % Cfg::WN;
  if (blockIdx.x == 0) begin_call(clear, clear_count, status, tid, Cfg::kThreads);
  if (guard.entries != nullptr && guard.entries[guard.blocks].y != guard.tag) {
    if (blockIdx.x == 0 && tid == 0 && status != nullptr) status[kStatusPlanMismatches] += 1;
    return;
  }
  // LDS is read by instruction: a read that the compiler can see waits for every request in flight.
  const uint32_t lds0 = (uint32_t)reinterpret_cast<uintptr_t>((lds_ptr_t)smem);
  auto lds_u16 = [&](uint32_t at) {
    uint32_t v;
    asm volatile("ds_read_u16 %0, %1\n\ts_waitcnt lgkmcnt(0)" : "=v"(v) : "v"(lds0 + at) : "memory");
    return (int)v;
  };
  auto lds_i32 = [&](uint32_t at) {
    int v;
    asm volatile("ds_read_b32 %0, %1\n\ts_waitcnt lgkmcnt(0)" : "=v"(v) : "v"(lds0 + at) : "memory");
    return v;
  };
  if (rows != nullptr) {
    uint16_t* s_rows = reinterpret_cast<uint16_t*>(smem + Cfg::kRowsAt);
    for (int i = tid; i < batch; i += Cfg::kThreads) s_rows[i] = (uint16_t)max(0, min(rows[i], R));
    __syncthreads();
  }
  // Units xcd * units_per_die + slot, + 32, ...: tiles of batches without rows are passed over.
  struct Tile {
    int b, col0, live;
  };
  const int xcd = blockIdx.x % kNumXcd;
  const int die_end = min(units, (xcd + 1) * units_per_die);
  int unit = xcd * units_per_die + blockIdx.x / kNumXcd;
  auto next_tile = [&](Tile& t) -> bool {
    for (; unit < die_end; unit += kCusPerXcd) {
      t.b = unit / tiles_n;
      t.col0 = (unit - t.b * tiles_n) * Cfg::BN;
      t.live = rows != nullptr ? __builtin_amdgcn_readfirstlane(lds_u16(Cfg::kRowsAt + t.b * 2)) : R;
      if (t.live > 0) {
        unit += kCusPerXcd;
        return true;
      }
    }
    return false;
  };
  Tile cur, nxt;
  if (!next_tile(cur)) return;

  // Requests: waves 0 - 3 ask for the rows, 4 - 7 for the weights.  Lane l of a request fetches a 16-byte piece
  // of row l / 8; the piece is the one that the XOR swizzle (row / 2) % 8 puts at position l % 8 of the
  // row in LDS.
  const bool b_wave = wave >= 4;
  const int w4 = wave & 3;
  const int lrow = lane >> 3;
  const int piece = (lane & 7) ^ ((w4 * 4 + (lrow >> 1)) & 7);
  uint32_t off[LA > LB ? LA : LB];
  __amdgpu_buffer_rsrc_t rsrc;
  auto uniform = [](const bf16_t* p) {
    const uint64_t bits = reinterpret_cast<uint64_t>(p);
    return reinterpret_cast<bf16_t*>(
        ((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(bits >> 32)) << 32) |
        (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)bits));
  };
  const uint32_t src_bytes = (uint32_t)(b_wave ? N : a_rows != nullptr ? a_items : R) * (uint32_t)Kd * 2u;
  // Row of request i: past the live rows the last of them again.
  auto row_of = [&](const Tile& t, int i, int l) { return min((i * 4 + w4) * 8 + l, t.live - 1); };
  // Turns the wave's request stream to a tile; index(i): the row of the items that row_of(i) is.
  auto set_source = [&](const Tile& t, auto index) {
    const bf16_t* src = b_wave ? Bt + (size_t)t.b * N * Kd : a_rows != nullptr ? A : A + (size_t)t.b * R * Kd;
    rsrc = __builtin_amdgcn_make_buffer_rsrc(uniform(src), 0, (int)src_bytes, 0x00020000);
    if (b_wave) {
#pragma unroll
      for (int i = 0; i < LB; ++i)
        off[i] = (uint32_t)min(t.col0 + (i * 4 + w4) * 8 + lrow, N - 1) * (uint32_t)Kd * 2u + piece * 16u;
    } else {
#pragma unroll
      for (int i = 0; i < LA; ++i) {
        int r = row_of(t, i, lrow);
        if (a_rows != nullptr) {
          r = index(i);
          r = (unsigned)r < (unsigned)a_items ? r : 0;
        }
        off[i] = (uint32_t)r * (uint32_t)Kd * 2u + piece * 16u;
      }
    }
  };
  // Addresses past an operand's end (k past Kd in its last row) read as zero.
  auto request_a = [&](int slot, int kt) {
#pragma unroll
    for (int i = 0; i < LA; ++i)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(
          rsrc, (lds_ptr_t)(smem + slot * Cfg::kABytes + (i * 4 + w4) * 1024), 16, off[i], kt * 128, 0, 0);
  };
  auto request_b = [&](int slot, int kt) {
#pragma unroll
    for (int i = 0; i < LB; ++i)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(
          rsrc, (lds_ptr_t)(smem + Cfg::kBAt + slot * Cfg::kBBytes + (i * 4 + w4) * 1024), 16, off[i], kt * 128, 0, 2);
  };
  const bool bias_by_dma = bias != nullptr && (reinterpret_cast<uintptr_t>(bias) & 3u) == 0;
  // The bias of tile t (two columns a lane, the wave's own) and the row numbers of the tile after it.
  auto request_extras = [&](const Tile& t, bool more, const Tile& after) {
    if (bias_by_dma) {
      const __amdgpu_buffer_rsrc_t bias_rsrc = __builtin_amdgcn_make_buffer_rsrc(
          uniform(bias + (size_t)t.b * N), 0, N * 2, 0x00020000);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(
          bias_rsrc, (lds_ptr_t)(smem + Cfg::kBiasAt + wave * 256), 4,
          (uint32_t)(t.col0 + wn * Cfg::TN + lane * 2) * 2u, 0, 0, 0);
    }
    if (!b_wave && a_rows != nullptr && more) {
      const __amdgpu_buffer_rsrc_t idx_rsrc = __builtin_amdgcn_make_buffer_rsrc(
          reinterpret_cast<void*>(uniform(reinterpret_cast<const bf16_t*>(a_rows + (size_t)after.b * R))), 0, R * 4, 0x00020000);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(
          idx_rsrc, (lds_ptr_t)(smem + Cfg::kIndexAt + wave * 256), 4,
          (uint32_t)row_of(after, min(lane >> 3, LA - 1), lane & 7) * 4u, 0, 0, 0);
    }
  };

  const int r16 = lane & 15, q = lane >> 4;
  floatx4 acc[FM][FN];
  auto clear_acc = [&]() {
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
      for (int j = 0; j < FN; ++j) acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};
  };
  clear_acc();
  // v_mfma_f32_16x16x32_bf16: a lane supplies 8 consecutive k of one row (row = lane % 16, k from
  // (lane / 16) * 8).
  typedef float frag_t __attribute__((ext_vector_type(4)));
  const uint32_t a_row = lds0 + (wm * Cfg::TM + r16) * 128;
  const uint32_t b_row = lds0 + Cfg::kBAt + (wn * Cfg::TN + r16) * 128;
  const uint32_t pos[2] = {(uint32_t)((q ^ (r16 >> 1)) * 16), (uint32_t)(((4 + q) ^ (r16 >> 1)) * 16)};
  frag_t fa[2][FM], fb[2][FN];         // of either half (32 k) of a stage
  int sa = 0, sb = 0;                  // slots of the k tile that is multiplied
  auto read_frags = [&](const int ks, int slot_a, int slot_b) {
    const uint32_t at_a = a_row + slot_a * Cfg::kABytes + pos[ks], at_b = b_row + slot_b * Cfg::kBBytes + pos[ks];
#pragma unroll
    for (int j = 0; j < FN; ++j)
      asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(fb[ks][j]) : "v"(at_b), "n"(j * 2048));
#pragma unroll
    for (int i = 0; i < FM; ++i)
      asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(fa[ks][i]) : "v"(at_a), "n"(i * 2048));
  };
  const int nk = (Kd + 63) / 64;
  bool has_next = next_tile(nxt);
  bool after_store = false;            // the tile before this one has left its stores in the count
  auto arrived = [&](const int ks, int t) {
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
    for (int j = 0; j < FN; ++j) asm volatile("" : "+v"(fb[ks][j]));
#pragma unroll
    for (int i = 0; i < FM; ++i) asm volatile("" : "+v"(fa[ks][i]));
    if (Kd % 64 != 0 && t + 1 == nk && t * 64 + ks * 32 + q * 8 >= Kd) {   // k past Kd counts as zero
#pragma unroll
      for (int j = 0; j < FN; ++j) fb[ks][j] = frag_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int i = 0; i < FM; ++i) fa[ks][i] = frag_t{0.f, 0.f, 0.f, 0.f};
    }
  };
  auto multiply = [&](const int ks) {
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
      for (int j = 0; j < FN; ++j)
        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
            __builtin_bit_cast(bf16x8, fb[ks][j]), __builtin_bit_cast(bf16x8, fa[ks][i]), acc[i][j], 0, 0, 0);
  };
  // Waits of either kind of wave: its requests of k tile t + 1 have landed.  Behind them are those of S - 2
  // more k tiles, and the last tile's stores where they came later.
  auto landed = [&](auto s_c, auto l_c, int t) {
    constexpr int S = decltype(s_c)::value, behind = (S - 2) * decltype(l_c)::value;
    if (after_store && t <= S - 3) wait_vmcnt<behind + Cfg::kStores>();
    else if (has_next || nk - 2 - t >= S - 2) wait_vmcnt<behind>();
    else wait_vmcnt<0>();
  };
  using CA = std::integral_constant<int, SA>;
  using CB = std::integral_constant<int, SB>;
  using NA = std::integral_constant<int, LA>;
  using NB = std::integral_constant<int, LB>;
  // Requests of k tile t + S, or of the next tile's k tile t + S - nk, into the slot of k tile t.
  auto ask = [&](auto s_c, int t, auto index, auto request) {
    constexpr int S = decltype(s_c)::value;
    if (t + S < nk) {
      request(t + S);
    } else if (has_next) {
      if (t + S == nk) set_source(nxt, index);
      request(t + S - nk);
    }
  };
  // Step t of a tile: MFMAs of the first half of k tile t over the fragment reads of the second; then
  // the wave's requests of t + 1 have landed; barrier (everyone's have, and everyone has read k tile t);
  // requests into its slots; fragment reads of t + 1; MFMAs of the second half.
  auto step = [&](int t) {
    arrived(0, t);
    read_frags(1, sa, sb);
    multiply(0);
    arrived(1, t);
    const int next_a = sa + 1 == SA ? 0 : sa + 1, next_b = sb + 1 == SB ? 0 : sb + 1;
    if (t + 1 < nk) {
      if (b_wave) landed(CB{}, NB{}, t);
      else landed(CA{}, NA{}, t);
      raw_barrier();
      if (b_wave)
        ask(CB{}, t, [](int) { return 0; }, [&](int kt) { request_b(sb, kt); });
      else
        ask(CA{}, t, [&](int i) { return lds_i32(Cfg::kIndexAt + wave * 256 + (i * 8 + lrow) * 4); },
            [&](int kt) { request_a(sa, kt); });
      read_frags(0, next_a, next_b);
    }
    multiply(1);
    sa = next_a;
    sb = next_b;
  };

  set_source(cur, [&](int i) { return a_rows[(size_t)cur.b * R + row_of(cur, i, lrow)]; });
  request_extras(cur, has_next, nxt);
  if (b_wave) {
    static_for<SB>([&](auto s) { request_b(s, s); });
    wait_vmcnt<(SB - 1) * LB>();
  } else {
    static_for<SA>([&](auto s) { request_a(s, s); });
    wait_vmcnt<(SA - 1) * LA>();
  }
  raw_barrier();
  read_frags(0, 0, 0);
  for (;;) {
    for (int t = 0; t < nk; ++t) step(t);
    // acc[i][j][v] = C[row i * 16 + lane % 16][column j * 16 + (lane / 16) * 4 + v].  Column blocks leave
    // in pairs, eight consecutive columns of a row per lane (gemm_bf16_w8.h); rows and columns past
    // the edge leave through the range check, so that every wave issues kStores stores.
    uint2 bias_pk[FN];
    if (bias_by_dma) {
#pragma unroll
      for (int j = 0; j < FN; ++j)
        asm volatile("ds_read_b64 %0, %1 offset:%2" : "=v"(bias_pk[j]) : "v"(lds0 + Cfg::kBiasAt + wave * 256 + q * 8), "n"(j * 32));
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
      for (int j = 0; j < FN; ++j) asm volatile("" : "+v"(bias_pk[j]));
    } else {
#pragma unroll
      for (int j = 0; j < FN; ++j) {
        bias_pk[j] = make_uint2(0x80008000u, 0x80008000u);     // no bias: x + -0 is x, -0 among them
        if (bias != nullptr)                                   // at an odd element: by ordinary loads
          __builtin_memcpy(&bias_pk[j], bias + (size_t)cur.b * N + min(cur.col0 + wn * Cfg::TN + j * 16 + q * 4, N - 4), 8);
      }
    }
    mfma_result_fence();
    const __amdgpu_buffer_rsrc_t c_rsrc =
        __builtin_amdgcn_make_buffer_rsrc(uniform(C + (size_t)cur.b * R * N), 0, R * N * 2, 0x00020000);
    const int wrow0 = wm * Cfg::TM, wcol0 = cur.col0 + wn * Cfg::TN;
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
        const bool ok = r16 < cur.live - (wrow0 + i * 16) && lane_col + 8 <= N - col_s;
        const uint32_t at = lane_off + (uint32_t)((wrow0 + i * 16) * N + col_s) * 2u;
        __builtin_amdgcn_raw_buffer_store_b128(v, c_rsrc, ok ? at : 0x80000000u, 0, EPI != kEpiBias ? 2 : 0);
        store_data_guard();
      }
    if (!has_next) break;
    cur = nxt;
    has_next = next_tile(nxt);
    request_extras(cur, has_next, nxt);
    clear_acc();
    after_store = true;
    // The tile's first k tile has landed; the slots of the last one of the tile before are free.
    if (b_wave) wait_vmcnt<(SB - 2) * LB + Cfg::kStores>();
    else wait_vmcnt<(SA - 2) * LA + Cfg::kStores>();
    raw_barrier();
    if (b_wave) request_b(sb == 0 ? SB - 1 : sb - 1, SB - 1);
    else request_a(sa == 0 ? SA - 1 : sa - 1, SA - 1);
    read_frags(0, sa, sb);
  }
#endif
}

template <typename Cfg, int EPI>
int launch_gemm_bf16_stream(const bf16_t* A, const bf16_t* Bt, const bf16_t* bias, bf16_t* C, int batch, int R,
                            int N, int Kd, hipStream_t stream, const int32_t* rows, const int32_t* a_rows,
                            int a_items, PlanRef guard, int32_t* clear, int clear_count, int32_t* status) {
  const int tiles_n = (N + Cfg::BN - 1) / Cfg::BN;
  const long long units = (long long)batch * tiles_n;
  if (units > 0x7ffffff0LL) return VMOE_E_OVERFLOW;
  const int per_die = (int)((units + kNumXcd - 1) / kNumXcd);
  auto kern = gemm_bf16_stream_kernel<Cfg, EPI>;
  hipError_t e = allow_dynamic_lds(reinterpret_cast<const void*>(kern), Cfg::kLdsBytes);
  if (e != hipSuccess) return (int)e;
  hipLaunchKernelGGL(kern, dim3(kCusPerXcd * kNumXcd), dim3(Cfg::kThreads), Cfg::kLdsBytes, stream, A, Bt, bias,
                     C, R, N, Kd, tiles_n, (int)units, per_die, batch, rows, a_rows, a_items, guard, clear,
                     clear_count, status);
  return launch_status();
}

}  // namespace vmoe
#endif  // VMOE_GEMM_BF16_STREAM_H_
