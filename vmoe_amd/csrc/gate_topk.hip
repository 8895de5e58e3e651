// Fused router gating for gfx950: logits = x @ W on the matrix cores, softmax
// over experts and top-K selection in registers with cross-lane reductions.
//
// Replaces vmoe/nn/routing.py:73-80 and the jax.lax.top_k of vmoe/moe.py:567.
//
// gate_topk_kernel (bfloat16, what the forms below do not take): a wave owns a tile of 32
// items.  The router kernel W (D x E) is staged once per workgroup in LDS, transposed to
// [expert][k] so that a lane's MFMA B fragment is one 16-byte read.  Item rows
// stream from HBM with 16-byte loads, 64 contiguous bytes per lane per step, through two
// register buffers that are refilled as soon as their
// MFMAs are issued, and the first loads go out before the router kernel is staged,
// so that every workgroup of the launch is resident and loading from the start.
// After the K loop the logits tile passes through a wave-private LDS tile, so
// that each lane holds half of one item's row: softmax and top-K are serial per
// lane, with one xor-32 shuffle per reduction to join the two halves.
// bfloat16 with up to 32 experts and no logits output takes gate_topk_stream_kernel,
// which fetches the item rows with coalesced DMA requests into LDS instead, or, with fewer
// tiles than CUs, gate_topk_split_kernel; with fewer tiles than CUs and up to 64 experts also
// gate_topk_tile_kernel.  float32 takes gate_topk_f32_kernel.
// (VMOE_GATE_DIRECT_LOADS=1 in the environment keeps the direct loads: the switch behind
// the before / after figures.)
#include <algorithm>
#include <cstdlib>
#include <type_traits>

#include "vmoe_common.h"
#include "router_metrics.h"

namespace vmoe {
namespace {

__device__ __forceinline__ float inv_orderable(uint32_t u) {
  uint32_t b = (u & 0x80000000u) ? (u & 0x7fffffffu) : ~u;
  return __builtin_bit_cast(float, b);
}

// Softmax and top-K of one item by two lanes: g holds the logits of experts h * EP / 2 ..., lane ^ 32 the
// others.  Sums and maxima are serial per lane; the halves meet with one xor-32 shuffle each.
// Logits -> exponentials; returns their sum.
template <int EP>
__device__ __forceinline__ float exponentials(float (&g)[EP / 2], int E, int h) {
  constexpr int CNT = EP / 2;
  const int n0 = h * CNT;
  float mx = -INFINITY;
#pragma unroll
  for (int j = 0; j < CNT; ++j) {
    g[j] = (n0 + j < E) ? g[j] : -INFINITY;
    mx = fmaxf(mx, g[j]);
  }
  mx = fmaxf(mx, __shfl_xor(mx, 32, kWave));
  float sum = 0.f;
#pragma unroll
  for (int j = 0; j < CNT; ++j) {
    g[j] = (n0 + j < E) ? expf(g[j] - mx) : 0.f;
    sum += g[j];
  }
  return sum + __shfl_xor(sum, 32, kWave);
}
// Exponentials and their sum -> gates and top-K.
template <typename T, int EP>
__device__ __forceinline__ void finish_exponentials(float (&g)[EP / 2], float sum, T* __restrict__ gates, float* __restrict__ topk_val,
                                                    int32_t* __restrict__ topk_idx, int row, int num_items, int E, int K, int h) {
  constexpr int CNT = EP / 2;
  const int n0 = h * CNT;
  const bool row_ok = row < num_items;
#pragma unroll
  for (int j = 0; j < CNT; ++j) g[j] = Elt<T>::round(g[j] / sum);
  if (gates != nullptr && row_ok) {
    T* grow = gates + (size_t)row * E + n0;
    if (sizeof(T) == 2 && (E & 7) == 0 && (reinterpret_cast<uintptr_t>(gates) & 15u) == 0) {
#pragma unroll
      for (int j = 0; j < CNT; j += 8) {
        if (n0 + j < E) {
          uint32_t pk[4];
#pragma unroll
          for (int t = 0; t < 4; ++t) pk[t] = pack_bf16x2(g[j + 2 * t], g[j + 2 * t + 1]);
          *reinterpret_cast<uint4*>(grow + j) = make_uint4(pk[0], pk[1], pk[2], pk[3]);
        }
      }
    } else if (sizeof(T) == 4 && (E & 3) == 0 && (reinterpret_cast<uintptr_t>(gates) & 15u) == 0) {
#pragma unroll
      for (int j = 0; j < CNT; j += 4)
        if (n0 + j < E) *reinterpret_cast<float4*>(grow + j) = make_float4(g[j], g[j + 1], g[j + 2], g[j + 3]);
    } else {
#pragma unroll
      for (int j = 0; j < CNT; ++j)
        if (n0 + j < E) Elt<T>::store(grow + j, g[j]);
    }
  }
  uint64_t taken = 0;
  for (int kk = 0; kk < K; ++kk) {
    uint64_t best = 0;
#pragma unroll
    for (int j = 0; j < CNT; ++j) {
      const int n = n0 + j;
      if (n < E && !(taken >> j & 1ull)) {
        uint64_t key = ((uint64_t)orderable(g[j]) << 32) | (uint32_t)(0xFFFFFFFFu - (uint32_t)n);
        best = key > best ? key : best;
      }
    }
    const uint32_t olo = __shfl_xor((uint32_t)best, 32, kWave);
    const uint32_t ohi = __shfl_xor((uint32_t)(best >> 32), 32, kWave);
    const uint64_t other = ((uint64_t)ohi << 32) | olo;
    best = other > best ? other : best;
    const int n_star = (int)(0xFFFFFFFFu - (uint32_t)best);
    if (n_star >= n0 && n_star < n0 + CNT) taken |= 1ull << (n_star - n0);
    if (h == 0 && row_ok) {
      topk_val[(size_t)row * K + kk] = inv_orderable((uint32_t)(best >> 32));
      topk_idx[(size_t)row * K + kk] = n_star;
    }
  }
}

template <typename T, int EP>
__device__ __forceinline__ void finish_row(float (&g)[EP / 2], T* __restrict__ gates, float* __restrict__ topk_val, int32_t* __restrict__ topk_idx,
                                           int row, int num_items, int E, int K, int h) {
  const float sum = exponentials<EP>(g, E, h);
  finish_exponentials<T, EP>(g, sum, gates, topk_val, topk_idx, row, num_items, E, K, h);
}

// The logits output of a tile of finished logits in LDS (row pitch `pitch`), by one wave.
__device__ __forceinline__ void store_logits(const float* st, int pitch, float* __restrict__ logits, int row0,
                                             int num_items, int E, int lane) {
  const int n = min(32, num_items - row0) * E;
  float* const out = logits + (size_t)row0 * E;
  for (int i = lane; i < n; i += kWave) {
    const int r = i / E;
    out[i] = st[r * pitch + i - r * E];
  }
}

// A 32 x 32 tile of finished bfloat16 logits (row pitch 33).
__device__ __forceinline__ void finish_tile32(const float* st, bf16_t* __restrict__ gates,
                                              float* __restrict__ topk_val, int32_t* __restrict__ topk_idx,
                                              int row0, int num_items, int E, int K, int m, int h) {
  float g[16];
#pragma unroll
  for (int j = 0; j < 16; ++j) g[j] = st[m * 33 + h * 16 + j];
  finish_row<bf16_t, 32>(g, gates, topk_val, topk_idx, row0 + m, num_items, E, K, h);
}

// Stages rows k0 .. k0 + kc of a bfloat16 router kernel (D x E) of any E and alignment in LDS as
// [expert][k]: a unit is eight k of one expert, read as eight 2-byte loads (neighbouring lanes read
// neighbouring experts) and written as one 16-byte piece.  The loads of four units per thread are in flight
// at once: every address is clamped into the matrix, so none waits on a branch.  Rows past D are zero;
// experts past E are left as they are (their logits are never read).
__device__ __forceinline__ void stage_router_any(const bf16_t* __restrict__ w, bf16_t* wl, int stride, int k0,
                                                 int kc, int D, int E, int tid, int threads) {
  constexpr int kBatch = 4;
  const int units = kc / 8 * E;
  for (int u0 = tid; u0 < units; u0 += kBatch * threads) {
    uint32_t raw[kBatch][8];
    int at[kBatch], left[kBatch];
#pragma unroll
    for (int t = 0; t < kBatch; ++t) {
      const int u = min(u0 + t * threads, units - 1);   // (a thread past the end repeats the last unit)
      const int kb = u / E, n = u - kb * E, k = k0 + kb * 8;
      at[t] = n * stride + kb * 8;
      left[t] = D - k;
#pragma unroll
      for (int i = 0; i < 8; ++i) raw[t][i] = w[(size_t)min(k + i, D - 1) * E + n];
    }
#pragma unroll
    for (int t = 0; t < kBatch; ++t) {
#pragma unroll
      for (int i = 0; i < 8; ++i) raw[t][i] = i < left[t] ? raw[t][i] : 0;
      *reinterpret_cast<uint4*>(wl + at[t]) = make_uint4(raw[t][0] | raw[t][1] << 16, raw[t][2] | raw[t][3] << 16,
                                                         raw[t][4] | raw[t][5] << 16, raw[t][6] | raw[t][7] << 16);
    }
  }
}

template <int NT, bool LOGITS, int WAVES>
__global__ __launch_bounds__(WAVES * kWave) void gate_topk_kernel(
    const bf16_t* __restrict__ x, const bf16_t* __restrict__ w, const float* __restrict__ bias,
    bf16_t* __restrict__ gates, float* __restrict__ logits, float* __restrict__ topk_val,
    int32_t* __restrict__ topk_idx,
    int num_items, int D, int E, int K, int KC, int num_chunks, int num_tiles, int stage_off) {
  extern __shared__ __align__(16) unsigned char smem[];
  bf16_t* wl = reinterpret_cast<bf16_t*>(smem);
  constexpr int kGateWaves = WAVES;
  constexpr int kGateThreads = kGateWaves * kWave;
  constexpr int EP = NT * 32;
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  const int m = lane & 31;
  const int h = lane >> 5;
  const int stride = KC + 8;
  const int tiles_per_iter = gridDim.x * kGateWaves;
  const int iters = (num_tiles + tiles_per_iter - 1) / tiles_per_iter;

  for (int it = 0; it < iters; ++it) {
    const int tile = it * tiles_per_iter + blockIdx.x * kGateWaves + wave;
    const bool active = tile < num_tiles;
    const int row0 = tile * 32;
    int r = row0 + m;
    if (r >= num_items) r = num_items - 1;
    if (r < 0) r = 0;
    const bf16_t* xrow = x + (size_t)r * D;

    floatx16 acc[NT];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[nt][i] = 0.f;

    // bf16: the loads of the first round of router-kernel blocks and of the first
    // batch of item rows go out together, before anything waits: the blocks come back
    // first and are staged under the latency of the rows.
    constexpr int UB = 2;   // 64-k blocks per batch; two batches (16 x 16-byte loads per lane) in flight
    uint4 wraw[8];
    uint4 a[2][UB][4];
    using Buf0 = std::integral_constant<int, 0>;
    using Buf1 = std::integral_constant<int, 1>;
    auto load_w_block = [&](int k0, int kb, int nb, bool in_range) {
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const int k = k0 + kb * 8 + i;
        wraw[i] = (in_range && k < D && nb * 8 < E)
                                  ? *reinterpret_cast<const uint4*>(w + (size_t)k * E + nb * 8)
                                  : make_uint4(0, 0, 0, 0);
      }
    };
    auto load_rows = [&](auto buf, int k0, int kb0, int nkb) {
#pragma unroll
      for (int u = 0; u < UB; ++u)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const int kg = k0 + (kb0 + u) * 64 + h * 32 + j * 8;
          a[decltype(buf)::value][u][j] = (kb0 + u < nkb && kg + 8 <= D)
                                              ? *reinterpret_cast<const uint4*>(xrow + kg)
                                              : make_uint4(0, 0, 0, 0);
        }
    };
    auto mma_rows = [&](auto buf, int kb0, int nkb) {
#pragma unroll
      for (int u = 0; u < UB; ++u) {
        if (kb0 + u >= nkb) break;
        const int kl = (kb0 + u) * 64 + h * 32;  // this lane's 32 k's inside the chunk
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          bf16x8 af = __builtin_bit_cast(bf16x8, a[decltype(buf)::value][u][j]);
#pragma unroll
          for (int nt = 0; nt < NT; ++nt) {
            uint4 b = *reinterpret_cast<const uint4*>(wl + (nt * 32 + m) * stride + kl + j * 8);
            acc[nt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(af, __builtin_bit_cast(bf16x8, b),
                                                              acc[nt], 0, 0, 0);
          }
        }
      }
    };
    {
      if (it == 0 && E % 8 == 0 && (reinterpret_cast<uintptr_t>(w) & 15u) == 0) {
        const int nbn = EP / 8;
        load_w_block(0, tid / nbn, tid % nbn, tid < (KC / 8) * nbn);
      }
      if (active) {
        load_rows(Buf0{}, 0, 0, KC / 64);
        load_rows(Buf1{}, 0, UB, KC / 64);
      }
    }

    for (int c = 0; c < num_chunks; ++c) {
      const int k0 = c * KC;
      if (num_chunks > 1 || it == 0) {
        __syncthreads();
        // Stage W[k0 : k0+KC, :] into LDS, zero padded in both directions.  When
        // a row of W is a whole number of 16-byte vectors the loads are vector
        // loads, all independent, so the staging costs one memory round trip.
        if (E % 8 == 0 && (reinterpret_cast<uintptr_t>(w) & 15u) == 0) {
          // bf16: a thread loads an 8(k) x 8(expert) block with eight 16-byte loads,
          // transposes it in registers and writes each expert's eight consecutive k
          // as one 16-byte chunk (2-byte LDS writes made this the longest phase of
          // the kernel).  The first round of loads was issued before the item rows.
          const int nbn = EP / 8, nblk = (KC / 8) * nbn;
          for (int b0 = 0; b0 < nblk; b0 += kGateThreads) {
            const int b = b0 + tid;
            const int kb = b / nbn, nb = b - kb * nbn;
            if (!(b0 == 0 && c == 0 && it == 0)) load_w_block(k0, kb, nb, b < nblk);
            if (b < nblk) {
#pragma unroll
              for (int j = 0; j < 8; ++j) {
                const uint32_t sel = (j & 1) ? 0x07060302u : 0x05040100u;
                uint32_t o[4];
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                  const uint32_t hi = reinterpret_cast<const uint32_t*>(&wraw[2 * q + 1])[j >> 1];
                  const uint32_t lo = reinterpret_cast<const uint32_t*>(&wraw[2 * q])[j >> 1];
                  o[q] = __builtin_amdgcn_perm(hi, lo, sel);
                }
                *reinterpret_cast<uint4*>(wl + (size_t)(nb * 8 + j) * stride + kb * 8) =
                    make_uint4(o[0], o[1], o[2], o[3]);
              }
            }
          }
        } else if constexpr (NT <= 2) {
          stage_router_any(w, wl, stride, k0, KC, D, E, tid, kGateThreads);
        } else {
          for (int idx = tid; idx < KC * EP; idx += kGateThreads) {
            int k = idx / EP, n = idx - k * EP;
            bf16_t v = 0;
            if (k0 + k < D && n < E) v = w[(size_t)(k0 + k) * E + n];
            wl[n * stride + k] = v;
          }
        }
        __syncthreads();
      }
      if (!active) continue;
      {
        const int nkb = KC / 64;
        if (c > 0) {
          load_rows(Buf0{}, k0, 0, nkb);
          load_rows(Buf1{}, k0, UB, nkb);
        }
        // A buffer is refilled as soon as its MFMAs are issued, so two batches stay in flight.
        for (int kb0 = 0; kb0 < nkb; kb0 += 2 * UB) {
          mma_rows(Buf0{}, kb0, nkb);
          load_rows(Buf0{}, k0, kb0 + 2 * UB, nkb);
          mma_rows(Buf1{}, kb0 + UB, nkb);
          load_rows(Buf1{}, k0, kb0 + 3 * UB, nkb);
          mfma_result_fence();
        }
      }
    }
    if (!active) continue;

    // Epilogue.  The 32 x EP tile of (rounded, biased) logits goes through a
    // wave-private LDS tile so that a lane ends up with half of one item's row in
    // registers (lane = item r, half h of the experts): softmax and top-K are then
    // serial per lane, and the two halves of a row meet with a single xor-32
    // shuffle per reduction instead of a five-step butterfly per row.
    float* st = reinterpret_cast<float*>(smem + stage_off) + (size_t)wave * 32 * (EP + 1);
    {
      float bn[NT];
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) {
        int n = nt * 32 + m;
        bn[nt] = (bias != nullptr && n < E) ? bias[n] : 0.f;
      }
#pragma unroll
      for (int nt = 0; nt < NT; ++nt)
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          const int rl = (i >> 2) * 8 + h * 4 + (i & 3);
          float v = bf16r(acc[nt][i]);
          if (bias != nullptr) v = bf16r(v + bn[nt]);
          st[rl * (EP + 1) + nt * 32 + m] = v;
        }
    }
    constexpr int CNT = EP / 2;          // experts per lane
    const int row = row0 + m;
    const int n0 = h * CNT;
    float g[CNT];
    float mx = -INFINITY;
#pragma unroll
    for (int j = 0; j < CNT; ++j) {
      float v = st[m * (EP + 1) + n0 + j];
      g[j] = (n0 + j < E) ? v : -INFINITY;
      mx = fmaxf(mx, g[j]);
    }
    if (LOGITS && row < num_items) {
#pragma unroll
      for (int j = 0; j < CNT; ++j)
        if (n0 + j < E) logits[(size_t)row * E + n0 + j] = g[j];
    }
    mx = fmaxf(mx, __shfl_xor(mx, 32, kWave));
    float sum = 0.f;
#pragma unroll
    for (int j = 0; j < CNT; ++j) {
      g[j] = (n0 + j < E) ? expf(g[j] - mx) : 0.f;
      sum += g[j];
    }
    sum += __shfl_xor(sum, 32, kWave);
#pragma unroll
    for (int j = 0; j < CNT; ++j) g[j] = Elt<bf16_t>::round(g[j] / sum);
    const bool row_ok = row < num_items;
    if (gates != nullptr && row_ok) {
      bf16_t* grow = gates + (size_t)row * E + n0;
      if ((E & 7) == 0 && (reinterpret_cast<uintptr_t>(gates) & 15u) == 0) {
#pragma unroll
        for (int j = 0; j < CNT; j += 8) {
          if (n0 + j < E) {
            uint32_t pk[4];
#pragma unroll
            for (int t = 0; t < 4; ++t) pk[t] = pack_bf16x2(g[j + 2 * t], g[j + 2 * t + 1]);
            *reinterpret_cast<uint4*>(grow + j) = make_uint4(pk[0], pk[1], pk[2], pk[3]);
          }
        }
      } else {
#pragma unroll
        for (int j = 0; j < CNT; ++j)
          if (n0 + j < E) Elt<bf16_t>::store(grow + j, g[j]);
      }
    }
    uint64_t taken = 0;
    for (int kk = 0; kk < K; ++kk) {
      uint64_t best = 0;
#pragma unroll
      for (int j = 0; j < CNT; ++j) {
        const int n = n0 + j;
        if (n < E && !(taken >> j & 1ull)) {
          uint64_t key = ((uint64_t)orderable(g[j]) << 32) | (uint32_t)(0xFFFFFFFFu - (uint32_t)n);
          best = key > best ? key : best;
        }
      }
      const uint32_t olo = __shfl_xor((uint32_t)best, 32, kWave);
      const uint32_t ohi = __shfl_xor((uint32_t)(best >> 32), 32, kWave);
      const uint64_t other = ((uint64_t)ohi << 32) | olo;
      best = other > best ? other : best;
      const int n_star = (int)(0xFFFFFFFFu - (uint32_t)best);
      if (n_star >= n0 && n_star < n0 + CNT) taken |= 1ull << (n_star - n0);
      if (h == 0 && row_ok) {
        topk_val[(size_t)row * K + kk] = inv_orderable((uint32_t)(best >> 32));
        topk_idx[(size_t)row * K + kk] = n_star;
      }
    }
  }
}

// float32 gating on the bfloat16 matrix cores: every value is taken apart into three bfloat16 values that add
// up to it exactly and six of the nine products are summed in float32, as in gemm_f32_split.h; hi.hi in one sum
// and the five smaller products in another, which meet once k is through: a large sum is rounded once per 16 k.
// Off from 64 bits (2-norm, 4 096 x 768 x 8): 8.0e-8 where float32 MFMAs are off by 2.5e-7; items with two or
// eight non-zero features 3.6e-8 and 5.3e-8, as those (with all six in one sum 4.5e-8 and 6.8e-8).  The waves of a workgroup (eight; four beyond 64
// experts, for the registers) share TW tiles of 32 items, WAVES / TW waves to a tile, each with its share of every chunk of KC rows of the router kernel; the
// launcher takes as many tiles per workgroup as keep the workgroups at one per CU.  The chunk is split and
// transposed on its way into LDS, [plane][expert][k], read as eight floats of an expert per thread with
// neighbouring lanes on neighbouring experts, whatever E and the address are.  Item rows come four 16-wide k
// steps at a time, two such batches in flight, the first two sent before the chunk is staged.  The partial
// logits of a tile meet in LDS, added in wave order, and its first wave finishes it.  (How many waves share a tile
// depends on the number of items, and with it the last bits of an item's logits.)
// Bound by the trips to memory (few items: 12 - 15 us; 2 688 items x 832, 38 experts: 73 us on float32 MFMAs with a
// scalar staging loop, 25 here) or by the splitting and the items' bytes (17 024 x 896, 51 experts: 114 to 50;
// 30 000 x 384, 16 experts: 21 to 19; 15 774 x 544, 6 experts: 35 to 18).
// The infinite and NaN logits of a tile (32 rows of pitch EP + 1 in LDS; xrow: the lane's row) again, on float32
// MFMAs, by one wave: an operand that is infinite or rounds to infinity leaves NaN in the sums of its pieces'
// products, which the softmax's sum shows.  (A call of its own: inline, its registers cost every launch 0.4 to 2 us.
// 196 x 768 x 8, nothing but NaN: 35 us; the check costs 0.2 us of the 12.)
template <int NT>
__device__ __noinline__ void retake_logits(const float* __restrict__ xrow, const float* __restrict__ w,
                                              const float* __restrict__ bias, float* st, int D, int E, int lane) {
  const int m = lane & 31, h = lane >> 5;
  floatx16 acc[NT];
#pragma unroll
  for (int nt = 0; nt < NT; ++nt)
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[nt][i] = 0.f;
  constexpr int kSteps = NT == 4 ? 2 : 4;         // of eight k; their loads are in flight together
#pragma unroll 1
  for (int k0 = 0; k0 < D; k0 += 8 * kSteps) {
    float4 x4[kSteps];
    float b[kSteps][4][NT];
#pragma unroll
    for (int s = 0; s < kSteps; ++s) {            // lanes 0 - 31 take the first four k of a step, 32 - 63 the others
      const int k = k0 + s * 8 + h * 4;
      x4[s] = *reinterpret_cast<const float4*>(xrow + min(k, D - 4));
#pragma unroll
      for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) b[s][t][nt] = w[(size_t)min(k + t, D - 1) * E + min(nt * 32 + m, E - 1)];
    }
#pragma unroll
    for (int s = 0; s < kSteps; ++s) {
      const bool in = k0 + s * 8 + h * 4 < D;
      const float v[4] = {x4[s].x, x4[s].y, x4[s].z, x4[s].w};
#pragma unroll
      for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int nt = 0; nt < NT; ++nt)
          acc[nt] = __builtin_amdgcn_mfma_f32_32x32x2f32(in ? v[t] : 0.f, in ? b[s][t][nt] : 0.f, acc[nt], 0, 0, 0);
    }
  }
  mfma_result_fence();
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) {
    const int n = nt * 32 + m;
    const float bn = bias != nullptr ? bias[min(n, E - 1)] : 0.f;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      float* const at = st + ((i >> 2) * 8 + h * 4 + (i & 3)) * (NT * 32 + 1) + n;
      if (!(*at - *at == 0.f)) *at = acc[nt][i] + bn;
    }
  }
  wait_lgkmcnt0();
}

constexpr int kNumCus = 256;

template <int NT, int WAVES, int TW>
__global__ __launch_bounds__(WAVES * kWave) void gate_topk_f32_kernel(
    const float* __restrict__ x, const float* __restrict__ w, const float* __restrict__ bias,
    float* __restrict__ gates, float* __restrict__ logits, float* __restrict__ topk_val,
    int32_t* __restrict__ topk_idx, int num_items, int D, int E, int K, int KC, int num_chunks, int num_tiles) {
  extern __shared__ __align__(16) unsigned char smem[];
  constexpr int KS = WAVES / TW, EP = NT * 32, kThreads = WAVES * kWave, FB = NT == 1 ? 4 : 2;
  const int stride = KC + 8;                               // bfloat16 per expert and plane
  bf16_t* const wl = reinterpret_cast<bf16_t*>(smem);
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int part = wave % KS, m = lane & 31, h = lane >> 5;
  float* const st = reinterpret_cast<float*>(smem) + (size_t)wave * 32 * (EP + 1);    // once W has been read
  const int kb_lo = part * (KC / 16 / KS), kb_hi = kb_lo + KC / 16 / KS;

  for (int tile0 = blockIdx.x * TW; tile0 < num_tiles; tile0 += gridDim.x * TW) {
    const int tile = tile0 + wave / KS;
    const int row0 = tile * 32;
    const float* const xrow = x + (size_t)min(row0 + m, num_items - 1) * D;
    floatx16 acc[NT], low[NT];                    // sums of hi.hi, and of the five smaller products
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[nt][i] = low[nt][i] = 0.f;
    float4 va[2][FB][2];
    // (what lies past the wave's share or past D is read from the row's end and multiplied by the zero
    // rows of W or not at all)
    auto load_rows = [&](const int u, int k0, int kb0) {
#pragma unroll
      for (int t = 0; t < FB; ++t)
#pragma unroll
        for (int j = 0; j < 2; ++j)
          va[u][t][j] = *reinterpret_cast<const float4*>(xrow + min(k0 + (kb0 + t) * 16 + h * 8 + j * 4, D - 4));
    };
    auto mma_rows = [&](const int u, int k0, int kb0) {
#pragma unroll
      for (int t = 0; t < FB; ++t) {
        if (kb0 + t >= kb_hi) break;
        const int kl = (kb0 + t) * 16 + h * 8;
        uint32_t a[3][4];
        const float v[8] = {va[u][t][0].x, va[u][t][0].y, va[u][t][0].z, va[u][t][0].w,
                            va[u][t][1].x, va[u][t][1].y, va[u][t][1].z, va[u][t][1].w};
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const bool in = k0 + kl + (i & 2) * 2 < D;       // (whole quads: D is a multiple of four)
          split3(in ? v[2 * i] : 0.f, in ? v[2 * i + 1] : 0.f, a[0][i], a[1][i], a[2][i]);
        }
        bf16x8 af[3];
#pragma unroll
        for (int p = 0; p < 3; ++p)
          af[p] = __builtin_bit_cast(bf16x8, make_uint4(a[p][0], a[p][1], a[p][2], a[p][3]));
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
          const bf16_t* const b = wl + (nt * 32 + m) * stride + kl;
          bf16x8 bf[3];
#pragma unroll
          for (int p = 0; p < 3; ++p) bf[p] = *reinterpret_cast<const bf16x8*>(b + (size_t)p * EP * stride);
          acc[nt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(af[0], bf[0], acc[nt], 0, 0, 0);
          constexpr int ta[5] = {2, 0, 1, 1, 0}, tb[5] = {0, 2, 1, 0, 1};
#pragma unroll
          for (int p = 0; p < 5; ++p)
            low[nt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(af[ta[p]], bf[tb[p]], low[nt], 0, 0, 0);
        }
      }
    };
    for (int c = 0; c < num_chunks; ++c) {
      const int k0 = c * KC;
      load_rows(0, k0, kb_lo);
      load_rows(1, k0, kb_lo + FB);
      __syncthreads();                            // the chunk, or the logits, before have been read
      constexpr int kBatch = NT == 1 ? 4 : NT == 2 ? 2 : 1;    // units in flight per thread
      const int units = KC / 8 * E;
      for (int u0 = tid; u0 < units; u0 += kBatch * kThreads) {
        float raw[kBatch][8];
        int at[kBatch], left[kBatch];
#pragma unroll
        for (int t = 0; t < kBatch; ++t) {
          const int u = min(u0 + t * kThreads, units - 1);   // (a thread past the end repeats the last unit)
          const int kb = u / E, n = u - kb * E, k = k0 + kb * 8;
          at[t] = n * stride + kb * 8;
          left[t] = D - k;
#pragma unroll
          for (int i = 0; i < 8; ++i) raw[t][i] = w[(size_t)min(k + i, D - 1) * E + n];
        }
#pragma unroll
        for (int t = 0; t < kBatch; ++t) {
          uint32_t o[3][4];
#pragma unroll
          for (int i = 0; i < 4; ++i)
            split3(2 * i < left[t] ? raw[t][2 * i] : 0.f, 2 * i + 1 < left[t] ? raw[t][2 * i + 1] : 0.f,
                       o[0][i], o[1][i], o[2][i]);
#pragma unroll
          for (int p = 0; p < 3; ++p)
            *reinterpret_cast<uint4*>(wl + (size_t)p * EP * stride + at[t]) = make_uint4(o[p][0], o[p][1], o[p][2], o[p][3]);
        }
      }
      __syncthreads();
      if (tile < num_tiles) {
        for (int kb0 = kb_lo; kb0 < kb_hi; kb0 += 2 * FB) {
          mma_rows(0, k0, kb0);
          if (kb0 + 2 * FB < kb_hi) load_rows(0, k0, kb0 + 2 * FB);
          mma_rows(1, k0, kb0 + FB);
          if (kb0 + 3 * FB < kb_hi) load_rows(1, k0, kb0 + 3 * FB);
          mfma_result_fence();
        }
      }
    }
    __syncthreads();                              // W's LDS takes the logits
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      const float bn = KS == 1 && bias != nullptr ? bias[min(nt * 32 + m, E - 1)] : -0.f;       // (x + -0 is x)
#pragma unroll
      for (int i = 0; i < 16; ++i) st[((i >> 2) * 8 + h * 4 + (i & 3)) * (EP + 1) + nt * 32 + m] = acc[nt][i] + low[nt][i] + bn;
    }
    __syncthreads();
    if constexpr (KS > 1) {
      for (int e = tid; e < TW * 32 * EP; e += kThreads) {
        const int n = e & (EP - 1), r = (e / EP) & 31;
        float* const at = reinterpret_cast<float*>(smem) + (size_t)(e / (32 * EP)) * KS * 32 * (EP + 1) + r * (EP + 1) + n;
        float v = at[0];
#pragma unroll
        for (int p = 1; p < KS; ++p) v += at[p * 32 * (EP + 1)];
        if (bias != nullptr) v += bias[min(n, E - 1)];
        at[0] = v;
      }
      __syncthreads();
    }
    if (part == 0 && tile < num_tiles) {
      constexpr int CNT = EP / 2;
      float g[CNT];
      auto read = [&]() {
#pragma unroll
        for (int j = 0; j < CNT; ++j) g[j] = st[m * (EP + 1) + h * CNT + j];
      };
      read();
      float sum = exponentials<EP>(g, E, h);
      if (__builtin_expect(__any(!(sum < INFINITY)), 0)) {
        retake_logits<NT>(xrow, w, bias, st, D, E, lane);
        read();
        sum = exponentials<EP>(g, E, h);
      }
      if (logits != nullptr) store_logits(st, EP + 1, logits, row0, num_items, E, lane);
      finish_exponentials<float, EP>(g, sum, gates, topk_val, topk_idx, row0 + m, num_items, E, K, h);
    }
  }
}

// Streaming form of the bfloat16 kernel for up to 32 experts (the routers' common case).
// The item rows are the whole traffic (77 MB on the headline layer, 0.05 MB of router
// kernel), so they are fetched the way a copy kernel fetches: every DMA request of a wave
// covers 8 rows x 128 contiguous bytes (a 64-wide k chunk of the wave's 32-row tile is four
// requests) and lands in a wave-private ring of LDS slots, from which the MFMA A fragments
// are read; the direct loads of gate_topk_kernel fetch 16 bytes per lane from 32 different
// rows per request and reach half the rate.  Eight waves per workgroup share one staged
// copy of the router kernel; a wave runs SLOTS - 1 chunks ahead of its MFMAs.  The chunk's
// 16-byte pieces are XOR-swizzled by row on their way in (the lane picks the global piece
// that belongs in its LDS position), so that the fragment reads spread over the banks.
// Epilogue as in gate_topk_kernel, its tile staged in the wave's own ring.  Headline layer
// (50 176 items x 768, 77 MB): 21.9 us against 29.5 - 31.3 with direct loads (kernel trace);
// two or three slots, seven or eight waves per workgroup make no difference.
constexpr int kStreamWaves = 8;
constexpr int kStreamChunkBytes = 32 * 128;      // 32 rows x 64 bfloat16

typedef __attribute__((address_space(3))) void* gate_lds_ptr_t;

// ANY: any number of experts and any alignment of w, and gate_topk_kernel's dealing of k to the products
// (a lane's half takes 32 consecutive k of a chunk), whose sums it repeats bit for bit (11 250 items x 704,
// 4 experts: 22 us with direct loads, 11 here; 38 060 x 256, 12 experts: 18 to 10).
template <int SLOTS, int WAVES, bool ANY>
__global__ __launch_bounds__(WAVES * kWave, 1) void gate_topk_stream_kernel(
    const bf16_t* __restrict__ x, const bf16_t* __restrict__ w, const float* __restrict__ bias,
    bf16_t* __restrict__ gates, float* __restrict__ topk_val, int32_t* __restrict__ topk_idx,
    int num_items, int D, int E, int K, int num_tiles, int w_bytes) {
#if defined(__HIP_DEVICE_COMPILE__)   // buffer-resource builtins exist in the device pass only
  extern __shared__ __align__(1024) unsigned char smem[];
  bf16_t* wl = reinterpret_cast<bf16_t*>(smem);
  constexpr int kThreads = WAVES * kWave;
  constexpr int EP = 32;
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int m = lane & 31;
  const int h = lane >> 5;
  const int stride = D + 8;                        // elements per expert row of the staged router kernel
  unsigned char* ring = smem + w_bytes + wave * (SLOTS * kStreamChunkBytes);

  const __amdgpu_buffer_rsrc_t x_rsrc = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<bf16_t*>(x), 0, -1, 0x00020000);
  typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
  const uint32_t ring_addr = (uint32_t)reinterpret_cast<uintptr_t>((gate_lds_ptr_t)ring);
  const uint32_t wl_addr = (uint32_t)reinterpret_cast<uintptr_t>((gate_lds_ptr_t)wl);
  const int nchunks = D / 64;
  const int lrow = lane >> 3;                      // row of this lane inside a request (8 rows x 8 pieces)
  const int swz = m & 7;
  const int tile0 = blockIdx.x * WAVES + wave;
  // Request i of a chunk fills LDS rows 8 i .. 8 i + 7; lane L lands in row 8 i + L / 8,
  // position L % 8, and therefore fetches piece (L % 8) ^ (row & 7) of that row.
  uint32_t goff[4];
  auto tile_offsets = [&](int tile) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int rl = i * 8 + lrow;
      const int r = min(tile * 32 + rl, num_items - 1);
      goff[i] = (uint32_t)r * (uint32_t)D * 2u + (uint32_t)(((lane & 7) ^ (rl & 7)) * 16);
    }
  };
  auto request = [&](int c) {
    unsigned char* s = ring + (c % SLOTS) * kStreamChunkBytes;
#pragma unroll
    for (int i = 0; i < 4; ++i)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(x_rsrc, (gate_lds_ptr_t)(s + i * 1024), 16, goff[i],
                                               c * 128, 0, 0);
  };
  // The first requests of the wave's first tile go out before the router kernel is staged:
  // every wave of the launch is loading from its first instruction on.
  if (tile0 < num_tiles) {
    tile_offsets(tile0);
#pragma unroll
    for (int c = 0; c < SLOTS - 1; ++c)
      if (c < nchunks) request(c);
  }

  // Router kernel -> LDS as [expert][k]: a thread loads an 8 (k) x 8 (expert) block with
  // eight 16-byte loads, transposes it in registers and writes each expert's eight
  // consecutive k as one 16-byte piece (E % 8 == 0 and a 16-byte aligned w: the launcher
  // checks); experts E .. 31 are zero.  The LDS writes are written as instructions, like the
  // fragment reads below: a write the compiler can see would wait for the requests above.
  if constexpr (ANY) {
    stage_router_any(w, wl, stride, 0, D, D, E, tid, kThreads);
  } else {
    const int nbn = EP / 8, nblk = (D / 8) * nbn;
    for (int b0 = 0; b0 < nblk; b0 += kThreads) {
      const int b = b0 + tid;
      const int kb = b / nbn, nb = b - kb * nbn;
      uint4 wraw[8];
#pragma unroll
      for (int i = 0; i < 8; ++i)
        wraw[i] = (b < nblk && nb * 8 < E)
                      ? *reinterpret_cast<const uint4*>(w + (size_t)(kb * 8 + i) * E + nb * 8)
                      : make_uint4(0, 0, 0, 0);
      if (b < nblk) {
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          const uint32_t sel = (j & 1) ? 0x07060302u : 0x05040100u;
          u32x4_t o;
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            const uint32_t hi = reinterpret_cast<const uint32_t*>(&wraw[2 * q + 1])[j >> 1];
            const uint32_t lo = reinterpret_cast<const uint32_t*>(&wraw[2 * q])[j >> 1];
            o[q] = __builtin_amdgcn_perm(hi, lo, sel);
          }
          asm volatile("ds_write_b128 %0, %1" ::"v"(wl_addr + (uint32_t)(((nb * 8 + j) * stride + kb * 8) * 2)), "v"(o)
                       : "memory");
        }
      }
    }
  }
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  __syncthreads();

  for (int tile = tile0; tile < num_tiles; tile += gridDim.x * WAVES) {
    const int row0 = tile * 32;
    floatx16 acc;
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[i] = 0.f;
    if (tile != tile0) {         // (the first tile's were issued before the router kernel was staged)
      tile_offsets(tile);
#pragma unroll
      for (int c = 0; c < SLOTS - 1; ++c)
        if (c < nchunks) request(c);
    }
    // The fragment reads are written as instructions: the compiler drains every DMA request
    // in front of an LDS read it can see (it cannot tell that the requests in flight fill
    // other slots), which would leave a wave with one chunk in flight.
    auto multiply = [&](int c) {
      const uint32_t sa = ring_addr + (uint32_t)((c % SLOTS) * kStreamChunkBytes + m * 128);
      const uint32_t sw = wl_addr + (uint32_t)((m * stride + c * 64 + h * (ANY ? 32 : 8)) * 2);
      u32x4_t a[4], b[4];
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) {
        asm volatile("ds_read_b128 %0, %1" : "=v"(a[ks]) : "v"(sa + (uint32_t)(((ANY ? h * 4 + ks : 2 * ks + h) ^ swz) * 16)));
        asm volatile("ds_read_b128 %0, %1" : "=v"(b[ks]) : "v"(sw + (uint32_t)(ks * (ANY ? 16 : 32))));
      }
      asm volatile("s_waitcnt lgkmcnt(0)"
                   : "+v"(a[0]), "+v"(a[1]), "+v"(a[2]), "+v"(a[3]), "+v"(b[0]), "+v"(b[1]), "+v"(b[2]), "+v"(b[3]));
#pragma unroll
      for (int ks = 0; ks < 4; ++ks)
        acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a[ks]),
                                                      __builtin_bit_cast(bf16x8, b[ks]), acc, 0, 0, 0);
    };
    int c = 0;
    for (; c + SLOTS - 1 < nchunks; ++c) {       // chunk c + SLOTS - 1 goes into the slot chunk c - 1 has left
      request(c + SLOTS - 1);
      wait_vmcnt<(SLOTS - 1) * 4>();
      multiply(c);
    }
    wait_vmcnt<0>();
    for (; c < nchunks; ++c) multiply(c);
    mfma_result_fence();

    // Epilogue (gate_topk_kernel's, for one tile of experts): logits through a wave-private
    // LDS tile so that a lane ends up with half of one item's row.
    float* st = reinterpret_cast<float*>(ring);
    {
      const float bn = (bias != nullptr && m < E) ? bias[m] : 0.f;
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int rl = (i >> 2) * 8 + h * 4 + (i & 3);
        float v = bf16r(acc[i]);
        if (bias != nullptr) v = bf16r(v + bn);
        st[rl * (EP + 1) + m] = v;
      }
    }
    finish_tile32(st, gates, topk_val, topk_idx, row0, num_items, E, K, m, h);
  }
#endif
}

// bfloat16, up to 32 experts, fewer tiles of items than CUs: a workgroup per tile of 32 items, the k
// range dealt to its waves in slices of 128, so that a launch is one trip to memory.  A wave loads its
// rows' slices in fragment order and, at the same time, an 8 (k) x 8 (expert) block of the router kernel
// per lane, which it transposes into its own piece of LDS (no barrier before the products); the waves'
// logits meet in LDS, added in wave order, and wave 0 finishes the tile.  gate_topk_kernel walks all of
// k in one wave per tile on a quarter of the workgroups, and stages the router kernel in two rounds.
// Bound by that trip and by wave 0's serial epilogue.  D = 768, 7 to 255 tiles: 7.8 us against 13.6 of
// gate_topk_kernel; D = 1024: 8.5 against 15.5.
constexpr int kSplitWaves = 8;
constexpr int kSplitSlice = 128;                       // k per wave and round
constexpr int kSplitStride = kSplitSlice + 8;          // elements per expert of a staged slice
constexpr int kSplitWaveBytes = 32 * kSplitStride * 2; // also holds the wave's 32 x 33 logits

__global__ __launch_bounds__(kSplitWaves * kWave, 1) void gate_topk_split_kernel(
    const bf16_t* __restrict__ x, const bf16_t* __restrict__ w, const float* __restrict__ bias,
    bf16_t* __restrict__ gates, float* __restrict__ topk_val, int32_t* __restrict__ topk_idx,
    int num_items, int D, int E, int K) {
  extern __shared__ __align__(16) unsigned char smem[];
  constexpr int EP = 32;
  static_assert(kSplitWaveBytes >= 32 * (EP + 1) * (int)sizeof(float), "the logits fit a wave's piece");
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, waves = blockDim.x >> 6;
  const int m = lane & 31, h = lane >> 5;
  const int row0 = blockIdx.x * 32;
  const bf16_t* xrow = x + (size_t)min(row0 + m, num_items - 1) * D;
  bf16_t* wl = reinterpret_cast<bf16_t*>(smem + wave * kSplitWaveBytes);
  const int kb = lane >> 2, nb = lane & 3;             // this lane's block of the router kernel

  floatx16 acc;
#pragma unroll
  for (int i = 0; i < 16; ++i) acc[i] = 0.f;
  for (int k0 = wave * kSplitSlice; k0 < D; k0 += waves * kSplitSlice) {
    uint4 wraw[8], a[2][4];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int k = k0 + kb * 8 + i;
      wraw[i] = make_uint4(0, 0, 0, 0);
      if (k < D && nb * 8 < E) wraw[i] = *reinterpret_cast<const uint4*>(w + (size_t)k * E + nb * 8);
    }
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int kg = k0 + u * 64 + h * 32 + j * 8;
        a[u][j] = make_uint4(0, 0, 0, 0);
        if (kg < D) a[u][j] = *reinterpret_cast<const uint4*>(xrow + kg);
      }
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const uint32_t sel = (j & 1) ? 0x07060302u : 0x05040100u;
      uint32_t o[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const uint32_t hi = reinterpret_cast<const uint32_t*>(&wraw[2 * q + 1])[j >> 1];
        const uint32_t lo = reinterpret_cast<const uint32_t*>(&wraw[2 * q])[j >> 1];
        o[q] = __builtin_amdgcn_perm(hi, lo, sel);
      }
      *reinterpret_cast<uint4*>(wl + (nb * 8 + j) * kSplitStride + kb * 8) = make_uint4(o[0], o[1], o[2], o[3]);
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); // the other lanes' blocks are read from here on
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const uint4 b = *reinterpret_cast<const uint4*>(wl + m * kSplitStride + u * 64 + h * 32 + j * 8);
        acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a[u][j]),
                                                      __builtin_bit_cast(bf16x8, b), acc, 0, 0, 0);
      }
    mfma_result_fence();
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); // and overwritten from here on
  }
  float* st = reinterpret_cast<float*>(wl);
#pragma unroll
  for (int i = 0; i < 16; ++i) st[((i >> 2) * 8 + h * 4 + (i & 3)) * (EP + 1) + m] = acc[i];
  __syncthreads();
  for (int e = threadIdx.x; e < 32 * EP; e += blockDim.x) {
    const int n = e & (EP - 1), at = (e >> 5) * (EP + 1) + n;
    float v = reinterpret_cast<const float*>(smem)[at];
    for (int ww = 1; ww < waves; ++ww) v += reinterpret_cast<const float*>(smem + ww * kSplitWaveBytes)[at];
    v = bf16r(v);
    if (bias != nullptr && n < E) v = bf16r(v + bias[n]);
    reinterpret_cast<float*>(smem)[at] = v;
  }
  __syncthreads();
  if (wave == 0)
    finish_tile32(reinterpret_cast<const float*>(smem), gates, topk_val, topk_idx, row0, num_items, E, K, m, h);
}

// bfloat16, fewer tiles of items than CUs, up to 64 experts (any number), any width: a workgroup of eight waves
// per tile of 32 items.  All of them fetch the item rows and the router kernel (KC columns of each) into LDS in
// one trip to memory; a wave per 32 experts multiplies, in gate_topk_kernel's order of k (same sums bit for
// bit), and wave 0 finishes the tile.  gate_topk_kernel walks k in one wave per tile on a quarter of the
// workgroups, with a scalar staging loop where E is no multiple of 8: 870 items x 1 024, 6 experts: 29 us to 9.7;
// 3 000 x 768, 50 experts: 44 to 15.
constexpr int kTileWaves = 8;

template <int NT>
__global__ __launch_bounds__(kTileWaves * kWave) void gate_topk_tile_kernel(
    const bf16_t* __restrict__ x, const bf16_t* __restrict__ w, const float* __restrict__ bias,
    bf16_t* __restrict__ gates, float* __restrict__ logits, float* __restrict__ topk_val,
    int32_t* __restrict__ topk_idx, int num_items, int D, int E, int K, int KC, int num_chunks, int x_off) {
  extern __shared__ __align__(16) unsigned char smem[];
  constexpr int EP = NT * 32, kThreads = kTileWaves * kWave, kBatch = 8;
  bf16_t* const wl = reinterpret_cast<bf16_t*>(smem);              // [EP][KC + 8]
  bf16_t* const xs = reinterpret_cast<bf16_t*>(smem + x_off);      // [32][KC + 8], later the logits [32][EP + 1]
  float* const st = reinterpret_cast<float*>(smem + x_off);
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int m = lane & 31, h = lane >> 5, stride = KC + 8;
  const int row0 = blockIdx.x * 32;
  const bool blocks8 = E % 8 == 0 && (reinterpret_cast<uintptr_t>(w) & 15u) == 0;
  floatx16 acc;
#pragma unroll
  for (int i = 0; i < 16; ++i) acc[i] = 0.f;
  for (int c = 0; c < num_chunks; ++c) {
    const int k0 = c * KC, per_row = KC / 8, pieces = 32 * per_row;
    uint4 raw[kBatch];
    auto load_x = [&](int p0) {
#pragma unroll
      for (int t = 0; t < kBatch; ++t) {
        const int p = min(p0 + t * kThreads, pieces - 1), r = p / per_row, k = k0 + (p - r * per_row) * 8;
        raw[t] = *reinterpret_cast<const uint4*>(x + (size_t)min(row0 + r, num_items - 1) * D + min(k, D - 8));
        if (k >= D) raw[t] = make_uint4(0, 0, 0, 0);
      }
    };
    auto store_x = [&](int p0) {
#pragma unroll
      for (int t = 0; t < kBatch; ++t) {
        const int p = min(p0 + t * kThreads, pieces - 1), r = p / per_row;   // (past the end: the last piece again)
        *reinterpret_cast<uint4*>(xs + r * stride + (p - r * per_row) * 8) = raw[t];
      }
    };
    load_x(tid);
    if (c > 0) __syncthreads();                   // the chunk before has been read
    if (blocks8) {
      const int nbn = E / 8, nblk = per_row * nbn;
      for (int b = tid; b < nblk; b += kThreads) {
        const int kb = b / nbn, nb = b - kb * nbn;
        uint4 wraw[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          const int k = k0 + kb * 8 + i;
          wraw[i] = k < D ? *reinterpret_cast<const uint4*>(w + (size_t)k * E + nb * 8) : make_uint4(0, 0, 0, 0);
        }
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          const uint32_t sel = (j & 1) ? 0x07060302u : 0x05040100u;
          uint32_t o[4];
#pragma unroll
          for (int q = 0; q < 4; ++q)
            o[q] = __builtin_amdgcn_perm(reinterpret_cast<const uint32_t*>(&wraw[2 * q + 1])[j >> 1],
                                         reinterpret_cast<const uint32_t*>(&wraw[2 * q])[j >> 1], sel);
          *reinterpret_cast<uint4*>(wl + (nb * 8 + j) * stride + kb * 8) = make_uint4(o[0], o[1], o[2], o[3]);
        }
      }
    } else {
      stage_router_any(w, wl, stride, k0, KC, D, E, tid, kThreads);
    }
    store_x(tid);
    for (int p0 = tid + kBatch * kThreads; p0 < pieces; p0 += kBatch * kThreads) {
      load_x(p0);
      store_x(p0);
    }
    __syncthreads();
    if (wave < NT) {
      const bf16_t* const a = xs + m * stride + h * 32;
      const bf16_t* const b = wl + (wave * 32 + m) * stride + h * 32;
      for (int kb = 0; kb < KC; kb += 64)
#pragma unroll
        for (int j = 0; j < 4; ++j)
          acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(*reinterpret_cast<const bf16x8*>(a + kb + j * 8),
                                                        *reinterpret_cast<const bf16x8*>(b + kb + j * 8), acc, 0, 0, 0);
      mfma_result_fence();
    }
  }
  __syncthreads();                                // the rows' LDS takes the logits
  if (wave < NT) {
    const int n = wave * 32 + m;
    const float bn = (bias != nullptr && n < E) ? bias[n] : 0.f;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      float v = bf16r(acc[i]);
      if (bias != nullptr) v = bf16r(v + bn);
      st[((i >> 2) * 8 + h * 4 + (i & 3)) * (EP + 1) + n] = v;
    }
  }
  __syncthreads();
  if (wave == 1 && logits != nullptr) store_logits(st, EP + 1, logits, row0, num_items, E, lane);
  if (wave == 0) {
    float g[EP / 2];
#pragma unroll
    for (int j = 0; j < EP / 2; ++j) g[j] = st[m * (EP + 1) + h * (EP / 2) + j];
    finish_row<bf16_t, EP>(g, gates, topk_val, topk_idx, row0 + m, num_items, E, K, h);
  }
}

// Top-K of given float32 gates, one wave per item, E <= 1024.
__global__ __launch_bounds__(256) void topk_kernel(const float* __restrict__ gates,
                                                   float* __restrict__ topk_val,
                                                   int32_t* __restrict__ topk_idx,
                                                   int num_items, int E, int K) {
  const int lane = threadIdx.x & 63;
  const int item = blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
  if (item >= num_items) return;
  const float* g = gates + (size_t)item * E;
  float v[16];
#pragma unroll
  for (int j = 0; j < 16; ++j) {
    int n = j * 64 + lane;
    v[j] = n < E ? g[n] : 0.f;
  }
  uint32_t taken = 0;
  for (int kk = 0; kk < K; ++kk) {
    uint64_t best = 0;
#pragma unroll
    for (int j = 0; j < 16; ++j) {
      int n = j * 64 + lane;
      if (n < E && !(taken >> j & 1u)) {
        uint64_t key = ((uint64_t)orderable(v[j]) << 32) | (uint32_t)(0xFFFFFFFFu - (uint32_t)n);
        best = key > best ? key : best;
      }
    }
#pragma unroll
    for (int msk = 1; msk < 64; msk <<= 1) {
      uint32_t lo = __shfl_xor((uint32_t)best, msk, kWave);
      uint32_t hi = __shfl_xor((uint32_t)(best >> 32), msk, kWave);
      uint64_t o = ((uint64_t)hi << 32) | lo;
      best = o > best ? o : best;
    }
    const int n_star = (int)(0xFFFFFFFFu - (uint32_t)best);
    if ((n_star & 63) == lane) taken |= 1u << (n_star >> 6);
    if (lane == 0) {
      // Return the stored bits of the winner (keeps -0.0 / payloads intact).
      topk_val[(size_t)item * K + kk] = g[n_star];
      topk_idx[(size_t)item * K + kk] = n_star;
    }
  }
}

// Per-group auxiliary losses: one workgroup of 1024 threads per group (router_metrics.h).
template <typename T>
__global__ __launch_bounds__(kMetricThreads) void router_metrics_kernel(
    const T* __restrict__ gates, const int32_t* __restrict__ top1, float* __restrict__ imp_loss,
    float* __restrict__ gsh_loss, float* __restrict__ aux_loss, float w_gsh, float w_imp,
    int S, int E, int top1_stride, int V) {
  extern __shared__ __align__(16) unsigned char smem[];
  router_metrics_group<T>(gates, top1, imp_loss, gsh_loss, aux_loss, w_gsh, w_imp, S, E,
                          top1_stride, V, blockIdx.x, smem);
}

int launch_gate_f32(const VmoeGateTopkParams* p, hipStream_t stream) {
  const int nt = (p->E + 31) / 32 == 3 ? 4 : (p->E + 31) / 32, ep = nt * 32;
  const int num_tiles = (p->num_items + 31) / 32;
  // Tiles per workgroup: one workgroup per CU as long as that leaves a wave per tile.
  const int per_cu = (num_tiles + kNumCus - 1) / kNumCus;
  const int waves = nt == 4 ? 4 : 8, tw = nt == 4 ? 1 : per_cu <= 1 ? 1 : per_cu <= 2 ? 2 : per_cu <= 4 ? 4 : 8;
  const int gran = 16 * waves, dpad = (p->D + gran - 1) / gran * gran;
  const int most = (156 * 1024 / (ep * 6) - 8) / gran * gran;        // rows of W whose planes fit
  const int num_chunks = (dpad + most - 1) / most;
  const int kc = ((dpad + num_chunks - 1) / num_chunks + gran - 1) / gran * gran;
  const size_t lds = std::max((size_t)ep * (kc + 8) * 6, (size_t)waves * 32 * (ep + 1) * sizeof(float));
  const int blocks = std::min((num_tiles + tw - 1) / tw, 1024);
  auto run = [&](auto kern) {
    hipError_t e = allow_dynamic_lds(reinterpret_cast<const void*>(kern), lds);
    if (e != hipSuccess) return (int)e;
    hipLaunchKernelGGL(kern, dim3(blocks), dim3(waves * kWave), lds, stream, (const float*)p->x, (const float*)p->w,
                       p->logit_bias, (float*)p->gates, p->logits, p->topk_val, p->topk_idx, p->num_items, p->D, p->E,
                       p->K, kc, num_chunks, num_tiles);
    return launch_status();
  };
  if (nt == 1) {
    switch (tw) {
      case 1: return run(gate_topk_f32_kernel<1, 8, 1>);
      case 2: return run(gate_topk_f32_kernel<1, 8, 2>);
      case 4: return run(gate_topk_f32_kernel<1, 8, 4>);
      default: return run(gate_topk_f32_kernel<1, 8, 8>);
    }
  }
  if (nt == 2) {
    switch (tw) {
      case 1: return run(gate_topk_f32_kernel<2, 8, 1>);
      case 2: return run(gate_topk_f32_kernel<2, 8, 2>);
      case 4: return run(gate_topk_f32_kernel<2, 8, 4>);
      default: return run(gate_topk_f32_kernel<2, 8, 8>);
    }
  }
  return run(gate_topk_f32_kernel<4, 4, 1>);
}

int launch_gate_bf16(const VmoeGateTopkParams* p, hipStream_t stream) {
  using T = bf16_t;
  const int nt = (p->E + 31) / 32;
  const int ep = (nt == 3 ? 4 : nt) * 32;
  constexpr int gran = 64;
  const int dpad = (p->D + gran - 1) / gran * gran;
  // LDS: the staged router kernel (split along D when it would not fit) and,
  // behind it, a 32 x (ep + 1) float32 logits tile per wave for the epilogue.
  // (33 .. 64 experts: one workgroup fits a CU either way, and a whole router kernel is staged once)
  const size_t budget = (nt == 2 ? 120 : 88) * 1024;
  int kc = dpad;
  while ((size_t)ep * (kc + 8) * sizeof(T) > budget && kc > gran) kc = ((kc / 2) + gran - 1) / gran * gran;
  const int num_chunks = (dpad + kc - 1) / kc;
  const size_t w_bytes = ((size_t)ep * (kc + 8) * sizeof(T) + 15) / 16 * 16;
  // Two workgroups of four waves per CU, each with its own staged copy of the router
  // kernel, where both copies fit in LDS; one workgroup of eight waves sharing a copy
  // where they do not (D = 1024), the registers allow it (up to 32 experts) and
  // four-wave workgroups would not all be resident at once anyway.
  const size_t tile_bytes = (size_t)32 * (ep + 1) * sizeof(float);
  const size_t lds_cu = 160 * 1024;
  const int num_tiles = (p->num_items + 31) / 32;
  const int waves = (nt == 1 && 2 * (w_bytes + 4 * tile_bytes) > lds_cu &&
                     w_bytes + 8 * tile_bytes <= lds_cu && num_tiles > 4 * 256) ? 8 : 4;
  const size_t stage_bytes = waves * tile_bytes;
  const size_t lds = w_bytes + stage_bytes;
  int blocks = (num_tiles + waves - 1) / waves;
  if (blocks > 1024) blocks = 1024;
  // bfloat16, up to 32 experts, no logits output, enough items to fill the chip: the
  // streaming kernel (coalesced DMA requests into wave-private LDS rings).
  {
    const size_t stream_w = ((size_t)32 * (p->D + 8) * 2 + 1023) / 1024 * 1024;
    const size_t ring3 = (size_t)kStreamWaves * 3 * kStreamChunkBytes, ring2 = (size_t)kStreamWaves * 2 * kStreamChunkBytes;
    const bool direct = getenv("VMOE_GATE_DIRECT_LOADS") != nullptr;
    const bool whole = p->E % 8 == 0 && aligned16(p->w);      // the router kernel comes in blocks of 8 x 8
    const bool simple = nt == 1 && p->logits == nullptr && whole && p->D % 64 == 0 && !direct;
    const bool stream_ok = nt == 1 && p->logits == nullptr && p->D % 64 == 0 && !direct &&
                           (int64_t)p->num_items * p->D * 2 < ((int64_t)1 << 32) &&
                           num_tiles >= 256 && stream_w + ring2 <= lds_cu;
    // Fewer tiles than CUs: the waves of a tile share its k range (255 tiles x 768: 8.0 us against 13.8
    // with direct loads).  Beyond, a CU runs two such workgroups, each with its own copy of the router
    // kernel, and the streaming form is level (300 to 512 tiles: 10.5 both) or faster (1 152: 24 to 15).
    if (simple && num_tiles < 256) {
      const int swaves = std::min((p->D + kSplitSlice - 1) / kSplitSlice, kSplitWaves);
      const size_t split_lds = (size_t)swaves * kSplitWaveBytes;
      hipError_t e = allow_dynamic_lds(reinterpret_cast<const void*>(gate_topk_split_kernel), split_lds);
      if (e != hipSuccess) return (int)e;
      hipLaunchKernelGGL(gate_topk_split_kernel, dim3(num_tiles), dim3(swaves * kWave), split_lds, stream,
                         (const bf16_t*)p->x, (const bf16_t*)p->w, p->logit_bias, (bf16_t*)p->gates,
                         p->topk_val, p->topk_idx, p->num_items, p->D, p->E, p->K);
      return launch_status();
    }
    if (nt <= 2 && num_tiles < 256 && !direct) {
      const int most = (int)((150 * 1024) / ((ep + 32) * sizeof(T)) - 8) / 64 * 64;
      const int chunks = (dpad + most - 1) / most, tkc = ((dpad + chunks - 1) / chunks + 63) / 64 * 64;
      const size_t x_off = (size_t)ep * (tkc + 8) * sizeof(T);
      const size_t tile_lds = x_off + std::max((size_t)32 * (tkc + 8) * sizeof(T), tile_bytes);
      auto trun = [&](auto kern) {
        hipError_t e = allow_dynamic_lds(reinterpret_cast<const void*>(kern), tile_lds);
        if (e != hipSuccess) return (int)e;
        hipLaunchKernelGGL(kern, dim3(num_tiles), dim3(kTileWaves * kWave), tile_lds, stream, (const T*)p->x,
                           (const T*)p->w, p->logit_bias, (T*)p->gates, p->logits, p->topk_val, p->topk_idx,
                           p->num_items, p->D, p->E, p->K, tkc, chunks, (int)x_off);
        return launch_status();
      };
      return nt == 1 ? trun(gate_topk_tile_kernel<1>) : trun(gate_topk_tile_kernel<2>);
    }
    if (stream_ok) {
      const bool three = stream_w + ring3 <= lds_cu;
      const size_t stream_lds = stream_w + (three ? ring3 : ring2);
      constexpr int swaves = kStreamWaves;
      int sblocks = (num_tiles + swaves - 1) / swaves;
      if (sblocks > 256) sblocks = 256;
      auto srun = [&](auto kern) {
        hipError_t e = allow_dynamic_lds(reinterpret_cast<const void*>(kern), stream_lds);
        if (e != hipSuccess) return (int)e;
        hipLaunchKernelGGL(kern, dim3(sblocks), dim3(swaves * kWave), stream_lds, stream,
                           (const bf16_t*)p->x, (const bf16_t*)p->w, p->logit_bias, (bf16_t*)p->gates,
                           p->topk_val, p->topk_idx, p->num_items, p->D, p->E, p->K, num_tiles,
                           (int)stream_w);
        return launch_status();
      };
      if (!whole) return three ? srun(gate_topk_stream_kernel<3, 8, true>) : srun(gate_topk_stream_kernel<2, 8, true>);
      return three ? srun(gate_topk_stream_kernel<3, 8, false>) : srun(gate_topk_stream_kernel<2, 8, false>);
    }
  }
  auto run = [&](auto kern) {
    hipError_t e = allow_dynamic_lds(reinterpret_cast<const void*>(kern), lds);
    if (e != hipSuccess) return (int)e;
    hipLaunchKernelGGL(kern, dim3(blocks), dim3(waves * kWave), lds, stream,
                       (const T*)p->x, (const T*)p->w, p->logit_bias, (T*)p->gates, p->logits,
                       p->topk_val, p->topk_idx, p->num_items, p->D, p->E, p->K, kc, num_chunks, num_tiles,
                       (int)w_bytes);
    return launch_status();
  };
  // The logits output is a separate instantiation: its extra live pointer costs
  // the common one a wave of occupancy.
  if (p->logits != nullptr) {
    switch (nt) {
      case 1: return waves == 8 ? run(gate_topk_kernel<1, true, 8>) : run(gate_topk_kernel<1, true, 4>);
      case 2: return run(gate_topk_kernel<2, true, 4>);
      default: return run(gate_topk_kernel<4, true, 4>);
    }
  }
  switch (nt) {
    case 1: return waves == 8 ? run(gate_topk_kernel<1, false, 8>) : run(gate_topk_kernel<1, false, 4>);
    case 2: return run(gate_topk_kernel<2, false, 4>);
    default: return run(gate_topk_kernel<4, false, 4>);
  }
}


// Noisy branch of the routers (vmoe/nn/routing.py:92-114): softmax of the noisy
// logits and, per group, the load loss (vmoe/nn/routing.py:159-183).  One
// workgroup per group, a wave per item, a lane per expert (two for E > 64).
constexpr int kNoisyWaves = 8;

__device__ __forceinline__ float wave_max_f(float v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o, kWave));
  return v;
}
__device__ __forceinline__ float wave_sum_f(float v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, kWave);
  return v;
}
__device__ __forceinline__ uint64_t wave_max_u64(uint64_t v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    const uint32_t lo = __shfl_xor((uint32_t)v, o, kWave);
    const uint32_t hi = __shfl_xor((uint32_t)(v >> 32), o, kWave);
    const uint64_t other = ((uint64_t)hi << 32) | lo;
    v = other > v ? other : v;
  }
  return v;
}

__global__ __launch_bounds__(kNoisyWaves * 64) void noisy_gates_kernel(
    const float* __restrict__ logits, const float* __restrict__ noise,
    float* __restrict__ gates, float* __restrict__ load_loss, int S, int E, int K,
    float noise_std) {
  __shared__ float psum[kNoisyWaves][128];
  const int g = blockIdx.x;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const bool has0 = lane < E, has1 = lane + 64 < E;
  const float inv = 1.0f / (noise_std * 1.41421356237309515f);
  float acc0 = 0.f, acc1 = 0.f;
  for (int s = wave; s < S; s += kNoisyWaves) {
    const size_t base = ((size_t)g * S + s) * E;
    const float l0 = has0 ? logits[base + lane] : 0.f;
    const float l1 = has1 ? logits[base + lane + 64] : 0.f;
    const float v0 = has0 ? l0 + noise_std * noise[base + lane] : -INFINITY;
    const float v1 = has1 ? l1 + noise_std * noise[base + lane + 64] : -INFINITY;
    const float mx = wave_max_f(fmaxf(v0, v1));
    const float e0 = has0 ? expf(v0 - mx) : 0.f;
    const float e1 = has1 ? expf(v1 - mx) : 0.f;
    const float sum = wave_sum_f(e0 + e1);
    if (has0) gates[base + lane] = e0 / sum;
    if (has1) gates[base + lane + 64] = e1 / sum;
    if (load_loss == nullptr) continue;
    // Value of the K-th largest noisy logit (lax.top_k order: equal values, lower index first).
    uint64_t k0 = has0 ? (((uint64_t)orderable(v0) << 32) | (0xFFFFFFFFu - (uint32_t)lane)) : 0;
    uint64_t k1 = has1 ? (((uint64_t)orderable(v1) << 32) | (0xFFFFFFFFu - (uint32_t)(lane + 64))) : 0;
    uint64_t best = 0;
    for (int kk = 0; kk < K; ++kk) {
      best = wave_max_u64(k0 > k1 ? k0 : k1);
      if (best == k0) k0 = 0;
      else if (best == k1) k1 = 0;
    }
    const float thr = inv_orderable((uint32_t)(best >> 32));
    // p = 1 - Phi(z) = erfc(z / sqrt(2)) / 2,  z = (thr - logit) / noise_std.
    if (has0) acc0 += 0.5f * erfcf((thr - l0) * inv);
    if (has1) acc1 += 0.5f * erfcf((thr - l1) * inv);
  }
  if (load_loss == nullptr) return;
  psum[wave][lane] = acc0;
  psum[wave][lane + 64] = acc1;
  __syncthreads();
  if (wave == 0) {
    float p0 = 0.f, p1 = 0.f;
#pragma unroll
    for (int w = 0; w < kNoisyWaves; ++w) {
      p0 += psum[w][lane];
      p1 += psum[w][lane + 64];
    }
    p0 = has0 ? p0 / (float)S : 0.f;
    p1 = has1 ? p1 / (float)S : 0.f;
    const float mean = wave_sum_f(p0 + p1) / (float)E;
    const float d0 = has0 ? p0 - mean : 0.f, d1 = has1 ? p1 - mean : 0.f;
    const float var = wave_sum_f(d0 * d0 + d1 * d1) / (float)E;
    if (lane == 0) load_loss[g] = var / (mean * mean);
  }
}

}  // namespace
}  // namespace vmoe

using namespace vmoe;

extern "C" int vmoe_gate_topk(const VmoeGateTopkParams* p, vmoe_stream_t stream) {
  if (p == nullptr || p->x == nullptr || p->w == nullptr || p->topk_val == nullptr ||
      p->topk_idx == nullptr)
    return VMOE_E_NULL;
  if (p->num_items < 1 || p->D < 1 || p->E < 1 || p->K < 1 || p->K > p->E) return VMOE_E_SHAPE;
  if (p->dtype != VMOE_F32 && p->dtype != VMOE_BF16) return VMOE_E_DTYPE;
  if (p->E > 128) return VMOE_E_UNSUPPORTED;
  const int vec = p->dtype == VMOE_BF16 ? 8 : 4;
  if (p->D % vec != 0 || !aligned16(p->x)) return VMOE_E_ALIGN;
  if ((int64_t)p->num_items * (p->D > p->E * p->K ? p->D : p->E * p->K) >= (int64_t)1 << 40)
    return VMOE_E_OVERFLOW;
  return p->dtype == VMOE_BF16 ? launch_gate_bf16(p, as_stream(stream))
                               : launch_gate_f32(p, as_stream(stream));
}

extern "C" int vmoe_topk(const VmoeTopkParams* p, vmoe_stream_t stream) {
  if (p == nullptr || p->gates == nullptr || p->topk_val == nullptr || p->topk_idx == nullptr)
    return VMOE_E_NULL;
  if (p->num_items < 1 || p->E < 1 || p->K < 1 || p->K > p->E) return VMOE_E_SHAPE;
  if (p->E > 1024) return VMOE_E_UNSUPPORTED;
  const int blocks = (p->num_items + 3) / 4;
  hipLaunchKernelGGL(topk_kernel, dim3(blocks), dim3(256), 0, as_stream(stream), p->gates,
                     p->topk_val, p->topk_idx, p->num_items, p->E, p->K);
  return launch_status();
}

extern "C" int vmoe_router_metrics(const VmoeRouterMetricsParams* p, vmoe_stream_t stream) {
  int rc = check_router_metrics(p);
  if (rc != VMOE_OK) return rc;
  int V;
  size_t lds;
  if (!router_metrics_geometry(p, &V, &lds)) return VMOE_E_UNSUPPORTED;
  if (p->dtype == VMOE_BF16)
    hipLaunchKernelGGL(router_metrics_kernel<bf16_t>, dim3(p->G), dim3(kMetricThreads), lds,
                       as_stream(stream), (const bf16_t*)p->gates, p->top1_idx, p->importance_loss,
                       p->gshard_loss, p->auxiliary_loss, p->gshard_loss_weight,
                       p->importance_loss_weight, p->S, p->E, p->top1_stride, V);
  else
    hipLaunchKernelGGL(router_metrics_kernel<float>, dim3(p->G), dim3(kMetricThreads), lds,
                       as_stream(stream), (const float*)p->gates, p->top1_idx, p->importance_loss,
                       p->gshard_loss, p->auxiliary_loss, p->gshard_loss_weight,
                       p->importance_loss_weight, p->S, p->E, p->top1_stride, V);
  return launch_status();
}

extern "C" int vmoe_noisy_gates(const VmoeNoisyGatesParams* p, vmoe_stream_t stream) {
  if (p == nullptr || p->logits == nullptr || p->noise == nullptr || p->gates_noisy == nullptr)
    return VMOE_E_NULL;
  if (p->G < 1 || p->S < 1 || p->E < 1 || p->K < 1 || p->K > p->E || !(p->noise_std > 0.f))
    return VMOE_E_SHAPE;
  if (p->E > 128) return VMOE_E_UNSUPPORTED;
  hipLaunchKernelGGL(noisy_gates_kernel, dim3(p->G), dim3(kNoisyWaves * 64), 0, as_stream(stream),
                     p->logits, p->noise, p->gates_noisy, p->load_loss, p->S, p->E, p->K,
                     p->noise_std);
  return launch_status();
}
