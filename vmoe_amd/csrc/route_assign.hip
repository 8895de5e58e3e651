// Capacity-bounded slot assignment with Batch Priority Routing for gfx950.
//
// Replaces vmoe/moe.py:568-589 (+ :646-648): the reference sorts items by their
// first-choice gate, flattens the (K, S) choices K-major, takes a one-hot over
// experts and a cumulative sum down the K*S rows.  Here one workgroup owns a
// group and works entirely in LDS:
//   1. 64-bit keys (descending-gate order bits << 32 | item) are bitonic-sorted;
//      the item index in the low word makes the order stable by construction.
//      The keys stay in registers (R consecutive keys per thread): exchanges at
//      distances below R are register moves, below 64*R lane exchanges, and only
//      the few stages beyond that go through LDS with barriers;
//   2. every (item, choice) sets bit  k*S + rank(item)  in its expert's bitmap
//      (integer LDS atomics: order-independent result);
//   3. an exclusive prefix of per-word popcounts turns "how many set bits come
//      before mine" -- the cumsum of the one-hot column -- into one table
//      lookup plus one masked popcount.
// The kernel also emits the two maps the data-movement kernels use: item ->
// slot row (-1 when over capacity) and slot row -> item (-1 when empty).
#include <mutex>
#include "vmoe_common.h"
#include "router_metrics.h"
#include "compact_rows.h"

namespace vmoe {
namespace {

constexpr int kRouteThreads = 1024;

__host__ __device__ inline int pow2ceil(int v) {
  int p = 1;
  while (p < v) p <<= 1;
  return p;
}

// One side of a compare-exchange: the smaller (take_min) or larger of two keys.
template <typename KeyT>
__device__ __forceinline__ KeyT pick(KeyT mine, KeyT other, bool take_min) {
  return ((other < mine) == take_min) ? other : mine;
}

__device__ __forceinline__ uint64_t lane_exchange(uint64_t v, int lane_xor) {
  return __shfl_xor((unsigned long long)v, lane_xor, kWave);
}
__device__ __forceinline__ uint32_t lane_exchange(uint32_t v, int lane_xor) {
  return __shfl_xor(v, lane_xor, kWave);
}

template <int R, int ST, typename KeyT>
__device__ __forceinline__ void bitonic_in_thread(KeyT (&key)[R], int size, int tid) {
#pragma unroll
  for (int r = 0; r < R; ++r) {
    if ((r & ST) == 0 && r + ST < R) {
      const bool up = (((tid * R + r) & size) == 0);
      const KeyT a = key[r], b = key[r + ST];
      const bool swap = (b < a) == up;
      key[r] = swap ? b : a;
      key[r + ST] = swap ? a : b;
    }
  }
}

// Ascending bitonic sort of SP (a power of two) keys, element tid*R + r in key[r] of
// thread tid < nact = SP / R.  Every thread of the workgroup calls it (the LDS stages
// have barriers); `xch` holds SP keys.
template <int R, typename KeyT>
__device__ __forceinline__ void bitonic_sort_regs(KeyT (&key)[R], KeyT* xch, int SP, int tid,
                                                  int nact) {
  const bool act = tid < nact;
  for (int size = 2; size <= SP; size <<= 1) {
    for (int stride = size >> 1; stride > 0; stride >>= 1) {
      if (stride >= 64 * R) {
        if (act) {
#pragma unroll
          for (int r = 0; r < R; ++r) xch[tid * R + r] = key[r];
        }
        __syncthreads();
        if (act) {
#pragma unroll
          for (int r = 0; r < R; ++r) {
            const int i = tid * R + r;
            key[r] = pick<KeyT>(key[r], xch[i ^ stride], ((i & stride) == 0) == ((i & size) == 0));
          }
        }
        __syncthreads();
      } else if (!act) {
        continue;
      } else if (stride >= R) {
        const int lane_xor = stride / R;
#pragma unroll
        for (int r = 0; r < R; ++r) {
          const int i = tid * R + r;
          const KeyT other = lane_exchange(key[r], lane_xor);
          key[r] = pick(key[r], other, ((i & stride) == 0) == ((i & size) == 0));
        }
      } else {
        if constexpr (R > 4) { if (stride == 4) bitonic_in_thread<R, 4, KeyT>(key, size, tid); }
        if constexpr (R > 2) { if (stride == 2) bitonic_in_thread<R, 2, KeyT>(key, size, tid); }
        if constexpr (R > 1) { if (stride == 1) bitonic_in_thread<R, 1, KeyT>(key, size, tid); }
      }
    }
  }
}

// Keys per thread for a sort of SP keys: as many threads as the workgroup has take part
// (a stage costs a wave its shuffles and selects per key, so more waves with fewer keys
// are faster: eight keys on an eighth of the threads took 35 us where two keys on all
// take 25); 0 = the keys do not fit in the registers and are sorted in LDS.
inline int keys_per_thread(int SP) {
  const int r = SP <= kRouteThreads ? 1 : SP / kRouteThreads;
  return r <= 8 ? r : 0;
}

// The same sort with the keys resident in LDS (any SP).
__device__ __forceinline__ void bitonic_sort_lds(uint64_t* keys, int SP, int tid) {
  for (int size = 2; size <= SP; size <<= 1) {
    for (int stride = size >> 1; stride > 0; stride >>= 1) {
      for (int t = tid; t < (SP >> 1); t += kRouteThreads) {
        int lo = 2 * t - (t & (stride - 1));
        int hi = lo + stride;
        bool up = (lo & size) == 0;
        uint64_t a = keys[lo], b = keys[hi];
        if ((a > b) == up) { keys[lo] = b; keys[hi] = a; }
      }
      __syncthreads();
    }
  }
}

constexpr int kHeld = 8;           // choices of a thread kept in registers
constexpr int kRankBins = 1024;    // bins of the counting rank: gates from 1 down to 2^-8
constexpr uint32_t kLongestBin = 512;

template <int R>
__device__ __forceinline__ void route_assign_group(
    const float* __restrict__ topk_val, const int32_t* __restrict__ topk_idx,
    int32_t* __restrict__ indices, int32_t* __restrict__ token_slot,
    int32_t* __restrict__ slot_token, int32_t* __restrict__ fill, int G, int S, int E, int K,
    int C, int bpr, int SP, int NK, int W, int g, unsigned char* smem) {
  // Layout: keys[NK] (u64, only with bpr) | bitmap[E*W] | prefix[E*W] | rank[S] | total[E]
  uint64_t* keys = reinterpret_cast<uint64_t*>(smem);
  uint32_t* bitmap = reinterpret_cast<uint32_t*>(smem + (bpr ? (size_t)NK * 8 : 0));
  uint32_t* prefix = bitmap + (size_t)E * W;
  int32_t* rank = reinterpret_cast<int32_t*>(prefix + (size_t)E * W);
  int32_t* total = rank + S;
  const int tid = threadIdx.x;
  const float* val = topk_val + (size_t)g * S * K;
  const int32_t* idx = topk_idx + (size_t)g * S * K;

  // The first kHeld choices of a thread are fetched together, before anything waits, and stay in
  // registers for both passes over them; only groups of more than kHeld * 1024 choices read the rest
  // from memory, twice.  (With that, and the segments' counts read four at a time: 17.6 -> 15.4 us for
  // 16 groups of 2 304 items with an unbalanced router, 13.3 -> 12.6 for 32 of 1 568.)
  const int SK = S * K;
  int held[kHeld], held_bit[kHeld];
#pragma unroll
  for (int j = 0; j < kHeld; ++j) {
    const int i = tid + j * kRouteThreads;
    held[j] = i < SK ? idx[i] : -1;
    held_bit[j] = 0;
  }
  auto item_of = [&](int i) { return K == 1 ? i : K == 2 ? i >> 1 : i / K; };

  for (int i = tid; i < E * W; i += kRouteThreads) bitmap[i] = 0u;
  if (bpr) {
    if constexpr (R == 0) {
      for (int s = tid; s < SP; s += kRouteThreads) {
        uint64_t key = ~0ull;
        if (s < S) key = bpr_key64(__builtin_bit_cast(uint32_t, val[(size_t)s * K]), s);
        keys[s] = key;
      }
      __syncthreads();
      bitonic_sort_lds(keys, SP, tid);
      for (int r = tid; r < S; r += kRouteThreads) rank[(uint32_t)keys[r]] = r;
    } else {
      // Gates that came out of a bfloat16 router are non-negative floats whose low 16
      // bits are zero: gate and item index then fit one 32-bit key (S <= 65536), and the
      // sort's compare-exchanges, which are what bounds this kernel, cost half as much.
      const int nact = SP / R;
      uint32_t bits[R];
      bool narrow_ok = S <= 65536;
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const int s = tid * R + r;
        bits[r] = (tid < nact && s < S) ? __builtin_bit_cast(uint32_t, val[(size_t)s * K]) : 0u;
        narrow_ok = narrow_ok && bpr_gate_is_narrow(bits[r]);
      }
      // Gates within a factor 2^8 of 1 (the largest gate of a softmax over up to 128
      // experts always is) fall into kRankBins bins by their high 16 bits, in descending order
      // as the bin number 0x3F80 - (bits >> 16) ascends (narrow gates of a bin are equal): the rank of
      // an item is then the number of items in lower bins plus the number of items of its own bin
      // with a lower bin_key32 -- a histogram, a prefix sum, a scatter into the bins' segments and a count
      // inside the item's own segment, four barriers in all, where the bitonic sort of 2 048 keys
      // takes 66 compare-exchange steps (15 of the kernel's 22 us on the headline layer; float32 gates,
      // 64-bit keys: 1 925 items x 4 of 7 experts 27 -> 17 us).
      // Every step counts, none depends on the order in which the threads arrive, so the
      // ranks are those of the sort.  The count is quadratic in a segment: where one holds more than
      // kLongestBin items (gates all equal, or float32 gates closer than 2^-8) the keys are sorted
      // after all, which takes about as long as counting one of that length.
      bool count_ok = S <= 65536;
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const uint32_t hi = bits[r] >> 16;
        if (tid < nact && tid * R + r < S) count_ok = count_ok && hi <= 0x3F80u && hi + kRankBins > 0x3F80u;
      }
      bool counted = __syncthreads_and(count_ok);
      if (counted) {
        uint32_t* hist = reinterpret_cast<uint32_t*>(keys);      // items per bin, then the bins' cursors
        uint32_t* start = hist + kRankBins;                      // first rank of each bin
        uint32_t* seg = start + kRankBins;                       // S keys, bin by bin
        for (int i = tid; i < kRankBins; i += kRouteThreads) hist[i] = 0u;
        __syncthreads();
        int bin[R];
#pragma unroll
        for (int r = 0; r < R; ++r) {
          bin[r] = (int)(0x3F80u - (bits[r] >> 16));
          if (tid < nact && tid * R + r < S) atomicAdd(&hist[bin[r]], 1u);
        }
        __syncthreads();
        // Exclusive prefix over the bins: kRankBins == kRouteThreads, one bin per thread.
        {
          static_assert(kRankBins == kRouteThreads, "one bin per thread");
          const int lane = tid & 63, wave = tid >> 6;
          const uint32_t c = hist[tid];
          uint32_t incl = c;
#pragma unroll
          for (int d = 1; d < 64; d <<= 1) {
            const uint32_t o = __shfl_up(incl, d, kWave);
            if (lane >= d) incl += o;
          }
          // A wave that saw a long bin says so in the top bit of its total (S is below it): a reduction over the
          // workgroup (__syncthreads_or) in place of this barrier made 32 x 1 568 items x 2 of 32 16.0 us in place of 14.5.
          __shared__ uint32_t wave_total[kRouteThreads / 64];
          const uint32_t long_bin = __any(c > kLongestBin) ? 0x80000000u : 0u;
          if (lane == 63) wave_total[wave] = incl | long_bin;
          __syncthreads();
          uint32_t before = 0, seen = 0;
#pragma unroll
          for (int w = 0; w < kRouteThreads / 64; ++w) {
            const uint32_t total = wave_total[w];
            seen |= total;
            before += w < wave ? total & 0x7fffffffu : 0u;
          }
          counted = (__builtin_amdgcn_readfirstlane((int)seen) & 0x80000000) == 0;
          start[tid] = before + incl - c;
          hist[tid] = before + incl - c;                       // cursor of the scatter
        }
        __syncthreads();
        if (counted) {
#pragma unroll
          for (int r = 0; r < R; ++r)
            if (tid < nact && tid * R + r < S) seg[atomicAdd(&hist[bin[r]], 1u)] = bin_key32(bits[r], tid * R + r);
          __syncthreads();
#pragma unroll
          for (int r = 0; r < R; ++r) {
            const int item = tid * R + r;
            if (tid >= nact || item >= S) continue;
            const uint32_t first = start[bin[r]], end = hist[bin[r]], mine = bin_key32(bits[r], item);
            uint32_t lower = 0;
            for (uint32_t q = first; q < end; q += 4)          // four reads in flight
#pragma unroll
              for (uint32_t u = 0; u < 4; ++u)
                lower += seg[min(q + u, end - 1)] < mine && q + u < end ? 1u : 0u;
            rank[item] = (int)(first + lower);
          }
        }
      }
      if (!counted && __syncthreads_and(narrow_ok)) {
        uint32_t key[R];
#pragma unroll
        for (int r = 0; r < R; ++r) {
          const int s = tid * R + r;
          key[r] = s < S ? bpr_key32(bits[r], s) : ~0u;
        }
        bitonic_sort_regs<R, uint32_t>(key, reinterpret_cast<uint32_t*>(keys), SP, tid, nact);
#pragma unroll
        for (int r = 0; r < R; ++r)
          if (tid < nact && tid * R + r < S) rank[key[r] & 0xffffu] = tid * R + r;
      } else if (!counted) {
        uint64_t key[R];
#pragma unroll
        for (int r = 0; r < R; ++r) {
          const int s = tid * R + r;
          key[r] = s < S ? bpr_key64(bits[r], s) : ~0ull;
        }
        bitonic_sort_regs<R, uint64_t>(key, keys, SP, tid, nact);
#pragma unroll
        for (int r = 0; r < R; ++r)
          if (tid < nact && tid * R + r < S) rank[(uint32_t)key[r]] = tid * R + r;
      }
    }
  } else {
    for (int s = tid; s < S; s += kRouteThreads) rank[s] = s;
  }
  __syncthreads();

  auto mark = [&](int i, int e) {
    if (e < 0 || e >= E) return 0;
    const int s = item_of(i);
    const int bit = choice_bit(i - s * K, S, rank[s]);
    atomicOr(&bitmap[(size_t)e * W + (bit >> 5)], 1u << (bit & 31));
    return bit;
  };
#pragma unroll
  for (int j = 0; j < kHeld; ++j)
    if (tid + j * kRouteThreads < SK) held_bit[j] = mark(tid + j * kRouteThreads, held[j]);
  for (int i = tid + kHeld * kRouteThreads; i < SK; i += kRouteThreads) mark(i, idx[i]);
  __syncthreads();
  // Exclusive prefix of popcounts per expert: one wave per expert, 64 words per step.
  {
    const int lane = tid & 63, wave = tid >> 6, nwaves = kRouteThreads >> 6;
    for (int e = wave; e < E; e += nwaves) {
      int carry = 0;
      for (int w0 = 0; w0 < W; w0 += 64) {
        int w = w0 + lane;
        int c = w < W ? __popc(bitmap[(size_t)e * W + w]) : 0;
        int incl = c;
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
          int o = __shfl_up(incl, d, kWave);
          if (lane >= d) incl += o;
        }
        if (w < W) prefix[(size_t)e * W + w] = (uint32_t)(carry + incl - c);
        carry += __shfl(incl, 63, kWave);
      }
      if (lane == 0) total[e] = carry;
    }
  }
  __syncthreads();

  auto emit = [&](int i, int e, int bit) {
    int pos = -1, slot = -1;
    if (e >= 0 && e < E) {
      const int w = bit >> 5;
      pos = position_from_bitmap(prefix[(size_t)e * W + w], bitmap[(size_t)e * W + w], bit);
      if (pos < C) {
        slot = slot_row(e, g, pos, G, E, C);
        slot_token[slot] = g * S + item_of(i);
      }
    }
    size_t o = (size_t)g * SK + i;
    indices[2 * o] = e;
    indices[2 * o + 1] = pos;
    token_slot[o] = slot;
  };
#pragma unroll
  for (int j = 0; j < kHeld; ++j)
    if (tid + j * kRouteThreads < SK) emit(tid + j * kRouteThreads, held[j], held_bit[j]);
  for (int i = tid + kHeld * kRouteThreads; i < SK; i += kRouteThreads) {
    const int e = idx[i], s = item_of(i);
    emit(i, e, choice_bit(i - s * K, S, rank[s]));
  }
  // Slots nobody claimed.
  for (int i = tid; i < E * C; i += kRouteThreads) {
    int e = i / C, c = i - e * C;
    if (c >= total[e]) slot_token[slot_row(e, g, c, G, E, C)] = -1;
  }
  if (fill != nullptr)
    for (int e = tid; e < E; e += kRouteThreads) fill[(size_t)g * E + e] = total[e] < C ? total[e] : C;
}

template <int R>
__global__ __launch_bounds__(kRouteThreads) void route_assign_kernel(
    const float* __restrict__ topk_val, const int32_t* __restrict__ topk_idx,
    int32_t* __restrict__ indices, int32_t* __restrict__ token_slot,
    int32_t* __restrict__ slot_token, int32_t* __restrict__ fill, int G, int S, int E, int K,
    int C, int bpr, int SP, int NK, int W) {
  extern __shared__ __align__(16) unsigned char smem[];
  route_assign_group<R>(topk_val, topk_idx, indices, token_slot, slot_token, fill, G, S, E, K, C,
                        bpr, SP, NK, W, blockIdx.x, smem);
}

// Slot assignment and the router's auxiliary losses in one launch: workgroups 0 .. G-1
// assign slots, workgroups G .. 2G-1 compute the losses of group blockIdx.x - G.  Both
// are one workgroup per group, bound by latency, and read the same top-k output, so side
// by side they take the time of the longer one.
template <int R, typename T>
__global__ __launch_bounds__(kRouteThreads) void route_assign_metrics_kernel(
    const float* __restrict__ topk_val, const int32_t* __restrict__ topk_idx,
    int32_t* __restrict__ indices, int32_t* __restrict__ token_slot,
    int32_t* __restrict__ slot_token, int32_t* __restrict__ fill, int G, int S, int E, int K,
    int C, int bpr, int SP, int NK, int W, RouterMetricsArgs m) {
  extern __shared__ __align__(16) unsigned char smem[];
  static_assert(kRouteThreads == kMetricThreads, "both roles use the launch's workgroup size");
  if ((int)blockIdx.x < G) {
    route_assign_group<R>(topk_val, topk_idx, indices, token_slot, slot_token, fill, G, S, E, K,
                          C, bpr, SP, NK, W, blockIdx.x, smem);
  } else {
    router_metrics_group<T>(static_cast<const T*>(m.gates), m.top1, m.imp_loss, m.gsh_loss,
                            m.aux_loss, m.w_gsh, m.w_imp, m.S, m.E, m.top1_stride, m.V,
                            (int)blockIdx.x - G, smem);
  }
}

// Experts-choice routing (vmoe/moe.py:655-694): every expert takes the C items
// with its largest gates (jax.lax.top_k over the transposed gates: descending,
// equal gates -> lower item index first).  The outputs are those of the
// slot-assignment kernel with one "choice" per expert (K = E), so the same
// dispatch / combine kernels serve both routing schemes.
//
// Two launches.  top_items_kernel ranks a column: one workgroup per (expert, group).
// Written from there, the item-major outputs would be three scattered stores per (item,
// expert), 4 or 8 bytes of a line each; so it leaves the ranks inside token_slot, each
// block of `chunk` items transposed (expert-major: runs of up to 256 bytes), and
// top_items_emit_kernel turns a block's ranks around in LDS and writes whole rows.
// 8 groups of 1 568 items, 32 experts, bfloat16: 35 us with scattered stores and the sort,
// 11 + 13 us this way (bound by latency).
struct TopItemsMetrics {
  int32_t* items_minmax;   // (2, G): fewest and most experts per item
  int32_t* counts;         // (num, G): items taken by at least 1, 2, 4, ... experts, and by all
  int num;
  int32_t* rows;           // (E,): G * C, or null
};

// Bins of the counting rank: the high halves of the floats from 1 down to 0.
constexpr int kGateBins = 16384;
static_assert(kGateBins > 0x3F80 && kGateBins % (kRouteThreads * 4) == 0, "whole 16-byte pieces per thread");
// Items of one gate that are counted rather than sorted: with 200 of them 8 x 1 568 x 32 takes 30 us
// (18 without, 32 sorted behind the histogram), 4 x 8 191 x 8 takes 68 (32, 90).  All gates equal,
// counted: 166 and 3 143 us.
constexpr uint32_t kLongestSegment = 256;
inline __host__ __device__ bool rank_by_counting(int SP) { return SP >= 512; }

template <typename T, int R>
__global__ __launch_bounds__(kRouteThreads) void top_items_kernel(
    const T* __restrict__ gates, int32_t* __restrict__ token_slot, int32_t* __restrict__ slot_token,
    float* __restrict__ sel_minmax, TopItemsMetrics m, int G, int S, int E, int C, int SP, int chunk) {
  extern __shared__ __align__(16) unsigned char smem[];
  uint64_t* keys = reinterpret_cast<uint64_t*>(smem);
  const int tid = threadIdx.x;
  const int e = blockIdx.x, g = blockIdx.y;
  const T* col = gates + (size_t)g * S * E + e;
  const int last = (C < S ? C : S) - 1;
  if (e == 0 && m.counts != nullptr) {      // what the next launch adds to
    if (tid < m.num) m.counts[(size_t)tid * G + g] = 0;
    if (tid == 0) {
      m.items_minmax[g] = INT32_MAX;
      m.items_minmax[G + g] = 0;
    }
  }
  if (g == 0 && tid == 0 && m.rows != nullptr) m.rows[e] = G * C;
  // Rank r of the column holds item s.
  auto emit = [&](int r, int s) {
    const int s0 = s & ~(chunk - 1);
    const int rows = min(chunk, S - s0);
    token_slot[((size_t)g * S + s0) * E + (size_t)e * rows + (s - s0)] = r;
    if (r < C) slot_token[slot_row(e, g, r, G, E, C)] = g * S + s;
    if (sel_minmax != nullptr && (r == last || r == 0)) {
      const float gate = Elt<T>::load(col + (size_t)s * E);
      if (r == last) sel_minmax[((size_t)g * E + e) * 2] = gate;
      if (r == 0) sel_minmax[((size_t)g * E + e) * 2 + 1] = gate;
    }
  };
  if constexpr (R == 0) {
    for (int s = tid; s < SP; s += kRouteThreads) {
      uint64_t key = ~0ull;
      if (s < S) key = bpr_key64(__builtin_bit_cast(uint32_t, Elt<T>::load(col + (size_t)s * E)), s);
      keys[s] = key;
    }
    __syncthreads();
    bitonic_sort_lds(keys, SP, tid);
    for (int r = tid; r < S; r += kRouteThreads) emit(r, (int)(uint32_t)keys[r]);
  } else {
    const int nact = SP / R;
    uint32_t bits[R];
    bool countable = true;
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int s = tid * R + r;
      bits[r] = (tid < nact && s < S) ? __builtin_bit_cast(uint32_t, Elt<T>::load(col + (size_t)s * E)) : 0u;
      countable = countable && bits[r] <= 0x3F800000u;       // 0 .. 1: not negative, not NaN
    }
    // Gates of a softmax fall into 0x3F81 bins by their high halves: rank by histogram, prefix, scatter
    // into the bins' segments and a count inside the item's own segment (see route_assign_group),
    // in place of 66 compare-exchange steps at 2 048 keys (float32, 65 x 268 items x 16: 29 -> 23 us).  Below 512 keys clearing the bins costs
    // what the sort does.  The count is quadratic in a segment: a column of equal gates (a router kernel
    // of zeros, tokens that repeat, gates that vanish) takes the sort after all.
    bool counted = rank_by_counting(SP) && __syncthreads_and(countable);
    if (counted) {
      uint32_t* hist = reinterpret_cast<uint32_t*>(smem);    // items per bin, then the bins' cursors
      uint32_t* seg = hist + kGateBins;                      // S keys, bin by bin
      constexpr int kPieces = kGateBins / kRouteThreads / 4; // 16-byte pieces of a thread's bins
      uint4* hist4 = reinterpret_cast<uint4*>(hist);
#pragma unroll
      for (int i = 0; i < kPieces; ++i) hist4[i * kRouteThreads + tid] = make_uint4(0, 0, 0, 0);
      __syncthreads();
#pragma unroll
      for (int r = 0; r < R; ++r)
        if (tid < nact && tid * R + r < S) atomicAdd(&hist[0x3F80u - (bits[r] >> 16)], 1u);
      __syncthreads();
      {
        uint4 c[kPieces];
        uint32_t sum = 0, longest = 0;
#pragma unroll
        for (int i = 0; i < kPieces; ++i) {
          c[i] = hist4[tid * kPieces + i];
          sum += c[i].x + c[i].y + c[i].z + c[i].w;
          longest = max(max(max(longest, c[i].x), max(c[i].y, c[i].z)), c[i].w);
        }
        const int lane = tid & 63, wave = tid >> 6;
        uint32_t incl = sum;
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
          const uint32_t o = __shfl_up(incl, d, kWave);
          if (lane >= d) incl += o;
        }
        __shared__ uint32_t wave_total[kRouteThreads / 64];
        if (lane == 63) wave_total[wave] = incl;
        counted = !__syncthreads_or(longest > kLongestSegment);
        uint32_t at = incl - sum;
        for (int w = 0; w < wave; ++w) at += wave_total[w];
#pragma unroll
        for (int i = 0; i < kPieces && counted; ++i) {
          const uint4 v = c[i];
          hist4[tid * kPieces + i] = make_uint4(at, at + v.x, at + v.x + v.y, at + v.x + v.y + v.z);
          at += v.x + v.y + v.z + v.w;
        }
      }
      __syncthreads();
#pragma unroll
      for (int r = 0; r < R; ++r)
        if (counted && tid < nact && tid * R + r < S)
          seg[atomicAdd(&hist[0x3F80u - (bits[r] >> 16)], 1u)] = bin_key32(bits[r], tid * R + r);
      __syncthreads();
      // A bin's cursor now stands at its end, which is where the next bin starts.
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const int s = tid * R + r;
        if (counted && tid < nact && s < S) {
          const uint32_t bin = 0x3F80u - (bits[r] >> 16);
          const uint32_t first = bin > 0 ? hist[bin - 1] : 0u, end = hist[bin], mine = bin_key32(bits[r], s);
          uint32_t lower = 0;
          for (uint32_t q = first; q < end; q += 4)          // four reads in flight
#pragma unroll
            for (uint32_t u = 0; u < 4; ++u)
              lower += seg[min(q + u, end - 1)] < mine && q + u < end ? 1u : 0u;
          emit((int)(first + lower), s);
        }
      }
    }
    if (!counted) {
      uint64_t key[R];
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const int s = tid * R + r;
        key[r] = (tid < nact && s < S) ? bpr_key64(bits[r], s) : ~0ull;
      }
      bitonic_sort_regs<R, uint64_t>(key, keys, SP, tid, nact);
#pragma unroll
      for (int r = 0; r < R; ++r)
        if (tid < nact && tid * R + r < S) emit(tid * R + r, (int)(uint32_t)key[r]);
    }
  }
  for (int c = S + tid; c < C; c += blockDim.x) slot_token[slot_row(e, g, c, G, E, C)] = -1;
}

// Items `chunk` at a time (a power of two up to 64): ranks -> indices, token_slot, weights, and the
// counts of the monitoring scalars (integer atomics: the order of the workgroups does not matter).
template <typename T>
__global__ __launch_bounds__(256) void top_items_emit_kernel(
    const T* __restrict__ gates, int32_t* __restrict__ indices, int32_t* __restrict__ token_slot,
    float* __restrict__ weights, TopItemsMetrics m, int G, int S, int E, int C, int chunk, int chunks) {
  extern __shared__ __align__(16) unsigned char smem[];
  int32_t* rank = reinterpret_cast<int32_t*>(smem);     // (E, chunk + 1): one word of padding per expert
  __shared__ int32_t taken[64];
  const int tid = threadIdx.x;
  const int g = blockIdx.x / chunks, s0 = (blockIdx.x - g * chunks) * chunk;
  const int rows = min(chunk, S - s0);
  const size_t base = ((size_t)g * S + s0) * E;
  const int n = rows * E;
  if (tid < 64) taken[tid] = 0;
  if (chunk > 1)
    for (int i = tid; i < n; i += 256) {
      const int e = i / rows;
      rank[e * (chunk + 1) + (i - e * rows)] = token_slot[base + i];
    }
  __syncthreads();
  int mine = 0;      // chunk == 1: experts that took the workgroup's one item
  for (int i = tid; i < n; i += 256) {
    const int o = i / E, e = i - o * E;
    const int r = chunk > 1 ? rank[e * (chunk + 1) + o] : token_slot[base + i];
    *reinterpret_cast<int2*>(indices + 2 * (base + i)) = make_int2(e, r);
    token_slot[base + i] = r < C ? slot_row(e, g, r, G, E, C) : -1;
    weights[base + i] = Elt<T>::load(gates + base + i);
    mine += r < C ? 1 : 0;
  }
  if (m.counts == nullptr) return;
  if (chunk > 1) {
    if (tid < rows) {
      int c = 0;
      for (int e = 0; e < E; ++e) c += rank[e * (chunk + 1) + tid] < C ? 1 : 0;
      taken[tid] = c;
    }
  } else {
    atomicAdd(&taken[0], mine);
  }
  __syncthreads();
  if (tid >= 64) return;
  const bool on = tid < rows;
  const int c = on ? taken[tid] : 0;
  int lo = on ? c : INT32_MAX, hi = c;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    lo = min(lo, __shfl_xor(lo, d, kWave));
    hi = max(hi, __shfl_xor(hi, d, kWave));
  }
  if (tid == 0) {
    atomicMin(&m.items_minmax[g], lo);
    atomicMax(&m.items_minmax[G + g], hi);
  }
  for (int i = 0; i < m.num; ++i) {
    const int at_least = i < m.num - 1 ? 1 << i : E;
    const int cnt = __popcll(__ballot(on && c >= at_least));
    if (tid == 0 && cnt > 0) atomicAdd(&m.counts[(size_t)i * G + g], cnt);
  }
}

// Counts -> shares of the group, in place; the smallest and largest selected gate of every group (a
// NaN among them stays one).
template <typename T>
__global__ __launch_bounds__(64) void top_items_finish_kernel(const float* __restrict__ sel_minmax,
                                                              T* __restrict__ gate_minmax,
                                                              TopItemsMetrics m, int G, int S, int E) {
  const int g = blockIdx.x, lane = threadIdx.x;
  auto lower = [](float a, float b) { return (b < a || b != b) ? b : a; };
  auto upper = [](float a, float b) { return (b > a || b != b) ? b : a; };
  const float* sel = sel_minmax + (size_t)g * E * 2;
  float lo = sel[0], hi = sel[1];
  for (int e = lane; e < E; e += 64) {
    lo = lower(lo, sel[2 * e]);
    hi = upper(hi, sel[2 * e + 1]);
  }
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    lo = lower(lo, __shfl_xor(lo, d, kWave));
    hi = upper(hi, __shfl_xor(hi, d, kWave));
  }
  if (lane == 0) {
    Elt<T>::store(gate_minmax + g, lo);
    Elt<T>::store(gate_minmax + G + g, hi);
  }
  if (lane < m.num) {
    int32_t* at = m.counts + (size_t)lane * G + g;
    *reinterpret_cast<float*>(at) = (float)*at / (float)S;
  }
}

// Empty slots and counters of indices_to_slots_kernel.
__global__ __launch_bounds__(256) void clear_slots_kernel(int32_t* p, size_t n, int32_t* num_dup, int32_t* num_inv) {
  size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = -1;
  if (i == 0) *num_dup = *num_inv = 0;
}

__global__ __launch_bounds__(256) void indices_to_slots_kernel(
    const int32_t* __restrict__ indices, int32_t* __restrict__ token_slot,
    int32_t* __restrict__ slot_token, int32_t* __restrict__ num_dup, int32_t* __restrict__ num_inv,
    int G, int S, int E, int K, int C) {
  size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  size_t n = (size_t)G * S * K;
  if (i >= n) return;
  const size_t item = i / K;
  bool invalid;
  const int slot = slot_of_index_pair(indices[2 * i], indices[2 * i + 1], (int)(item / S), G, E, C,
                                      &invalid);
  if (invalid) atomicAdd(num_inv, 1);
  if (slot >= 0) {
    const int prev = atomicExch(&slot_token[slot], (int)item);
    if (prev >= 0) atomicAdd(num_dup, 1);
  }
  token_slot[i] = slot;
}

__global__ __launch_bounds__(256) void densify_kernel(
    const int32_t* __restrict__ indices, const float* __restrict__ weights,
    float* __restrict__ combine, uint8_t* __restrict__ dispatch, int G, int S, int E, int K, int C) {
  size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  size_t n = (size_t)G * S * K;
  if (i >= n) return;
  int e = indices[2 * i], c = indices[2 * i + 1];
  if (e < 0 || c < 0 || e >= E || c >= C) return;
  size_t item = i / K;
  size_t o = (item * E + e) * C + c;
  if (combine != nullptr) combine[o] = weights[i];
  if (dispatch != nullptr) dispatch[o] = 1;
}


// Packed expert rows, step 1: exclusive prefix over the groups of fill[:, e], one
// workgroup per expert; the total is the expert's row count.
__global__ __launch_bounds__(256) void fill_prefix_kernel(
    const int32_t* __restrict__ fill, int32_t* __restrict__ prefix,
    int32_t* __restrict__ rows_per_expert, int G, int E) {
  __shared__ int32_t wsum[4];
  const int e = blockIdx.x;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  int carry = 0;
  for (int g0 = 0; g0 < G; g0 += 256) {
    const int g = g0 + tid;
    const int v = g < G ? fill[(size_t)g * E + e] : 0;
    int x = v;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int y = __shfl_up(x, o, kWave);
      if (lane >= o) x += y;
    }
    if (lane == 63) wsum[wave] = x;
    __syncthreads();
    int woff = 0, total = 0;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      if (w < wave) woff += wsum[w];
      total += wsum[w];
    }
    if (g < G) prefix[(size_t)g * E + e] = carry + woff + x - v;
    carry += total;
    __syncthreads();
  }
  if (tid == 0) rows_per_expert[e] = carry;
}

// Step 2: token_slot = e*G*C + r(g, c)  ->  token_row = e*G*C + prefix[g][e] + c.
__global__ __launch_bounds__(256) void compact_rows_kernel(
    const int32_t* __restrict__ prefix, const int32_t* __restrict__ token_slot,
    int32_t* __restrict__ token_row, int32_t* __restrict__ row_token, int G, int E, int C,
    int per_group, int K, size_t n) {
  const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  const int slot = token_slot[i];
  int row = -1;
  if (slot >= 0) {
    const int g = (int)(i / per_group);
    row = packed_row(slot, prefix[(size_t)g * E + slot_expert(slot, G, C)], G, C);
    if (row_token != nullptr) row_token[row] = (int)(i / K);
  }
  token_row[i] = row;
}

// Both steps in one launch, for E <= 256 and at least 256 assignments per group (a
// workgroup then touches at most two groups): the workgroup adds up the fill counts of
// the groups before its first group itself -- 256 / E threads per expert, each a strided
// share of the groups, joined in LDS -- instead of reading a prefix that another launch
// wrote.  Workgroup 0 also writes the experts' row counts.
__global__ __launch_bounds__(256) void compact_rows_fused_kernel(
    const int32_t* __restrict__ fill, const int32_t* __restrict__ token_slot,
    int32_t* __restrict__ token_row, int32_t* __restrict__ row_token,
    int32_t* __restrict__ rows_per_expert, int G, int E, int C, int per_group, int K, size_t n) {
  compact_rows_fused_block(fill, token_slot, token_row, row_token, rows_per_expert, G, E, C,
                           per_group, K, n, blockIdx.x);
}

}  // namespace
}  // namespace vmoe

using namespace vmoe;

static int check_route_shapes(int G, int S, int E, int K, int C) {
  if (G < 1 || S < 1 || E < 1 || K < 1 || C < 1 || K > E) return VMOE_E_SHAPE;
  if ((int64_t)G * S * K * 2 >= INT32_MAX || (int64_t)E * G * C >= INT32_MAX) return VMOE_E_OVERFLOW;
  return VMOE_OK;
}

static int check_route_assign(const VmoeRouteAssignParams* p) {
  if (p == nullptr || p->topk_idx == nullptr || p->indices == nullptr ||
      p->token_slot == nullptr || p->slot_token == nullptr)
    return VMOE_E_NULL;
  if (p->batch_priority && p->topk_val == nullptr) return VMOE_E_NULL;
  return check_route_shapes(p->G, p->S, p->E, p->K, p->C);
}

// Launches the slot assignment, with the router's losses as extra workgroups when m is given.
static int launch_route_assign(const VmoeRouteAssignParams* p, const VmoeRouterMetricsParams* m,
                               vmoe_stream_t stream) {
  const int SP = pow2ceil(p->S);
  const int W = (p->S * p->K + 31) / 32;
  const int R = keys_per_thread(SP);
  // (the region of the sort keys also serves the counting rank: two arrays of kRankBins
  // words and one of S)
  const int rank_words = 2 * kRankBins + p->S;
  const int NK = SP > (rank_words + 1) / 2 ? SP : (rank_words + 1) / 2;
  size_t lds = (p->batch_priority ? (size_t)NK * 8 : 0) + (size_t)p->E * W * 8 +
               (size_t)p->S * 4 + (size_t)p->E * 4;
  RouterMetricsArgs ma{};
  if (m != nullptr) {
    size_t mlds;
    int V;
    if (!router_metrics_geometry(m, &V, &mlds)) return VMOE_E_UNSUPPORTED;
    if (mlds > lds) lds = mlds;
    ma = RouterMetricsArgs{m->gates, m->top1_idx, m->importance_loss, m->gshard_loss,
                           m->auxiliary_loss, m->gshard_loss_weight, m->importance_loss_weight,
                           m->S, m->E, m->top1_stride, V};
  }
  if (lds > 160 * 1024) return VMOE_E_UNSUPPORTED;
  auto launch = [&](auto kern, auto... extra) -> int {
    hipError_t e = allow_dynamic_lds(reinterpret_cast<const void*>(kern), lds);
    if (e != hipSuccess) return (int)e;
    hipLaunchKernelGGL(kern, dim3(m != nullptr ? 2 * p->G : p->G), dim3(kRouteThreads), lds,
                       as_stream(stream), p->topk_val, p->topk_idx, p->indices, p->token_slot,
                       p->slot_token, p->fill, p->G, p->S, p->E, p->K, p->C,
                       p->batch_priority ? 1 : 0, SP, NK, W, extra...);
    return launch_status();
  };
  if (m == nullptr) {
    switch (R) {
      case 1: return launch(route_assign_kernel<1>);
      case 2: return launch(route_assign_kernel<2>);
      case 4: return launch(route_assign_kernel<4>);
      case 8: return launch(route_assign_kernel<8>);
      default: return launch(route_assign_kernel<0>);
    }
  }
  if (m->dtype == VMOE_BF16) {
    switch (R) {
      case 1: return launch(route_assign_metrics_kernel<1, bf16_t>, ma);
      case 2: return launch(route_assign_metrics_kernel<2, bf16_t>, ma);
      case 4: return launch(route_assign_metrics_kernel<4, bf16_t>, ma);
      case 8: return launch(route_assign_metrics_kernel<8, bf16_t>, ma);
      default: return launch(route_assign_metrics_kernel<0, bf16_t>, ma);
    }
  }
  switch (R) {
    case 1: return launch(route_assign_metrics_kernel<1, float>, ma);
    case 2: return launch(route_assign_metrics_kernel<2, float>, ma);
    case 4: return launch(route_assign_metrics_kernel<4, float>, ma);
    case 8: return launch(route_assign_metrics_kernel<8, float>, ma);
    default: return launch(route_assign_metrics_kernel<0, float>, ma);
  }
}

extern "C" int vmoe_route_assign(const VmoeRouteAssignParams* p, vmoe_stream_t stream) {
  int rc = check_route_assign(p);
  if (rc != VMOE_OK) return rc;
  return launch_route_assign(p, nullptr, stream);
}

extern "C" int vmoe_route_assign_metrics(const VmoeRouteAssignParams* p,
                                         const VmoeRouterMetricsParams* m, vmoe_stream_t stream) {
  int rc = check_route_assign(p);
  if (rc != VMOE_OK) return rc;
  rc = check_router_metrics(m);
  if (rc != VMOE_OK) return rc;
  if (m->G != p->G || m->S != p->S || m->E != p->E) return VMOE_E_SHAPE;
  return launch_route_assign(p, m, stream);
}

extern "C" int vmoe_indices_to_slots(const VmoeIndicesToSlotsParams* p, vmoe_stream_t stream) {
  if (p == nullptr || p->indices == nullptr || p->token_slot == nullptr ||
      p->slot_token == nullptr || p->num_duplicates == nullptr || p->num_invalid == nullptr)
    return VMOE_E_NULL;
  if (p->G < 1 || p->S < 1 || p->E < 1 || p->K < 1 || p->C < 1) return VMOE_E_SHAPE;
  if ((int64_t)p->G * p->S * p->K * 2 >= INT32_MAX || (int64_t)p->E * p->G * p->C >= INT32_MAX)
    return VMOE_E_OVERFLOW;
  const size_t ns = (size_t)p->E * p->G * p->C;
  const size_t n = (size_t)p->G * p->S * p->K;
  hipLaunchKernelGGL(clear_slots_kernel, dim3((unsigned)((ns + 255) / 256)), dim3(256), 0,
                     as_stream(stream), p->slot_token, ns, p->num_duplicates, p->num_invalid);
  hipLaunchKernelGGL(indices_to_slots_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0,
                     as_stream(stream), p->indices, p->token_slot, p->slot_token,
                     p->num_duplicates, p->num_invalid, p->G, p->S, p->E, p->K, p->C);
  return launch_status();
}

extern "C" int vmoe_densify(const VmoeDensifyParams* p, vmoe_stream_t stream) {
  if (p == nullptr || p->indices == nullptr) return VMOE_E_NULL;
  if (p->combine != nullptr && p->weights == nullptr) return VMOE_E_NULL;
  if (p->G < 1 || p->S < 1 || p->E < 1 || p->K < 1 || p->C < 1) return VMOE_E_SHAPE;
  const size_t n = (size_t)p->G * p->S * p->K;
  hipLaunchKernelGGL(densify_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0,
                     as_stream(stream), p->indices, p->weights, p->combine, p->dispatch, p->G,
                     p->S, p->E, p->K, p->C);
  return launch_status();
}

template <typename T>
static int launch_top_items(const VmoeTopItemsParams* p, const TopItemsMetrics& m, T* gate_minmax,
                            vmoe_stream_t stream) {
  const int SP = pow2ceil(p->S < 2 ? 2 : p->S);
  const int R = keys_per_thread(SP);
  const T* gates = (const T*)p->gates;
  size_t lds = (size_t)SP * 8;
  if (R > 0 && rank_by_counting(SP)) {
    const size_t counting = ((size_t)kGateBins + p->S) * 4;
    if (counting > lds) lds = counting;
  }
  if (lds > 160 * 1024) return VMOE_E_UNSUPPORTED;
  // Columns that are sorted in registers, a key per thread, take no more threads than keys: many small groups
  // are as many workgroups, and 16 waves of which one works held up the others (50 experts x 23 groups of
  // 244 items, bfloat16: 20 -> 11 us; 26 x 119 of 54, float32: 28 -> 8).
  const int threads = R == 1 && !rank_by_counting(SP) ? (SP > kWave ? SP : kWave) : kRouteThreads;
  int chunk = 64;      // items per workgroup of the second launch: their ranks take up to 64 KB of LDS
  while (chunk > 1 && (size_t)p->E * (chunk + 1) * 4 > 64 * 1024) chunk >>= 1;
  const int chunks = (p->S + chunk - 1) / chunk;
  const size_t emit_lds = chunk > 1 ? (size_t)p->E * (chunk + 1) * 4 : 0;
  auto launch = [&](auto kern) -> int {
    hipError_t e = allow_dynamic_lds(reinterpret_cast<const void*>(kern), lds);
    if (e != hipSuccess) return (int)e;
    hipLaunchKernelGGL(kern, dim3(p->E, p->G), dim3(threads), lds, as_stream(stream), gates,
                       p->token_slot, p->slot_token, p->sel_minmax, m, p->G, p->S, p->E, p->C, SP, chunk);
    return launch_status();
  };
  int rc;
  switch (R) {
    case 1: rc = launch(top_items_kernel<T, 1>); break;
    case 2: rc = launch(top_items_kernel<T, 2>); break;
    case 4: rc = launch(top_items_kernel<T, 4>); break;
    case 8: rc = launch(top_items_kernel<T, 8>); break;
    default: rc = launch(top_items_kernel<T, 0>); break;
  }
  if (rc != VMOE_OK) return rc;
  hipError_t e = allow_dynamic_lds(reinterpret_cast<const void*>(top_items_emit_kernel<T>), emit_lds);
  if (e != hipSuccess) return (int)e;
  hipLaunchKernelGGL(top_items_emit_kernel<T>, dim3((unsigned)(p->G * chunks)), dim3(256), emit_lds,
                     as_stream(stream), gates, p->indices, p->token_slot, p->weights, m, p->G, p->S, p->E,
                     p->C, chunk, chunks);
  rc = launch_status();
  if (rc != VMOE_OK || m.counts == nullptr) return rc;
  hipLaunchKernelGGL(top_items_finish_kernel<T>, dim3((unsigned)p->G), dim3(64), 0, as_stream(stream),
                     p->sel_minmax, gate_minmax, m, p->G, p->S, p->E);
  return launch_status();
}

static int top_items(const VmoeTopItemsParams* p, const TopItemsMetrics& m, void* gate_minmax,
                     vmoe_stream_t stream) {
  if (p == nullptr || p->gates == nullptr || p->indices == nullptr || p->token_slot == nullptr ||
      p->slot_token == nullptr || p->weights == nullptr)
    return VMOE_E_NULL;
  if (p->G < 1 || p->S < 1 || p->E < 1 || p->C < 1) return VMOE_E_SHAPE;
  if (p->dtype != VMOE_F32 && p->dtype != VMOE_BF16) return VMOE_E_DTYPE;
  if (p->G > 65535) return VMOE_E_UNSUPPORTED;
  if ((int64_t)p->E * p->G * p->C >= INT32_MAX || (int64_t)p->G * p->S * p->E >= INT32_MAX)
    return VMOE_E_OVERFLOW;
  return p->dtype == VMOE_BF16 ? launch_top_items<bf16_t>(p, m, (bf16_t*)gate_minmax, stream)
                               : launch_top_items<float>(p, m, (float*)gate_minmax, stream);
}

extern "C" int vmoe_top_items_per_expert(const VmoeTopItemsParams* p, vmoe_stream_t stream) {
  return top_items(p, TopItemsMetrics{}, nullptr, stream);
}

extern "C" int vmoe_top_items_metrics(const VmoeTopItemsParams* p, int32_t* items_minmax, void* gate_minmax,
                                      float* ratios, int32_t* rows_per_expert, vmoe_stream_t stream) {
  if (p == nullptr || p->sel_minmax == nullptr || items_minmax == nullptr || gate_minmax == nullptr ||
      ratios == nullptr)
    return VMOE_E_NULL;
  TopItemsMetrics m{items_minmax, reinterpret_cast<int32_t*>(ratios), 2, rows_per_expert};
  while (p->E >> (m.num - 1)) ++m.num;     // floor(log2 E) + 2
  return top_items(p, m, gate_minmax, stream);
}

// Launches the row compaction with `prefix` as the (G, E) scratch of its two-launch form.
static int launch_compact_rows(const VmoeCompactRowsParams* p, int32_t* prefix,
                               vmoe_stream_t stream) {
  const size_t n = (size_t)p->G * p->S * p->K;
  if (compact_rows_fused_ok(p->G, p->S, p->E, p->K)) {
    hipLaunchKernelGGL(compact_rows_fused_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0,
                       as_stream(stream), p->fill, p->token_slot, p->token_row, p->row_token,
                       p->rows_per_expert, p->G, p->E, p->C, p->S * p->K, p->K, n);
    return launch_status();
  }
  hipLaunchKernelGGL(fill_prefix_kernel, dim3(p->E), dim3(256), 0, as_stream(stream), p->fill,
                     prefix, p->rows_per_expert, p->G, p->E);
  hipLaunchKernelGGL(compact_rows_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0,
                     as_stream(stream), prefix, p->token_slot, p->token_row, p->row_token, p->G,
                     p->E, p->C, p->S * p->K, p->K, n);
  return launch_status();
}

static int check_compact_rows(const VmoeCompactRowsParams* p) {
  if (p == nullptr || p->fill == nullptr || p->token_slot == nullptr || p->token_row == nullptr ||
      p->rows_per_expert == nullptr)
    return VMOE_E_NULL;
  return check_route_shapes(p->G, p->S, p->E, p->K, p->C);
}

extern "C" int vmoe_compact_rows(const VmoeCompactRowsParams* p, vmoe_stream_t stream) {
  int rc = check_compact_rows(p);
  if (rc != VMOE_OK) return rc;
  if (p->prefix == nullptr) return VMOE_E_NULL;
  return launch_compact_rows(p, p->prefix, stream);
}

// ---------------------------------------------------------------- no allocation
// vmoe_compact_rows for callers that cannot allocate: the (G, E) scratch is a file-scope
// device array.  Its name is only a host-side handle; the device address is asked for once
// per device (each device holds its own copy) and only that address is given to kernels.
static __device__ __align__(256) int32_t scratch[VMOE_COMPACT_ROWS_STATIC_MAX_GE];

namespace {
constexpr int kMaxDevices = 64;
std::mutex scratch_mutex;
int32_t* scratch_ptr[kMaxDevices];   // device address of `scratch` on each device, null until asked
}  // namespace

// Device address of this device's copy of `scratch` (the current device), or null with *err set.
static int32_t* scratch_address(int* err) {
  int dev = -1;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) { *err = (int)e; return nullptr; }
  if (dev < 0 || dev >= kMaxDevices) { *err = VMOE_E_UNSUPPORTED; return nullptr; }
  std::lock_guard<std::mutex> lock(scratch_mutex);
  if (scratch_ptr[dev] == nullptr) {
    void* ptr = nullptr;
    e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
    if (e != hipSuccess || ptr == nullptr) {
      *err = e != hipSuccess ? (int)e : (int)hipErrorInvalidSymbol;
      return nullptr;
    }
    scratch_ptr[dev] = static_cast<int32_t*>(ptr);
  }
  return scratch_ptr[dev];
}

extern "C" int vmoe_compact_rows_static(const VmoeCompactRowsParams* p, vmoe_stream_t stream) {
  int rc = check_compact_rows(p);
  if (rc != VMOE_OK) return rc;
  if ((int64_t)p->G * p->E > VMOE_COMPACT_ROWS_STATIC_MAX_GE) return VMOE_E_WORKSPACE;
  int err = VMOE_OK;
  int32_t* prefix = scratch_address(&err);
  if (prefix == nullptr) return err;
  // Every entry of the scratch that the second launch reads (g < G, e < E) is written by the
  // first one: nothing has to start at zero, whatever an earlier call left behind.
  return launch_compact_rows(p, prefix, stream);
}
