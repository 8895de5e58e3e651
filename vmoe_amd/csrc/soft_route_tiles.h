// Soft MoE routing for any number of slots, width and group size, float32 and bfloat16, in two
// launches over row tiles instead of one workgroup per group.
//
// soft_logits_kernel: a workgroup takes 16 RB item rows of one group.  It loads them once
// (coalesced), takes their norms in registers, writes the unit-norm rows to LDS and multiplies them
// with all slots; the slot parameters come in fragment order (soft_prep_mu_kernel: every fragment
// load of a wave is 1 KB of consecutive memory) out of L2.  The logits of its rows, rounded to the
// data type, meet in LDS for the softmax over slots, and leave both as combine weights and, to the
// array of the dispatch weights, as logits.
// soft_columns_kernel: workgroups over (group, chunk of slots) turn those logits into the softmax over
// items, in place; soft_stats_kernel takes the monitoring sums.
//
// What bounds it.  64 groups of 196 items x 768 and 256 slots move 39 MB, 6 us of HBM time, in three
// short launches that are each one round of latencies (29 + 17 + 8 us): every tile reads all slot
// parameters (390 KB through one CU's L2 port, 8 us), norms and softmaxes are serial behind their
// loads.  The workgroup per group that this replaces walked its rows with four waves, read the items
// again for every 128 slots and took the column softmax with one thread per slot: 536 us, and 18 for
// the sums.  float32, 32 groups of 49 items x 512 and 48 slots: 10 + 5 + 4 us, 186 + 19 before (one
// value per lane and MFMA).
#ifndef VMOE_SOFT_ROUTE_TILES_H_
#define VMOE_SOFT_ROUTE_TILES_H_
#include <type_traits>

#include "vmoe_common.h"

namespace vmoe {
namespace soft {

constexpr float kNormEps = 1e-6f;

// A 16-byte piece of a row: V values, and the k steps that one piece per lane covers: 4 V k per step.
// bfloat16: a lane holds 8 consecutive k of row lane % 16, from (lane / 16) * 8 on.  float32: k = 4 j +
// lane / 16, j = 0 .. 3, so that the four MFMAs of a step add the products in the order of k: a
// float32 layer rounds its experts' outputs to bfloat16 (Bfloat16Dispatcher), where a last bit of the
// weights can turn a rounding, so float32 keeps one order of every sum whatever the tiling.
template <typename T> struct Piece;
template <> struct Piece<bf16_t> {
  static constexpr int V = 8;
  __device__ static __forceinline__ void unpack(const uint4& r, float (&v)[8]) {
    v[0] = bf_lo(r.x); v[1] = bf_hi(r.x); v[2] = bf_lo(r.y); v[3] = bf_hi(r.y);
    v[4] = bf_lo(r.z); v[5] = bf_hi(r.z); v[6] = bf_lo(r.w); v[7] = bf_hi(r.w);
  }
  __device__ static __forceinline__ uint4 pack(const float (&v)[8]) {
    return make_uint4(pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]), pack_bf16x2(v[4], v[5]),
                      pack_bf16x2(v[6], v[7]));
  }
  __device__ static __forceinline__ floatx4 mma(const uint4& slots, const uint4& rows, floatx4 acc) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, slots),
                                                   __builtin_bit_cast(bf16x8, rows), acc, 0, 0, 0);
  }
};
template <> struct Piece<float> {
  static constexpr int V = 4;
  __device__ static __forceinline__ void unpack(const uint4& r, float (&v)[4]) {
    v[0] = __builtin_bit_cast(float, r.x); v[1] = __builtin_bit_cast(float, r.y);
    v[2] = __builtin_bit_cast(float, r.z); v[3] = __builtin_bit_cast(float, r.w);
  }
  __device__ static __forceinline__ uint4 pack(const float (&v)[4]) {
    return make_uint4(__builtin_bit_cast(uint32_t, v[0]), __builtin_bit_cast(uint32_t, v[1]),
                      __builtin_bit_cast(uint32_t, v[2]), __builtin_bit_cast(uint32_t, v[3]));
  }
  __device__ static __forceinline__ floatx4 mma(const uint4& slots, const uint4& rows, floatx4 acc) {
    float a[4], b[4];
    unpack(slots, a);
    unpack(rows, b);
#pragma unroll
    for (int t = 0; t < 4; ++t) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a[t], b[t], acc, 0, 0, 0);
    return acc;
  }
};

// k steps of a width, padded to whole groups of four (the loop's prefetch distance).
template <typename T> inline int padded_steps(int D) {
  const int k = 4 * Piece<T>::V;
  return ((D + k - 1) / k + 3) / 4 * 4;
}

constexpr int logits_waves(int rb) { return rb >= 4 ? 8 : 4; }      // 16 RB rows per workgroup

struct LogitsLds {
  int row_bytes, lg_row, total;
  int lg;           // offset of the logits
};
template <typename T> inline LogitsLds logits_lds(int D, int N, int rows) {
  LogitsLds l;
  l.row_bytes = padded_steps<T>(D) * 64 + 16;                   // + 16: rows in different banks
  l.lg_row = (N + 15) / 16 * 16 * (int)sizeof(T) + 16;
  l.lg = rows * l.row_bytes;
  l.total = l.lg + rows * l.lg_row;
  return l;
}

__device__ __forceinline__ float wave_max(float v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o, 64));
  return v;
}
__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}

// PIECES: 16-byte pieces of an item row per lane (rows of up to 1 KB x PIECES); VEC (bfloat16): rows of
// slots are whole pieces at aligned addresses.  PAIR: see below.
template <typename T, int RB, int PIECES, bool VEC, bool PAIR>
__global__ __launch_bounds__(64 * logits_waves(RB), PIECES > 4 ? 1 : !PAIR && PIECES <= 2 && RB < 4 ? 3 : 2) void soft_logits_kernel(
    const T* __restrict__ x, const uint4* __restrict__ mu, T* __restrict__ logits, T* __restrict__ combine_w,
    T* __restrict__ logits_out, float scale, int scale_x, int S, int D, int N, int steps, int row_tiles,
    LogitsLds L) {
  using P = Piece<T>;
  constexpr bool kBf16 = sizeof(T) == 2;
  constexpr int V = P::V, kRows = 16 * RB, kWaves = logits_waves(RB), kPerWave = kRows / kWaves;
  extern __shared__ __align__(16) unsigned char smem[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = blockIdx.x / row_tiles, row0 = (blockIdx.x - g * row_tiles) * kRows;
  const int r16 = lane & 15, q = lane >> 4;
  const float sc = Elt<T>::round(scale);

  // The slot fragments of the wave's first block and steps go out ahead of everything else.
  const int blocks = (N + 15) / 16;
  // What a wave multiplies at a time: every row block with two blocks of slots, or, where the
  // slots are too few to give every wave two blocks, one row block with one block of slots.
  constexpr int IB = PAIR ? RB : 1, JB = PAIR ? 2 : 1;
  const int items = PAIR ? (blocks + 1) / 2 : RB * blocks;
  uint4 f[2][4][JB];
  auto fetch = [&](const int u, int item, int s) {
    const int b0 = PAIR ? item * 2 : item % blocks;
#pragma unroll
    for (int j = 0; j < JB; ++j) {
      const uint4* m = mu + ((size_t)min(b0 + j, blocks - 1) * steps + s) * 64 + lane;
#pragma unroll
      for (int t = 0; t < 4; ++t) f[u][t][j] = m[t * 64];
    }
  };
  if (wave < items) fetch(0, wave, 0);

  if constexpr (kBf16) {
    // Rows: a wave loads its rows' pieces, as many rows in flight as the registers hold.
    constexpr int kBatch = PIECES <= 2 ? kPerWave : 4;
    const int pieces = (D + V - 1) / V, all_pieces = steps * 4;
#pragma unroll
    for (int i0 = 0; i0 < kPerWave; i0 += kBatch) {
      uint4 raw[kBatch][PIECES];
#pragma unroll
      for (int i = 0; i < kBatch; ++i) {
        const int s = min(row0 + wave * kPerWave + i0 + i, S - 1);
        const T* row = x + ((size_t)g * S + s) * D;
#pragma unroll
        for (int c = 0; c < PIECES; ++c) {
          const int p = lane + 64 * c;
          raw[i][c] = make_uint4(0, 0, 0, 0);
          if (p >= pieces) continue;
          raw[i][c] = *reinterpret_cast<const uint4*>(row + p * V);
        }
      }
      float sum[kBatch];
#pragma unroll
      for (int i = 0; i < kBatch; ++i) {
        sum[i] = 0.f;
#pragma unroll
        for (int c = 0; c < PIECES; ++c) {
          float v[V];
          P::unpack(raw[i][c], v);
#pragma unroll
          for (int j = 0; j < V; ++j) sum[i] += v[j] * v[j];
        }
      }
#pragma unroll
      for (int o = 32; o > 0; o >>= 1)
#pragma unroll
        for (int i = 0; i < kBatch; ++i) sum[i] += __shfl_xor(sum[i], o, 64);
#pragma unroll
      for (int i = 0; i < kBatch; ++i) {
        const float inv = 1.0f / sqrtf(sum[i] + kNormEps);
        unsigned char* dst = smem + (wave * kPerWave + i0 + i) * L.row_bytes;
#pragma unroll
        for (int c = 0; c < PIECES; ++c) {
          const int p = lane + 64 * c;
          float v[V];
          P::unpack(raw[i][c], v);
#pragma unroll
          for (int j = 0; j < V; ++j) {
            v[j] = Elt<T>::round(v[j] * inv);
            if (scale_x) v[j] = Elt<T>::round(v[j] * sc);
          }
          if (p < all_pieces) *reinterpret_cast<uint4*>(dst + p * 16) = P::pack(v);
        }
      }
    }
  } else {
    // Values d = lane + 64 i of a row, four rows at a time; the sum of squares in that order.
    constexpr int kVals = 4 * PIECES;
#pragma unroll
    for (int i0 = 0; i0 < kPerWave; i0 += 4) {
      float v[4][kVals], sum[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const T* row = x + ((size_t)g * S + min(row0 + wave * kPerWave + i0 + i, S - 1)) * D;
#pragma unroll
        for (int c = 0; c < kVals; ++c) v[i][c] = lane + 64 * c < D ? row[lane + 64 * c] : 0.f;
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        sum[i] = 0.f;
#pragma unroll
        for (int c = 0; c < kVals; ++c)
          if (lane + 64 * c < D) sum[i] += v[i][c] * v[i][c];
      }
#pragma unroll
      for (int o = 32; o > 0; o >>= 1)
#pragma unroll
        for (int i = 0; i < 4; ++i) sum[i] += __shfl_xor(sum[i], o, 64);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float inv = 1.0f / sqrtf(sum[i] + kNormEps);
        float* dst = reinterpret_cast<float*>(smem + (wave * kPerWave + i0 + i) * L.row_bytes);
#pragma unroll
        for (int c = 0; c < kVals; ++c) {
          const int d = lane + 64 * c;
          float a = v[i][c] * inv;
          if (scale_x) a = a * sc;
          if (d < steps * 16) dst[(d & ~15) + (d & 3) * 4 + ((d & 15) >> 2)] = a;
        }
      }
    }
  }
  __syncthreads();

  // Logits; four steps' slot fragments are in flight while the four before them are multiplied.
  const unsigned char* xrow = smem + r16 * L.row_bytes + q * 16;
  for (int item = wave; item < items; item += kWaves) {
    const int b0 = PAIR ? item * 2 : item % blocks, i0 = PAIR ? 0 : item / blocks;
    floatx4 acc[IB][JB];
#pragma unroll
    for (int i = 0; i < IB; ++i)
#pragma unroll
      for (int j = 0; j < JB; ++j) acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};
    auto multiply = [&](const int u, int s) {
#pragma unroll
      for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int i = 0; i < IB; ++i) {
          const uint4 a = *reinterpret_cast<const uint4*>(xrow + (i0 + i) * 16 * L.row_bytes + (s + t) * 64);
#pragma unroll
          for (int j = 0; j < JB; ++j) acc[i][j] = P::mma(f[u][t][j], a, acc[i][j]);
        }
    };
    for (int s = 0; s < steps; s += 8) {          // steps is a multiple of four
      const bool second = s + 4 < steps;
      if (second) fetch(1, item, s + 4);
      else fetch(0 + 1, min(item + kWaves, items - 1), 0);
      __builtin_amdgcn_sched_barrier(0);
      multiply(0, s);
      __builtin_amdgcn_sched_barrier(0);
      if (second) {
        if (s + 8 < steps) fetch(0, item, s + 8);
        else fetch(0, min(item + kWaves, items - 1), 0);
        __builtin_amdgcn_sched_barrier(0);
        multiply(1, s + 4);
        __builtin_amdgcn_sched_barrier(0);
      } else {
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
          for (int j = 0; j < JB; ++j) f[0][t][j] = f[1][t][j];
      }
    }
    mfma_result_fence();
    // acc[i][j][v]: row (i0 + i) * 16 + lane % 16, slot (b0 + j) * 16 + (lane / 16) * 4 + v
#pragma unroll
    for (int i = 0; i < IB; ++i)
#pragma unroll
      for (int j = 0; j < JB; ++j) {
        if (b0 + j >= blocks) continue;
        T* dst = reinterpret_cast<T*>(smem + L.lg + ((i0 + i) * 16 + r16) * L.lg_row) + (b0 + j) * 16 + q * 4;
        if constexpr (sizeof(T) == 2)
          *reinterpret_cast<uint2*>(dst) = make_uint2(pack_bf16x2(acc[i][j][0], acc[i][j][1]),
                                                      pack_bf16x2(acc[i][j][2], acc[i][j][3]));
        else
          *reinterpret_cast<floatx4*>(dst) = acc[i][j];
      }
  }
  __syncthreads();

  if constexpr (kBf16) {
    // Softmax over the slots of each row: `span` lanes (a power of two) per row, 64 / span rows of the
    // wave side by side.
    const int slot_pieces = (N + V - 1) / V;
    const int span = slot_pieces > 32 ? 64 : slot_pieces > 16 ? 32 : slot_pieces > 8 ? 16 : 8;
    const int sl = lane & (span - 1), sub = lane / span;
    for (int i = sub; i < kPerWave; i += 64 / span) {
      const int s = row0 + wave * kPerWave + i;
      const bool live = s < S;
      const unsigned char* src = smem + L.lg + (wave * kPerWave + i) * L.lg_row;
      const size_t base = ((size_t)g * S + s) * N;
      auto read = [&](int p, float (&v)[V]) {
        P::unpack(*reinterpret_cast<const uint4*>(src + p * 16), v);
        if (!VEC) {
#pragma unroll
          for (int j = 0; j < V; ++j)
            if (p * V + j >= N) v[j] = -INFINITY;
        }
      };
      float mx = -INFINITY, sum = 0.f;
      for (int p = sl; p < slot_pieces; p += span) {
        float v[V];
        read(p, v);
#pragma unroll
        for (int j = 0; j < V; ++j) mx = fmaxf(mx, v[j]);
      }
      for (int o = span >> 1; o > 0; o >>= 1) mx = fmaxf(mx, __shfl_xor(mx, o, 64));
      for (int p = sl; p < slot_pieces; p += span) {
        float v[V];
        read(p, v);
#pragma unroll
        for (int j = 0; j < V; ++j) sum += expf(v[j] - mx);
      }
      for (int o = span >> 1; o > 0; o >>= 1) sum += __shfl_xor(sum, o, 64);
      for (int p = sl; p < slot_pieces; p += span) {
        float v[V], e[V];
        read(p, v);
#pragma unroll
        for (int j = 0; j < V; ++j) e[j] = expf(v[j] - mx) / sum;
        if (!live) continue;
        if (VEC) {
          *reinterpret_cast<uint4*>(combine_w + base + p * V) = P::pack(e);
          *reinterpret_cast<uint4*>(logits + base + p * V) = P::pack(v);
          if (logits_out != nullptr) *reinterpret_cast<uint4*>(logits_out + base + p * V) = P::pack(v);
        } else {
#pragma unroll
          for (int j = 0; j < V; ++j) {
            if (p * V + j >= N) continue;
            Elt<T>::store(combine_w + base + p * V + j, e[j]);
            Elt<T>::store(logits + base + p * V + j, v[j]);
            if (logits_out != nullptr) Elt<T>::store(logits_out + base + p * V + j, v[j]);
          }
        }
      }
    }
  } else {
    // A wave per row, slot n in lane n % 64, four rows side by side.
    for (int i0 = 0; i0 < kPerWave; i0 += 4) {
      const float* src[4];
      float mx[4], sum[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        src[i] = reinterpret_cast<const float*>(smem + L.lg + (wave * kPerWave + i0 + i) * L.lg_row);
        mx[i] = -INFINITY;
        sum[i] = 0.f;
      }
      for (int n = lane; n < N; n += 64)
#pragma unroll
        for (int i = 0; i < 4; ++i) mx[i] = fmaxf(mx[i], src[i][n]);
#pragma unroll
      for (int o = 32; o > 0; o >>= 1)
#pragma unroll
        for (int i = 0; i < 4; ++i) mx[i] = fmaxf(mx[i], __shfl_xor(mx[i], o, 64));
      for (int n = lane; n < N; n += 64)
#pragma unroll
        for (int i = 0; i < 4; ++i) sum[i] += expf(src[i][n] - mx[i]);
#pragma unroll
      for (int o = 32; o > 0; o >>= 1)
#pragma unroll
        for (int i = 0; i < 4; ++i) sum[i] += __shfl_xor(sum[i], o, 64);
      for (int n = lane; n < N; n += 64)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int s = row0 + wave * kPerWave + i0 + i;
          if (s >= S) continue;
          const size_t at = ((size_t)g * S + s) * N + n;
          const float l = src[i][n];
          combine_w[at] = expf(l - mx[i]) / sum[i];
          logits[at] = l;
          if (logits_out != nullptr) logits_out[at] = l;
        }
    }
  }
}

// A workgroup per group and chunk of `columns` pieces (VEC: V slots each, else one); a thread keeps
// one piece column and every `lanes`-th row of it; the threads of a column meet in LDS.
constexpr int kColThreads = 256;

template <typename T, bool VEC>
__global__ __launch_bounds__(kColThreads) void soft_columns_kernel(T* __restrict__ dispatch_w, int S, int N,
                                                                   int all_columns, int columns, int chunks,
                                                                   int lanes) {
  using P = Piece<T>;
  constexpr int V = VEC ? P::V : 1;
  __shared__ float lds[kColThreads * V], lds2[kColThreads * V];      // [lanes][columns * V]
  const int tid = threadIdx.x;
  const int g = blockIdx.x / chunks, c0 = (blockIdx.x - g * chunks) * columns, width = columns * V;
  const int col = tid % columns, rl = tid / columns;
  const bool on = rl < lanes && c0 + col < all_columns;
  T* dw = dispatch_w + (size_t)g * S * N + (size_t)(c0 + col) * V;
  auto load = [&](const T* p, float (&v)[V]) {
    if constexpr (VEC) P::unpack(*reinterpret_cast<const uint4*>(p), v);
    else v[0] = Elt<T>::load(p);
  };
  constexpr int U = 8;         // rows in flight
  float mx[V], sum[V];
#pragma unroll
  for (int j = 0; j < V; ++j) { mx[j] = -INFINITY; sum[j] = 0.f; }
  if (on) {
    for (int r0 = rl; r0 < S; r0 += U * lanes) {
      float v[U][V];
#pragma unroll
      for (int u = 0; u < U; ++u) load(dw + (size_t)min(r0 + u * lanes, S - 1) * N, v[u]);
#pragma unroll
      for (int j = 0; j < V; ++j) {
        float m = mx[j];
#pragma unroll
        for (int u = 0; u < U; ++u)
          if (r0 + u * lanes < S) m = fmaxf(m, v[u][j]);
        // (a column of nothing but -infinity or NaN so far keeps the maximum -infinity: its
        // exponentials are 0 and NaN, not exp(-inf + inf))
        const float from = m > -INFINITY ? m : 0.f;
        float s = mx[j] == m ? sum[j] : sum[j] * expf(mx[j] - from);
#pragma unroll
        for (int u = 0; u < U; ++u)
          if (r0 + u * lanes < S) s += expf(v[u][j] - from);
        mx[j] = m;
        sum[j] = s;
      }
    }
  }
  if (rl < lanes) {
#pragma unroll
    for (int j = 0; j < V; ++j) {
      lds[rl * width + col * V + j] = mx[j];
      lds2[rl * width + col * V + j] = sum[j];
    }
  }
  __syncthreads();
  // The row lanes of a column are joined in two steps: `parts` threads per column first, each with
  // every parts-th lane, then one; its first row lane's place takes the maximum and the sum.
  auto join = [&](int c, int first, int step, int end) {
    float m = -INFINITY, s = 0.f;
    for (int l = first; l < end; l += step) m = fmaxf(m, lds[l * width + c]);
    const float from = m > -INFINITY ? m : 0.f;       // (every lane's sum counts: a NaN item spoils its column)
    for (int l = first; l < end; l += step) s += lds2[l * width + c] * expf(lds[l * width + c] - from);
    return make_float2(m, s);
  };
  const int parts = min(lanes, kColThreads / width);
  if (parts > 1) {
    const int c = tid % width, part = tid / width;
    float2 ms = make_float2(0.f, 0.f);
    if (part < parts) ms = join(c, part, parts, lanes);
    __syncthreads();
    if (part < parts) { lds[part * width + c] = ms.x; lds2[part * width + c] = ms.y; }
    __syncthreads();
  }
  for (int c = tid; c < width; c += kColThreads) {
    const float2 ms = join(c, 0, 1, parts > 1 ? parts : lanes);
    lds[c] = ms.x;
    lds2[c] = ms.y;
  }
  __syncthreads();
  if (!on) return;
  float m[V], total[V];
#pragma unroll
  for (int j = 0; j < V; ++j) { m[j] = lds[col * V + j]; total[j] = lds2[col * V + j]; }
  for (int r0 = rl; r0 < S; r0 += U * lanes) {
    float v[U][V];
#pragma unroll
    for (int u = 0; u < U; ++u) load(dw + (size_t)min(r0 + u * lanes, S - 1) * N, v[u]);
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (r0 + u * lanes >= S) continue;
#pragma unroll
      for (int j = 0; j < V; ++j) v[u][j] = expf(v[u][j] - m[j]) / total[j];
      T* p = dw + (size_t)(r0 + u * lanes) * N;
      if constexpr (VEC) *reinterpret_cast<uint4*>(p) = P::pack(v[u]);
      else Elt<T>::store(p, v[u][0]);
    }
  }
}

// float32: the exponentials of a chunk of `columns` slots side by side in LDS (rows of columns + 1), then
// one thread per slot adds its column up in the order of the items.
__global__ __launch_bounds__(kColThreads) void soft_columns_f32_kernel(float* __restrict__ dispatch_w, int S, int N,
                                                                       int columns, int chunks) {
  extern __shared__ __align__(16) float lds[];       // S x (columns + 1), then columns sums
  __shared__ float red[kColThreads];
  const int tid = threadIdx.x;
  const int g = blockIdx.x / chunks, c0 = (blockIdx.x - g * chunks) * columns;
  const int here = min(columns, N - c0), pitch = columns + 1, lanes = kColThreads / here;
  const int col = tid % here, rl = tid / here;
  float* const sums = lds + S * pitch;
  float* dw = dispatch_w + (size_t)g * S * N + c0 + col;
  float mx = -INFINITY;
  if (rl < lanes) {
#pragma unroll 8
    for (int s = rl; s < S; s += lanes) {
      const float l = dw[(size_t)s * N];
      lds[s * pitch + col] = l;
      mx = fmaxf(mx, l);
    }
    red[rl * here + col] = mx;
  }
  __syncthreads();
  for (int l = 0; l < lanes; ++l) mx = fmaxf(mx, red[l * here + col]);
  if (rl < lanes)
#pragma unroll 4
    for (int s = rl; s < S; s += lanes) lds[s * pitch + col] = expf(lds[s * pitch + col] - mx);
  __syncthreads();
  if (tid < here) {
    float sum = 0.f;
#pragma unroll 16
    for (int s = 0; s < S; ++s) sum += lds[s * pitch + tid];
    sums[tid] = sum;
  }
  __syncthreads();
  if (rl < lanes) {
    const float sum = sums[col];
#pragma unroll 4
    for (int s = rl; s < S; s += lanes) dw[(size_t)s * N] = lds[s * pitch + col] / sum;
  }
}

// The router's monitoring sums of a group (vmoe/projects/soft_moe/router.py:119-125): blockIdx.y = 0
// the row extremes of the combine weights, 1 the column extremes of the dispatch weights.
constexpr int kStatThreads = 1024;

template <typename T, bool VEC>
__global__ __launch_bounds__(kStatThreads) void soft_stats_kernel(const T* __restrict__ combine_w,
                                                                  const T* __restrict__ dispatch_w,
                                                                  float* __restrict__ partial, int S, int N,
                                                                  int columns, int lanes) {
  using P = Piece<T>;
  constexpr int V = VEC ? P::V : 1;
  extern __shared__ __align__(16) float lds[];          // twice lanes x (columns * V + 1), then 16 x 2
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int g = blockIdx.x, width = columns * V;
  float* const lds2 = lds + lanes * (width + 1);
  float* const red = lds2 + lanes * (width + 1);
  const int col = tid % columns, rl = tid / columns;
  const bool on = rl < lanes;
  const T* src = dispatch_w + (size_t)g * S * N + (size_t)col * V;
  constexpr int U = VEC ? 4 : 8;         // rows in flight
  float lo_sum = 0.f, hi_sum = 0.f;
  float lo[V], hi[V];
#pragma unroll
  for (int j = 0; j < V; ++j) { lo[j] = INFINITY; hi[j] = -INFINITY; }
  auto take = [&](const T* p, float (&v)[V]) {
    if constexpr (VEC) P::unpack(*reinterpret_cast<const uint4*>(p), v);
    else v[0] = Elt<T>::load(p);
  };
  if (blockIdx.y == 0) {
    // `span` lanes (a power of two) per row, U rows of each at a time.
    const int span = columns > 32 ? 64 : columns > 16 ? 32 : columns > 8 ? 16 : 8;
    const int sl = lane & (span - 1), groups = kStatThreads / span, mine = tid / span;
    const T* base = combine_w + (size_t)g * S * N;
    for (int r0 = mine; r0 < S; r0 += U * groups) {
      float a[U], b[U];
#pragma unroll
      for (int u = 0; u < U; ++u) { a[u] = INFINITY; b[u] = -INFINITY; }
      for (int c = sl; c < columns; c += span) {
        float v[U][V];
#pragma unroll
        for (int u = 0; u < U; ++u) take(base + (size_t)min(r0 + u * groups, S - 1) * N + c * V, v[u]);
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
          for (int j = 0; j < V; ++j) { a[u] = fminf(a[u], v[u][j]); b[u] = fmaxf(b[u], v[u][j]); }
      }
      for (int o = span >> 1; o > 0; o >>= 1)
#pragma unroll
        for (int u = 0; u < U; ++u) {
          a[u] = fminf(a[u], __shfl_xor(a[u], o, 64));
          b[u] = fmaxf(b[u], __shfl_xor(b[u], o, 64));
        }
#pragma unroll
      for (int u = 0; u < U; ++u)
        if (sl == 0 && r0 + u * groups < S) { lo_sum += a[u]; hi_sum += b[u]; }
    }
  } else if (on) {
    for (int r0 = rl; r0 < S; r0 += U * lanes) {
      float v[U][V];
#pragma unroll
      for (int u = 0; u < U; ++u) take(src + (size_t)min(r0 + u * lanes, S - 1) * N, v[u]);   // (a row again at the end)
#pragma unroll
      for (int u = 0; u < U; ++u)
#pragma unroll
        for (int j = 0; j < V; ++j) { lo[j] = fminf(lo[j], v[u][j]); hi[j] = fmaxf(hi[j], v[u][j]); }
    }
  }
  if (blockIdx.y == 1) {
    if (on) {
#pragma unroll
      for (int j = 0; j < V; ++j) {
        lds[rl * width + col * V + j] = lo[j];
        lds2[rl * width + col * V + j] = hi[j];
      }
    }
    __syncthreads();
    for (int c = tid; c < width; c += kStatThreads) {
      float a = lds[c], b = lds2[c];
      for (int l = 1; l < lanes; ++l) {
        a = fminf(a, lds[l * width + c]);
        b = fmaxf(b, lds2[l * width + c]);
      }
      lo_sum += a;
      hi_sum += b;
    }
  }
  lo_sum = wave_sum(lo_sum);
  hi_sum = wave_sum(hi_sum);
  if (lane == 0) { red[wave * 2] = lo_sum; red[wave * 2 + 1] = hi_sum; }
  __syncthreads();
  if (tid < 2) {
    float t = 0.f;
    for (int w = 0; w < kStatThreads / 64; ++w) t += red[w * 2 + tid];
    partial[(size_t)g * 4 + blockIdx.y * 2 + tid] = t;
  }
}

template <typename T>
inline int launch_stats(const T* combine_w, const T* dispatch_w, float* partial, int G, int S, int N,
                        hipStream_t stream) {
  constexpr int V = Piece<T>::V;
  const bool vec = N % V == 0 && aligned16(combine_w) && aligned16(dispatch_w);
  const int columns = vec ? N / V : N;
  int lanes = kStatThreads / columns;
  if (lanes < 1) return VMOE_E_UNSUPPORTED;
  if (lanes > 64) lanes = 64;
  if (lanes > S) lanes = S;
  const size_t lds = ((size_t)2 * lanes * (columns * (vec ? V : 1) + 1) + 64) * sizeof(float);
  auto kern = vec ? soft_stats_kernel<T, true> : soft_stats_kernel<T, false>;
  hipError_t e = allow_dynamic_lds(reinterpret_cast<const void*>(kern), lds);
  if (e != hipSuccess) return (int)e;
  hipLaunchKernelGGL(kern, dim3((unsigned)G, 2), dim3(kStatThreads), lds, stream, combine_w, dispatch_w, partial, S,
                     N, columns, lanes);
  return launch_status();
}

// Whether the tile kernels take the shape: the rows of a 16-row tile and their logits fit LDS.
// (float32: and 8 columns of the group's logits)
template <typename T> inline bool tiles_ok(int S, int D, int N) {
  if (sizeof(T) == 4 && (int64_t)S * 9 > 38 * 1024) return false;
  return D * (int)sizeof(T) <= 8192 && logits_lds<T>(D, N, 16).total <= 160 * 1024;
}

template <typename T>
inline int launch_tiles(const T* x, const void* prepared_mu, T* dispatch_w, T* combine_w, T* logits_out, float scale, int scale_x, int G,
                        int S, int D, int N, hipStream_t stream) {
  constexpr int V = Piece<T>::V;
  const int steps = padded_steps<T>(D);
  const bool vec = sizeof(T) == 2 && N % V == 0 && aligned16(dispatch_w) && aligned16(combine_w) &&
                   (logits_out == nullptr || aligned16(logits_out));
  // Tile height: every workgroup reads all slot parameters, so with many slots taller tiles pay
  // (256 slots: 64 rows, one workgroup of eight waves per CU); with few the loads, the norms and the
  // softmaxes of more workgroups per CU hide each other better.  16 rows where 32 would leave CUs
  // without a tile or leave a CU room for one workgroup only.
  const auto tiles = [&](int rows) { return (int64_t)G * ((S + rows - 1) / rows); };
  int rb = 1;
  if (logits_lds<T>(D, N, 32).total <= 80 * 1024 && tiles(32) >= 256) rb = 2;
  if (N >= 160 && D * (int)sizeof(T) <= 4096 && logits_lds<T>(D, N, 64).total <= 160 * 1024 && tiles(64) >= 128) rb = 4;
  const LogitsLds L = logits_lds<T>(D, N, 16 * rb);
  const int rows = 16 * rb, row_tiles = (S + rows - 1) / rows;
  if ((int64_t)G * row_tiles > 0x7fffffff) return VMOE_E_OVERFLOW;
  const int per_lane = ((D + V - 1) / V + 63) / 64;
  // (the padding up to whole groups of steps is written by the same lanes)
  const int pieces = (steps * 4 + 63) / 64 > per_lane ? (steps * 4 + 63) / 64 : per_lane;
  using Kern = void (*)(const T*, const uint4*, T*, T*, T*, float, int, int, int, int, int, int, LogitsLds);
  const bool pair = N > 16 * 2 * (logits_waves(rb) - 1);       // every wave finds two blocks of slots
  auto pick = [&](auto rb, auto pc) -> Kern {
    constexpr int RB = decltype(rb)::value, PC = decltype(pc)::value;
    if constexpr (sizeof(T) == 2)
      if (vec) return pair ? (Kern)soft_logits_kernel<T, RB, PC, true, true> : (Kern)soft_logits_kernel<T, RB, PC, true, false>;
    return pair ? (Kern)soft_logits_kernel<T, RB, PC, false, true> : (Kern)soft_logits_kernel<T, RB, PC, false, false>;
  };
  // (64 rows and their logits of 160 slots leave a row two pieces per lane at most, 32 rows in half of LDS four)
  auto by_pieces = [&](auto rb) -> Kern {
    constexpr int RB = decltype(rb)::value;
    if (pieces <= 1) return pick(rb, std::integral_constant<int, 1>{});
    if (pieces <= 2 || RB == 4) return pick(rb, std::integral_constant<int, 2>{});
    if (pieces <= 4 || RB == 2) return pick(rb, std::integral_constant<int, RB == 4 ? 2 : 4>{});
    return pick(rb, std::integral_constant<int, RB == 4 ? 2 : RB == 2 ? 4 : 8>{});
  };
  Kern kern = rb == 4   ? by_pieces(std::integral_constant<int, 4>{})
              : rb == 2 ? by_pieces(std::integral_constant<int, 2>{})
                        : by_pieces(std::integral_constant<int, 1>{});
  hipError_t e = allow_dynamic_lds(reinterpret_cast<const void*>(kern), L.total);
  if (e != hipSuccess) return (int)e;
  hipLaunchKernelGGL(kern, dim3((unsigned)(G * row_tiles)), dim3(64 * logits_waves(rb)), L.total, stream, x,
                     (const uint4*)prepared_mu, dispatch_w, combine_w, logits_out, scale, scale_x, S, D, N, steps,
                     row_tiles, L);
  int rc = launch_status();
  if (rc != VMOE_OK) return rc;
  if constexpr (sizeof(T) == 4) {
    int columns = N < 64 ? N : 64;
    while (columns > 8 && ((int64_t)G * ((N + columns - 1) / columns) < 512 || (int64_t)S * (columns + 1) > 16 * 1024))
      columns = (columns + 1) / 2;
    const int chunks = (N + columns - 1) / columns;
    const size_t lds = ((size_t)S * (columns + 1) + columns) * sizeof(float);
    if ((int64_t)G * chunks > 0x7fffffff || lds > 156 * 1024) return VMOE_E_UNSUPPORTED;
    e = allow_dynamic_lds(reinterpret_cast<const void*>(soft_columns_f32_kernel), lds);
    if (e != hipSuccess) return (int)e;
    hipLaunchKernelGGL(soft_columns_f32_kernel, dim3((unsigned)(G * chunks)), dim3(kColThreads), lds, stream,
                       dispatch_w, S, N, columns, chunks);
    return launch_status();
  }
  // Chunks of columns such that the launch has a few workgroups per CU, a row's share of a chunk
  // at least 64 bytes where the row is that long.
  const int all = vec ? N / V : N, least = vec ? 4 : 64 / (int)sizeof(T);
  int columns = all < kColThreads ? all : kColThreads;
  while (columns > least && (int64_t)G * ((all + columns - 1) / columns) < 768) columns = (columns + 1) / 2;
  const int chunks = (all + columns - 1) / columns;
  if ((int64_t)G * chunks > 0x7fffffff) return VMOE_E_OVERFLOW;
  int lanes = kColThreads / columns;
  if (lanes > S) lanes = S;
  auto cols = vec ? soft_columns_kernel<T, true> : soft_columns_kernel<T, false>;
  hipLaunchKernelGGL(cols, dim3((unsigned)(G * chunks)), dim3(kColThreads), 0, stream, dispatch_w, S, N, all, columns,
                     chunks, lanes);
  return launch_status();
}

}  // namespace soft
}  // namespace vmoe
#endif  // VMOE_SOFT_ROUTE_TILES_H_
