// Routing consumers: the quantities the training loop derives from each
// MoE layer's router outputs, computed in one pass over the [T, E] router
// probabilities (or scores) per layer instead of the reference's
// topk + one_hot + mean chains and per-metric host reads.
//
//   topk_stats      weighted top-k selection counts, weighted column sums of
//                   the probabilities, and the k-th / (k+1)-th margin
//                   (src/models/load_balancing.py:45-88,
//                    src/utils/routing_stats.py:53-80, :143-191)
//   seq_stats       per-sequence selection counts and mean normalised scores
//                   of the DeepSeek-V3 sequence-wise loss (load_balancing.py:
//                   134-166), and its backward through the normalisation
//   switch_aux_bwd  the Switch loss gradient, a per-expert coefficient times
//                   a per-token weight
//   seq_aux_loss, switch_aux_loss   either loss of a whole model: the same
//                   passes over all layers at once, and the assembly of the
//                   scalar.  A layer by itself is 8 MB (T = 16384, E = 128),
//                   too little for the chip and less than its launches cost;
//                   16 layers one by one, with ten small tensor operators
//                   each, took 1.33 ms; together 0.27 ms, of it 90 us on the
//                   GPU (statistics 34, gradients 46 us for 270 MB read and
//                   134 MB written) and the rest the caller's host time
//   update_biases   the aux-loss-free expert-bias update of every router in
//                   one launch (train.py:79-139)
//
// Every sum is deterministic: a lane accumulates the experts it owns in
// registers (fp32, at most 16 tokens while the grid may grow), the lane groups
// and waves of a block are combined in order and the block partials in block
// order, both in fp64.  No float atomics.
#include "common.h"
#include "wave_topk.h"

namespace moe {
namespace {

constexpr int kWaves = 4;
constexpr int kTokensPerWave = 8;  // topk_stats: tokens per wave (grid sizing)
constexpr int kSeqChunk = 64;      // seq_stats: tokens per block (one layer)
constexpr int kMaxLayers = 32;     // layers per launch of the whole-model passes

// The layers' tensors of one launch, by value in the kernel's arguments (no
// pointer array to copy to the device).
struct Layers {
  const void* in[kMaxLayers];        // probabilities or scores [T,E]
  const int64_t* sel[kMaxLayers];    // routed indices [T,K] (seq; may be null)
  void* out[kMaxLayers];             // gradients
};

__device__ __forceinline__ float load_val(const void* p, int dtype, int64_t i) {
  return dtype == MOE_DTYPE_BF16 ? bf2f(((const bf16*)p)[i]) : ((const float*)p)[i];
}

int stats_blocks(int64_t T) {
  int64_t b = (T + kWaves * kTokensPerWave - 1) / (kWaves * kTokensPerWave);
  if (b > 1024) b = 1024;
  if (b < 1) b = 1;
  return (int)b;
}

// Combines the four waves' per-lane accumulators of one [E] vector in wave
// order, in fp64, and writes the block's partial: kWaves entries per lane at a
// time, one by each wave.
constexpr int kCombineBuf = kWaves * kWaves * 64;  // floats of `buf`
template <int NV>
__device__ void block_combine(const float (&acc)[NV], int E, float* buf, double* out) {
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
#pragma unroll
  for (int j0 = 0; j0 < NV; j0 += kWaves) {
    __syncthreads();
#pragma unroll
    for (int q = 0; q < kWaves && j0 + q < NV; ++q) buf[(q * kWaves + wid) * 64 + lane] = acc[j0 + q];
    __syncthreads();
    const int e = (j0 + wid) * 64 + lane;
    if (e < E && j0 + wid < NV) {
      double s = 0.0;
#pragma unroll
      for (int w = 0; w < kWaves; ++w) s += (double)buf[(wid * kWaves + w) * 64 + lane];
      out[e] = s;
    }
  }
}

// The same statistics with G lanes per token (E <= 16*G, K <= G): lane g of
// a group owns experts g*V .. g*V+V-1, ranks through rank_key with G-lane DPP
// butterflies (as the softmax router's group kernel).  The block partial is
// the fp64 sum over the block's kWaves*64/G token groups in group order, through
// LDS ([groups][E] floats, dynamic shared memory): only a group's own tokens
// (up to 16, stats_blocks' limit apart) are added in fp32.
template <int G, int V>
__global__ __launch_bounds__(64 * kWaves) void topk_stats_group_kernel(
    Layers layers, int dtype, const float* __restrict__ tok_w, int64_t T, int E,
    int K, double* __restrict__ part_cnt, double* __restrict__ part_sum,
    double* __restrict__ part_margin) {
  const void* const __restrict__ probs = layers.in[blockIdx.y];
  const size_t part = (size_t)blockIdx.y * gridDim.x + blockIdx.x;  // this block's partials
  constexpr int TPW = 64 / G, ROWS = kWaves * TPW;
  extern __shared__ float sbuf[];  // [ROWS][E]
  __shared__ double msh[ROWS], mmn[ROWS];
  const int lane = threadIdx.x & 63, g = lane & (G - 1), sub = lane / G;
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int row = wid * TPW + sub, e0 = g * V;
  const bool vec = E == G * V && (dtype == MOE_DTYPE_F32 ? V % 4 == 0 : V % 8 == 0) &&
                   (((uintptr_t)probs & 15) == 0);
  float cnt[V], psum[V];
#pragma unroll
  for (int j = 0; j < V; ++j) cnt[j] = psum[j] = 0.f;
  double msum = 0.0;
  float mmin = INFINITY;
  const int64_t stride = (int64_t)gridDim.x * kWaves * TPW;
  for (int64_t tb = ((int64_t)blockIdx.x * kWaves + wid) * TPW; tb < T; tb += stride) {
    const int64_t t = tb + sub;
    const bool tok = t < T;
    const int64_t tt = tok ? t : T - 1;
    const float w = tok ? (tok_w ? tok_w[t] : 1.f) : 0.f;
    float v[V];
    if (vec) {
      if (dtype == MOE_DTYPE_F32) {
        const f32x4* src = (const f32x4*)((const float*)probs + tt * E + e0);
#pragma unroll
        for (int q = 0; q < V / 4; ++q) {
          const f32x4 a = src[q];
#pragma unroll
          for (int h = 0; h < 4; ++h) v[4 * q + h] = a[h];
        }
      } else {
        const u32x4* src = (const u32x4*)((const bf16*)probs + tt * E + e0);
#pragma unroll
        for (int q = 0; q < (V + 7) / 8; ++q) {
          const u32x4 a = src[q];
#pragma unroll
          for (int h = 0; h < 8; ++h)
            if (8 * q + h < V) v[8 * q + h] = (h & 1) ? bf_hi(a[h >> 1]) : bf_lo(a[h >> 1]);
        }
      }
    } else {
#pragma unroll
      for (int j = 0; j < V; ++j)
        v[j] = e0 + j < E ? load_val(probs, dtype, tt * E + e0 + j) : -INFINITY;
    }
    uint64_t key[V];
#pragma unroll
    for (int j = 0; j < V; ++j) {
      if (tok && e0 + j < E) psum[j] += w * v[j];
      key[j] = e0 + j < E ? rank_key(v[j], e0 + j) : 0ull;
    }
    float vk = 0.f;  // value of the k-th selection
    for (int k = 0; k < K; ++k) {
      uint64_t b = key[0];
#pragma unroll
      for (int j = 1; j < V; ++j) b = key[j] > b ? key[j] : b;
      b = group_max_key<G>(b);
#pragma unroll
      for (int j = 0; j < V; ++j) key[j] = key[j] == b ? 0ull : key[j];
      vk = key_value(b);
    }
    if (tok) {
#pragma unroll
      for (int j = 0; j < V; ++j)
        if (e0 + j < E && key[j] == 0ull) cnt[j] += w;  // selected (real keys are never 0)
    }
    if (K < E) {  // margin between the k-th and (k+1)-th largest value
      uint64_t b = key[0];
#pragma unroll
      for (int j = 1; j < V; ++j) b = key[j] > b ? key[j] : b;
      b = group_max_key<G>(b);
      const float m = vk - key_value(b);
      if (tok) {
        msum += (double)m;
        mmin = fminf(mmin, m);
      }
    }
  }
  // Block partials: rows in group order, per expert.
  auto combine = [&](const float (&acc)[V], double* out) {
    __syncthreads();
#pragma unroll
    for (int j = 0; j < V; ++j)
      if (e0 + j < E) sbuf[row * E + e0 + j] = acc[j];
    __syncthreads();
    for (int e = threadIdx.x; e < E; e += blockDim.x) {
      double s = 0.0;
      for (int r = 0; r < ROWS; ++r) s += (double)sbuf[r * E + e];
      out[e] = s;
    }
  };
  combine(cnt, part_cnt + part * E);
  combine(psum, part_sum + part * E);
  if (!part_margin) return;
  if (g == 0) {
    msh[row] = msum;
    mmn[row] = (double)mmin;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    double sm = 0.0, mn = INFINITY;
    for (int r = 0; r < ROWS; ++r) {
      sm += msh[r];
      mn = fmin(mn, mmn[r]);
    }
    part_margin[blockIdx.x * 2] = sm;
    part_margin[blockIdx.x * 2 + 1] = mn;
  }
}

// One wave per token (grid-stride).  Per block: partial weighted selection
// counts [E], weighted probability sums [E], and the margin sum and minimum.
template <int NV>
__global__ __launch_bounds__(64 * kWaves) void topk_stats_kernel(
    Layers layers, int dtype, const float* __restrict__ tok_w, int64_t T, int E,
    int K, double* __restrict__ part_cnt, double* __restrict__ part_sum,
    double* __restrict__ part_margin) {
  const void* const __restrict__ probs = layers.in[blockIdx.y];
  const size_t part = (size_t)blockIdx.y * gridDim.x + blockIdx.x;  // this block's partials
  __shared__ float buf[kCombineBuf];
  __shared__ double mbuf[kWaves * 2];
  const int lane = threadIdx.x & 63;
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  float cnt[NV], psum[NV];
#pragma unroll
  for (int j = 0; j < NV; ++j) cnt[j] = psum[j] = 0.f;
  double msum = 0.0;
  float mmin = INFINITY;
  const int64_t nwaves = (int64_t)gridDim.x * kWaves;
  for (int64_t t = (int64_t)blockIdx.x * kWaves + wid; t < T; t += nwaves) {
    const float w = tok_w ? tok_w[t] : 1.f;
    float v[NV];
    uint64_t taken = 0;
#pragma unroll
    for (int j = 0; j < NV; ++j) {
      const int e = j * 64 + lane;
      if (e < E) {
        v[j] = load_val(probs, dtype, t * E + e);
        psum[j] += w * v[j];
      } else {
        v[j] = -INFINITY;
        taken |= 1ull << j;
      }
    }
    const uint64_t pad = taken;
    float vk = 0.f;  // value of the k-th selection
    for (int k = 0; k < K; ++k) {
      float bv;
      int be;
      lane_best<NV>(v, taken, lane, bv, be);
      wave_argmax(bv, be);
      vk = bv;
      if ((be & 63) == lane) taken |= 1ull << (be >> 6);
    }
#pragma unroll
    for (int j = 0; j < NV; ++j)
      if (((taken & ~pad) >> j) & 1ull) cnt[j] += w;
    if (K < E) {  // margin between the k-th and (k+1)-th largest value
      float bv;
      int be;
      lane_best<NV>(v, taken, lane, bv, be);
      wave_argmax(bv, be);
      const float m = vk - bv;
      msum += (double)m;
      mmin = fminf(mmin, m);
    }
  }
  block_combine<NV>(cnt, E, buf, part_cnt + part * E);
  block_combine<NV>(psum, E, buf, part_sum + part * E);
  if (!part_margin) return;
  if (lane == 0) {
    mbuf[wid * 2] = msum;
    mbuf[wid * 2 + 1] = (double)mmin;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    double s = 0.0, m = INFINITY;
    for (int w = 0; w < kWaves; ++w) {
      s += mbuf[w * 2];
      m = fmin(m, mbuf[w * 2 + 1]);
    }
    part_margin[blockIdx.x * 2] = s;
    part_margin[blockIdx.x * 2 + 1] = m;
  }
}

// Fixed-order wave reduction of one fp64 value per lane (butterfly).
__device__ __forceinline__ double wave_sum_f64(double v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}

// One wave per expert (blocks 0..E-1): lane l sums the partials of blocks l,
// l+64, ... in order, then the lanes are combined by a fixed butterfly.
// Block E reduces the margin partials the same way.
__global__ __launch_bounds__(64) void topk_stats_finalize_kernel(
    const double* __restrict__ part_cnt, const double* __restrict__ part_sum,
    const double* __restrict__ part_margin, int nblk, int E, double* __restrict__ counts,
    double* __restrict__ sums, double* __restrict__ margin) {
  const int lane = threadIdx.x, e = blockIdx.x;
  if (e < E) {
    double c = 0.0, s = 0.0;
    for (int b = lane; b < nblk; b += 64) {
      c += part_cnt[(size_t)b * E + e];
      s += part_sum[(size_t)b * E + e];
    }
    c = wave_sum_f64(c);
    s = wave_sum_f64(s);
    if (lane == 0) {
      counts[e] = c;
      sums[e] = s;
    }
  } else {
    double s = 0.0, m = INFINITY;
    for (int b = lane; b < nblk; b += 64) {
      s += part_margin[b * 2];
      m = fmin(m, part_margin[b * 2 + 1]);
    }
    s = wave_sum_f64(s);
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) m = fmin(m, __shfl_xor(m, o, 64));
    if (lane == 0) {
      margin[0] = s;
      margin[1] = m;
    }
  }
}

// Block (c, b, l): tokens [c*chunk, ...) of sequence b of layer l.  Normalised scores
// s' = s / (sum s + 1e-20) per token; per block the selection counts of the
// sequence's experts (the routed indices if given, else the top-k of s') and
// the sums of s'.
// seq_stats with G lanes per token (as topk_stats_group_kernel): block
// (chunk c, sequence b, layer l) covers chunk tokens; the partial is the sum over
// the block's token groups in group order through LDS.
// Lane g of a group holds experts (q*G + g)*4 + h in entry 4q + h, so that a
// row moves as whole 128- or 256-byte pieces (with V consecutive experts per
// lane the gradient's stores were 16 bytes in every 64: 218 us against 46).  Given indices are counted in
// LDS (integers: any order), the top-k of s' in registers.
template <int G>
__device__ __forceinline__ int expert_of(int g, int j) { return ((j >> 2) * G + g) * 4 + (j & 3); }

// Sum of N values as a tree, so that a row's fp32 sum (with the butterfly over
// its G lanes) has log2 E roundings in a chain, as with a wave per row: V
// additions in a row cost the gradient 10% (5.6e-7 against 5.2e-7 from the
// 64-bit one at 16 layers of 8 x 2048 tokens, E = 128).
template <int N>
__device__ __forceinline__ float tree_sum(const float* v) {
  if constexpr (N == 1) return v[0];
  else return tree_sum<N / 2>(v) + tree_sum<N - N / 2>(v + N / 2);
}

// Entries of one row (E == G*V, aligned) as 16-byte (fp32) or 8-byte vectors.
template <int G, int V>
__device__ __forceinline__ void load_row(const void* row0, int dtype, int64_t t, int g,
                                         float (&v)[V]) {
#pragma unroll
  for (int q = 0; q < V / 4; ++q) {
    const int64_t at = t * (G * V) + (q * G + g) * 4;
    if (dtype == MOE_DTYPE_F32) {
      const f32x4 a = *(const f32x4*)((const float*)row0 + at);
#pragma unroll
      for (int h = 0; h < 4; ++h) v[4 * q + h] = a[h];
    } else {
      const u32x2 a = *(const u32x2*)((const bf16*)row0 + at);
#pragma unroll
      for (int h = 0; h < 4; ++h) v[4 * q + h] = (h & 1) ? bf_hi(a[h >> 1]) : bf_lo(a[h >> 1]);
    }
  }
}

template <int G, int V>
__global__ __launch_bounds__(64 * kWaves) void seq_stats_group_kernel(
    Layers layers, int dtype, int64_t S, int chunk, int E, int K, double* __restrict__ part_cnt,
    double* __restrict__ part_sum) {
  const void* const __restrict__ scores = layers.in[blockIdx.z];
  const int64_t* const __restrict__ selected = layers.sel[blockIdx.z];
  constexpr int TPW = 64 / G, ROWS = kWaves * TPW;
  extern __shared__ float sbuf[];  // [ROWS][E], then int counts [E]
  int* const hist = (int*)(sbuf + ROWS * E);
  const int lane = threadIdx.x & 63, g = lane & (G - 1), sub = lane / G;
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int row = wid * TPW + sub;
  const int b = blockIdx.y, c = blockIdx.x;
  const bool vec = E == G * V && (((uintptr_t)scores & 15) == 0);
  float cnt[V], psum[V];
#pragma unroll
  for (int j = 0; j < V; ++j) cnt[j] = psum[j] = 0.f;
  if (selected) {
    for (int e = threadIdx.x; e < E; e += blockDim.x) hist[e] = 0;
    __syncthreads();
  }
  const int64_t s0 = (int64_t)c * chunk;
  const int64_t s1 = s0 + chunk < S ? s0 + chunk : S;
  for (int64_t sb = s0 + (int64_t)wid * TPW; sb < s1; sb += kWaves * TPW) {
    const int64_t st = sb + sub;
    const bool tok = st < s1;
    const int64_t t = (int64_t)b * S + (tok ? st : s1 - 1);
    const int64_t ek = (selected && tok && g < K) ? selected[t * K + g] : -1;
    float v[V];
    if (vec) {
      load_row<G, V>(scores, dtype, t, g, v);
    } else {
#pragma unroll
      for (int j = 0; j < V; ++j) {
        const int e = expert_of<G>(g, j);
        v[j] = e < E ? load_val(scores, dtype, t * E + e) : 0.f;
      }
    }
    const float rs = group_sum<G>(tree_sum<V>(v)) + 1e-20f;
#pragma unroll
    for (int j = 0; j < V; ++j) {
      v[j] = v[j] / rs;
      if (tok) psum[j] += v[j];  // entries past E are zero
    }
    if (selected) {
      if (ek >= 0 && ek < E) atomicAdd(&hist[ek], 1);
    } else {
      uint64_t key[V];
#pragma unroll
      for (int j = 0; j < V; ++j) {
        const int e = expert_of<G>(g, j);
        key[j] = e < E ? rank_key(v[j], e) : 0ull;
      }
      for (int k = 0; k < K; ++k) {
        uint64_t m = key[0];
#pragma unroll
        for (int j = 1; j < V; ++j) m = key[j] > m ? key[j] : m;
        m = group_max_key<G>(m);
#pragma unroll
        for (int j = 0; j < V; ++j) key[j] = key[j] == m ? 0ull : key[j];
      }
      if (tok) {
#pragma unroll
        for (int j = 0; j < V; ++j)
          if (expert_of<G>(g, j) < E && key[j] == 0ull) cnt[j] += 1.f;  // selected (real keys are never 0)
      }
    }
  }
  const size_t slot = (((size_t)blockIdx.z * gridDim.y + b) * gridDim.x + c) * E;
  auto combine = [&](const float (&acc)[V], double* out) {
    __syncthreads();
#pragma unroll
    for (int j = 0; j < V; ++j)
      if (expert_of<G>(g, j) < E) sbuf[row * E + expert_of<G>(g, j)] = acc[j];
    __syncthreads();
    for (int e = threadIdx.x; e < E; e += blockDim.x) {
      double sm = 0.0;
      for (int r = 0; r < ROWS; ++r) sm += (double)sbuf[r * E + e];
      out[e] = sm;
    }
  };
  combine(psum, part_sum + slot);  // (its barriers come after every count)
  if (selected) {
    for (int e = threadIdx.x; e < E; e += blockDim.x) part_cnt[slot + e] = (double)hist[e];
  } else {
    combine(cnt, part_cnt + slot);
  }
}

template <int NV>
__global__ __launch_bounds__(64 * kWaves) void seq_stats_kernel(
    Layers layers, int dtype, int64_t S, int chunk, int E, int K, double* __restrict__ part_cnt,
    double* __restrict__ part_sum) {
  const void* const __restrict__ scores = layers.in[blockIdx.z];
  const int64_t* const __restrict__ selected = layers.sel[blockIdx.z];
  __shared__ float buf[kCombineBuf];
  const int lane = threadIdx.x & 63;
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int b = blockIdx.y, c = blockIdx.x;
  float cnt[NV], psum[NV];
#pragma unroll
  for (int j = 0; j < NV; ++j) cnt[j] = psum[j] = 0.f;
  const int64_t s0 = (int64_t)c * chunk;
  const int64_t s1 = s0 + chunk < S ? s0 + chunk : S;
  for (int64_t st = s0 + wid; st < s1; st += kWaves) {
    const int64_t t = (int64_t)b * S + st;
    float v[NV];
    uint64_t taken = 0;
    float rs = 0.f;
#pragma unroll
    for (int j = 0; j < NV; ++j) {
      const int e = j * 64 + lane;
      v[j] = e < E ? load_val(scores, dtype, t * E + e) : 0.f;
      rs += v[j];
      if (e >= E) taken |= 1ull << j;
    }
    rs = wave_sum(rs) + 1e-20f;
#pragma unroll
    for (int j = 0; j < NV; ++j) {
      v[j] = v[j] / rs;
      psum[j] += v[j];
    }
    if (selected) {
      for (int k = 0; k < K; ++k) {
        const int64_t ek = selected[t * K + k];
        if (ek >= 0 && ek < E && (ek & 63) == lane) {
#pragma unroll
          for (int j = 0; j < NV; ++j)
            if ((ek >> 6) == j) cnt[j] += 1.f;
        }
      }
    } else {
      const uint64_t pad = taken;
#pragma unroll
      for (int j = 0; j < NV; ++j)
        if ((pad >> j) & 1ull) v[j] = -INFINITY;
      for (int k = 0; k < K; ++k) {
        float bv;
        int be;
        lane_best<NV>(v, taken, lane, bv, be);
        wave_argmax(bv, be);
        if ((be & 63) == lane) taken |= 1ull << (be >> 6);
      }
#pragma unroll
      for (int j = 0; j < NV; ++j)
        if (((taken & ~pad) >> j) & 1ull) cnt[j] += 1.f;
    }
  }
  const size_t slot = (((size_t)blockIdx.z * gridDim.y + b) * gridDim.x + c) * E;
  block_combine<NV>(cnt, E, buf, part_cnt + slot);
  block_combine<NV>(psum, E, buf, part_sum + slot);
}

// One wave per (b, e): counts[b][e] = sum over chunks, mean[b][e] = sum over
// chunks / S, in the fixed order of wave_sum_f64.
__global__ __launch_bounds__(64) void seq_stats_finalize_kernel(
    const double* __restrict__ part_cnt, const double* __restrict__ part_sum, int nchunk, int B,
    int E, int64_t S, double* __restrict__ counts, double* __restrict__ mean) {
  const int lane = threadIdx.x;
  const int64_t i = blockIdx.x;
  const int b = (int)(i / E), e = (int)(i % E);
  double c = 0.0, s = 0.0;
  for (int k = lane; k < nchunk; k += 64) {
    const size_t o = ((size_t)b * nchunk + k) * E + e;
    c += part_cnt[o];
    s += part_sum[o];
  }
  c = wave_sum_f64(c);
  s = wave_sum_f64(s);
  if (lane == 0) {
    counts[i] = c;
    mean[i] = s / (double)S;
  }
}

// Sum of one fp64 value per thread over a block of 256 or 1024 threads, in a
// fixed order; every thread gets it.  tmp: 17 doubles of LDS.
__device__ double block_sum_f64(double v, double* tmp) {
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6, nw = blockDim.x >> 6;
  v = wave_sum_f64(v);
  __syncthreads();
  if (lane == 0) tmp[wid] = v;
  __syncthreads();
  double s = 0.0;
  for (int w = 0; w < nw; ++w) s += tmp[w];
  return s;
}

// Sequence-wise loss, block (b, l): per expert, its selections c and the sum
// of its normalised scores over the sequence's chunks (in chunk order, a
// thread per expert: rows of partials are read whole), f = c * f_scale, the
// gradient coefficient coef[l][b][e] = f * coef_scale, and the block's part
// sum_e f * mean score of the loss.
__global__ __launch_bounds__(256) void seq_loss_finalize_kernel(
    const double* __restrict__ part_cnt, const double* __restrict__ part_sum, int nchunk, int E,
    int64_t S, double f_scale, double coef_scale, double* __restrict__ coef,
    double* __restrict__ part_loss) {
  __shared__ double tmp[17];
  const size_t lb = (size_t)blockIdx.y * gridDim.x + blockIdx.x;
  double loss = 0.0;
  for (int e = threadIdx.x; e < E; e += 256) {
    double c = 0.0, s = 0.0;
    const double* pc = part_cnt + lb * nchunk * E + e;
    const double* ps = part_sum + lb * nchunk * E + e;
#pragma unroll 8
    for (int k = 0; k < nchunk; ++k) {
      c += pc[(size_t)k * E];
      s += ps[(size_t)k * E];
    }
    const double f = c * f_scale;
    coef[lb * E + e] = f * coef_scale;
    loss += f * (s / (double)S);
  }
  loss = block_sum_f64(loss, tmp);
  if (threadIdx.x == 0) part_loss[lb] = loss;
}

// loss = scale * sum of n parts, in a fixed order.
__global__ __launch_bounds__(256) void loss_sum_kernel(const double* __restrict__ part, int n,
                                                       double scale, double* __restrict__ loss64,
                                                       float* __restrict__ loss) {
  __shared__ double tmp[17];
  double s = 0.0;
  for (int i = threadIdx.x; i < n; i += 256) s += part[i];
  s = block_sum_f64(s, tmp);
  if (threadIdx.x == 0) {
    *loss64 = s * scale;
    *loss = (float)(s * scale);
  }
}

// Switch loss, block (l, i): layer l's counts and sums of 64 experts from its
// blocks' partials (sums64: [L][2][E]); the 16 waves take the partials in turn
// and are added in wave order.  (One block per layer read a wide layer's
// partials alone: 16384 x 1792 with gradients 672 us, now 446.)
__global__ __launch_bounds__(1024) void switch_layer_sums_kernel(
    const double* __restrict__ part_cnt, const double* __restrict__ part_sum, int nblk, int E,
    double* __restrict__ sums64) {
  __shared__ double red[2][16][64];
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  const size_t base = (size_t)blockIdx.x * nblk * E;
  const int e = blockIdx.y * 64 + lane;
  double c = 0.0, s = 0.0;
  if (e < E)
#pragma unroll 4
    for (int k = wid; k < nblk; k += 16) {
      c += part_cnt[base + (size_t)k * E + e];
      s += part_sum[base + (size_t)k * E + e];
    }
  red[0][wid][lane] = c;
  red[1][wid][lane] = s;
  __syncthreads();
  if (wid < 2 && e < E) {
    double v = 0.0;
    for (int w = 0; w < 16; ++w) v += red[wid][w][lane];
    sums64[((size_t)blockIdx.x * 2 + wid) * E + e] = v;
  }
}

// ... and the loss E * sum_e (counts / d) (sums / d) with the gradient
// coefficients coef[e] = counts / d * num_experts / d; d = denom, or
// denom * *denom_dev.
__global__ __launch_bounds__(1024) void switch_loss_kernel(
    const double* __restrict__ sums64, int L, int E, double num_experts, double denom,
    const double* __restrict__ denom_dev, double* __restrict__ coef, double* __restrict__ loss) {
  __shared__ double tmp[17];
  const double d = denom_dev ? denom * *denom_dev : denom;
  double acc = 0.0;
  for (int e = threadIdx.x; e < E; e += 1024) {
    double c = 0.0, s = 0.0;
    for (int l = 0; l < L; ++l) {
      c += sums64[((size_t)l * 2) * E + e];
      s += sums64[((size_t)l * 2 + 1) * E + e];
    }
    const double tpe = c / d;
    coef[e] = tpe * (num_experts / d);
    acc += tpe * (s / d);
  }
  acc = block_sum_f64(acc, tmp);
  if (threadIdx.x == 0) *loss = acc * num_experts;
}

// Sum of one fp64 value per lane over groups of G lanes.
template <int G>
__device__ __forceinline__ double group_sum_f64(double v) {
  group_steps<G>([&](auto c) {
    const uint64_t b = __builtin_bit_cast(uint64_t, v);
    const uint32_t lo = dpp_u32<decltype(c)::value>((uint32_t)b);
    const uint32_t hi = dpp_u32<decltype(c)::value>((uint32_t)(b >> 32));
    v += __builtin_bit_cast(double, (uint64_t)hi << 32 | lo);
  });
  return v;
}

// Gradient of the sequence-wise loss with G lanes per token (E == G*V), all
// layers in one launch: block (c, b, l) holds its lanes' coefficients of
// sequence b in registers and streams tokens [c*chunk, ...) through 16-byte
// vectors.  seq_aux_bwd_kernel's formula, with the inner product <g, s'> and
// its difference from g in fp64: balanced routing cancels most of g there, and
// in fp32 the roundings of the products (each on its own, where a lane of the
// wave-per-row kernel fuses all but its first) were most of the error: 2-norm
// 4.9e-7 -> 3.4e-7 from 64 bits at E = 128, 9.5e-7 -> 6.1e-7 at 64, in the same
// time (49 us for 16 layers of 16384 x 128).
template <int G, int V>
__global__ __launch_bounds__(64 * kWaves) void seq_aux_bwd_group_kernel(
    Layers layers, int dtype, const double* __restrict__ coef, const float* __restrict__ grad,
    int64_t S, int chunk) {
  constexpr int TPW = 64 / G, E = G * V;
  const int lane = threadIdx.x & 63, g = lane & (G - 1), sub = lane / G;
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int b = blockIdx.y;
  const void* const __restrict__ scores = layers.in[blockIdx.z];
  void* const __restrict__ out = layers.out[blockIdx.z];
  const double up = grad ? (double)*grad : 1.0;
  double gc[V];
#pragma unroll
  for (int j = 0; j < V; ++j)
    gc[j] = coef[((size_t)blockIdx.z * gridDim.y + b) * E + expert_of<G>(g, j)] * up;
  const int64_t s0 = (int64_t)blockIdx.x * chunk;
  const int64_t s1 = s0 + chunk < S ? s0 + chunk : S;
  for (int64_t sb = s0 + (int64_t)wid * TPW; sb < s1; sb += kWaves * TPW) {
    const int64_t st = sb + sub;
    const bool tok = st < s1;
    const int64_t t = (int64_t)b * S + (tok ? st : s1 - 1);
    float v[V];
    load_row<G, V>(scores, dtype, t, g, v);
    const float rs = group_sum<G>(tree_sum<V>(v)) + 1e-20f;
    double dot = 0.0;
#pragma unroll
    for (int j = 0; j < V; ++j) dot = fma(gc[j], (double)(v[j] / rs), dot);
    dot = group_sum_f64<G>(dot);
    if (!tok) continue;
#pragma unroll
    for (int q = 0; q < V / 4; ++q) {
      float d[4];
#pragma unroll
      for (int h = 0; h < 4; ++h) d[h] = (float)(gc[4 * q + h] - dot) / rs;
      const int64_t at = t * E + (q * G + g) * 4;
      if (dtype == MOE_DTYPE_F32) *(f32x4*)((float*)out + at) = f32x4{d[0], d[1], d[2], d[3]};
      else *(u32x2*)((bf16*)out + at) = u32x2{pack_bf2(d[0], d[1]), pack_bf2(d[2], d[3])};
    }
  }
}

// d s from d s' through s' = s / (sum s + eps): (g - <g, s'>) / (sum s + eps),
// with g[t][e] = coef[l][b(t)][e] (times *grad when given), layer l = blockIdx.y.
template <int NV>
__global__ __launch_bounds__(64 * kWaves) void seq_aux_bwd_kernel(
    Layers layers, int dtype, const double* __restrict__ coef_all, const float* __restrict__ grad,
    int64_t T, int64_t S, int E) {
  const void* const __restrict__ scores = layers.in[blockIdx.y];
  void* const __restrict__ d_scores = layers.out[blockIdx.y];
  const double* const __restrict__ coef = coef_all + (size_t)blockIdx.y * (T / S) * E;
  const double up = grad ? (double)*grad : 1.0;
  const int lane = threadIdx.x & 63;
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t nwaves = (int64_t)gridDim.x * kWaves;
  for (int64_t t = (int64_t)blockIdx.x * kWaves + wid; t < T; t += nwaves) {
    const int64_t b = t / S;
    float v[NV], g[NV];
    float rs = 0.f;
#pragma unroll
    for (int j = 0; j < NV; ++j) {
      const int e = j * 64 + lane;
      v[j] = e < E ? load_val(scores, dtype, t * E + e) : 0.f;
      g[j] = e < E ? (float)(coef[b * E + e] * up) : 0.f;
      rs += v[j];
    }
    rs = wave_sum(rs) + 1e-20f;
    float dot = 0.f;
#pragma unroll
    for (int j = 0; j < NV; ++j) dot += g[j] * (v[j] / rs);
    dot = wave_sum(dot);
#pragma unroll
    for (int j = 0; j < NV; ++j) {
      const int e = j * 64 + lane;
      if (e < E) {
        const float d = (g[j] - dot) / rs;
        if (dtype == MOE_DTYPE_BF16) ((bf16*)d_scores)[t * E + e] = f2bf(d);
        else ((float*)d_scores)[t * E + e] = d;
      }
    }
  }
}

// grad[t][e] = coef[e] * *up * (w ? w[t] : 1), four experts at a time (E % 4
// == 0), all layers in one launch.
__global__ __launch_bounds__(256) void switch_aux_bwd_vec_kernel(Layers layers,
                                                                 const double* __restrict__ coef,
                                                                 const float* __restrict__ up,
                                                                 const float* __restrict__ tok_w,
                                                                 int64_t T, int E, int dtype) {
  void* const __restrict__ grad = layers.out[blockIdx.y];
  const int q = E / 4;
  const double u = (double)*up;
  const int64_t stride = (int64_t)gridDim.x * 256;
  const int64_t n = T * (int64_t)q;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += stride) {
    const int64_t t = i / q;
    const int e = (int)(i - t * q) * 4;
    const float w = tok_w ? tok_w[t] : 1.f;
    float g[4];
#pragma unroll
    for (int h = 0; h < 4; ++h) g[h] = (float)(coef[e + h] * u) * w;
    if (dtype == MOE_DTYPE_BF16)
      ((u32x2*)grad)[i] = u32x2{pack_bf2(g[0], g[1]), pack_bf2(g[2], g[3])};
    else __builtin_nontemporal_store(f32x4{g[0], g[1], g[2], g[3]}, (f32x4*)grad + i);
  }
}

// The same of one layer, any E.
__global__ __launch_bounds__(256) void switch_aux_bwd_kernel(const double* __restrict__ coef,
                                                             const float* __restrict__ up,
                                                             const float* __restrict__ tok_w,
                                                             int64_t T, int E, int dtype,
                                                             void* __restrict__ grad) {
  const double u = up ? (double)*up : 1.0;
  const int64_t n = T * (int64_t)E;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x) {
    const int64_t t = i / E;
    const int e = (int)(i - t * E);
    const float g = (float)(coef[e] * u) * (tok_w ? tok_w[t] : 1.f);
    if (dtype == MOE_DTYPE_BF16) ((bf16*)grad)[i] = f2bf(g);
    else ((float*)grad)[i] = g;
  }
}

// One block: every router's bias moves by sign(mean - count) * rate (per
// layer, pooled over layers, or alpha-blended), in fp32 with the reference's
// operation order; counts are then zeroed.  stats = mean, unbiased std, min,
// max of all new biases (fp64).
__global__ __launch_bounds__(1024) void update_biases_kernel(float* const* __restrict__ counts,
                                                             float* const* __restrict__ biases,
                                                             int L, int E, float rate,
                                                             int is_global, float alpha,
                                                             float one_minus_alpha,
                                                             double* __restrict__ stats) {
  extern __shared__ float sh[];  // lmean[L+1] (per layer, then pooled), pool[E]
  __shared__ double red[1024];
  float* lmean = sh;
  float* pool = sh + L + 1;
  const int tid = threadIdx.x;
  // Counts are integers below 2^24, so every fp32 sum below is exact in any
  // order and each mean is one rounding of sum / E, as in the reference.
  for (int e = tid; e < E; e += blockDim.x) {
    float s = 0.f;
    for (int k = 0; k < L; ++k) s += counts[k][e];
    pool[e] = s;
  }
  for (int l = tid; l < L; l += blockDim.x) {
    float s = 0.f;
    for (int e = 0; e < E; ++e) s += counts[l][e];
    lmean[l] = s / (float)E;
  }
  __syncthreads();
  if (tid == 0) {
    float s = 0.f;
    for (int e = 0; e < E; ++e) s += pool[e];
    lmean[L] = s / (float)E;
  }
  __syncthreads();
  auto sgn = [](float x) { return (float)((x > 0.f) - (x < 0.f)); };
  for (int64_t i = tid; i < (int64_t)L * E; i += blockDim.x) {
    const int l = (int)(i / E), e = (int)(i % E);
    const float c = counts[l][e];
    float d;
    if (is_global) {
      const float gd = sgn(lmean[L] - pool[e]) * rate;
      if (alpha > 0.f) {
        const float ld = sgn(lmean[l] - c) * rate;
        d = __fadd_rn(__fmul_rn(alpha, ld), __fmul_rn(one_minus_alpha, gd));
      } else {
        d = gd;
      }
    } else {
      d = sgn(lmean[l] - c) * rate;
    }
    biases[l][e] = __fadd_rn(biases[l][e], d);
  }
  __syncthreads();
  for (int64_t i = tid; i < (int64_t)L * E; i += blockDim.x) counts[i / E][i % E] = 0.f;
  // Statistics of the new biases (fixed-order tree reductions).
  const int64_t n = (int64_t)L * E;
  double s = 0.0, mn = INFINITY, mx = -INFINITY;
  for (int64_t i = tid; i < n; i += blockDim.x) {
    const double v = (double)biases[i / E][i % E];
    s += v;
    mn = fmin(mn, v);
    mx = fmax(mx, v);
  }
  auto tree = [&](double v, int op) {
    red[tid] = v;
    __syncthreads();
    for (int o = blockDim.x / 2; o > 0; o >>= 1) {
      if (tid < o) {
        const double a = red[tid], b2 = red[tid + o];
        red[tid] = op == 0 ? a + b2 : (op == 1 ? fmin(a, b2) : fmax(a, b2));
      }
      __syncthreads();
    }
    const double r = red[0];
    __syncthreads();
    return r;
  };
  const double mean = tree(s, 0) / (double)n;
  mn = tree(mn, 1);
  mx = tree(mx, 2);
  double q = 0.0;
  for (int64_t i = tid; i < n; i += blockDim.x) {
    const double v = (double)biases[i / E][i % E] - mean;
    q += v * v;
  }
  q = tree(q, 0);
  if (tid == 0) {
    stats[0] = mean;
    stats[1] = n > 1 ? sqrt(q / (double)(n - 1)) : 0.0;
    stats[2] = mn;
    stats[3] = mx;
  }
}

#define MOE_DISPATCH_NV_B(E, KERNEL, ...)                        \
  do {                                                           \
    int nv_ = ((E) + 63) / 64;                                   \
    if (nv_ <= 1) KERNEL<1><<<__VA_ARGS__;                       \
    else if (nv_ <= 2) KERNEL<2><<<__VA_ARGS__;                  \
    else if (nv_ <= 4) KERNEL<4><<<__VA_ARGS__;                  \
    else if (nv_ <= 8) KERNEL<8><<<__VA_ARGS__;                  \
    else if (nv_ <= 16) KERNEL<16><<<__VA_ARGS__;                \
    else if (nv_ <= 32) KERNEL<32><<<__VA_ARGS__;                \
    else KERNEL<64><<<__VA_ARGS__;                               \
  } while (0)

int check_stats_shape(int64_t T, int E, int K, int dtype, const char* who) {
  MOE_REQUIRE(T >= 0 && E >= 1 && E <= 4096, MOE_ERR_ARG, "%s: T=%lld E=%d out of range", who,
              (long long)T, E);
  MOE_REQUIRE(K >= 1 && K <= E && K <= 64, MOE_ERR_ARG, "%s: K=%d outside [1,min(E,64)]", who, K);
  MOE_REQUIRE(dtype == MOE_DTYPE_F32 || dtype == MOE_DTYPE_BF16, MOE_ERR_DTYPE,
              "%s: dtype %d (fp32 or bf16)", who, dtype);
  return MOE_OK;
}

size_t seq_chunks(int64_t S) { return (size_t)((S + kSeqChunk - 1) / kSeqChunk); }

// topk_stats of layers, nb blocks each (partials [layer][block][E]).
void launch_topk_stats(const Layers& layers, int nl, int dtype, const float* token_weights,
                       int64_t T, int E, int K, int nb, double* pc, double* ps, double* pm,
                       hipStream_t st) {
  int G, V;
  group_shape(E, K, G, V);
  const dim3 grid(nb, nl);
  if (G) {
    const size_t shm = (size_t)kWaves * (64 / G) * E * sizeof(float);
#define MOE_STATS_GROUP(G_, V_)                                                               \
  topk_stats_group_kernel<G_, V_><<<grid, 64 * kWaves, shm, st>>>(layers, dtype, token_weights, \
                                                                  T, E, K, pc, ps, pm)
    if (G == 8 && V == 4) MOE_STATS_GROUP(8, 4);
    else if (G == 8 && V == 8) MOE_STATS_GROUP(8, 8);
    else if (G == 8) MOE_STATS_GROUP(8, 16);
    else if (V == 4) MOE_STATS_GROUP(16, 4);
    else if (V == 8) MOE_STATS_GROUP(16, 8);
    else MOE_STATS_GROUP(16, 16);
#undef MOE_STATS_GROUP
  } else {
    MOE_DISPATCH_NV_B(E, topk_stats_kernel, grid, 64 * kWaves, 0, st>>>(
        layers, dtype, token_weights, T, E, K, pc, ps, pm));
  }
}

// seq_stats of nl layers, nc chunks of `chunk` tokens per sequence (partials
// [layer][sequence][chunk][E]).
void launch_seq_stats(const Layers& layers, int nl, int dtype, int64_t S, int B, int nc, int chunk,
                      int E, int K, double* pc, double* ps, hipStream_t st) {
  int G, V;
  group_shape(E, K, G, V);
  const dim3 grid(nc, B, nl);
  if (G) {
    const size_t shm = ((size_t)kWaves * (64 / G) + 1) * E * sizeof(float);
#define MOE_SEQ_GROUP(G_, V_)                                                               \
  seq_stats_group_kernel<G_, V_><<<grid, 64 * kWaves, shm, st>>>(layers, dtype, S, chunk, E, K, \
                                                                 pc, ps)
    if (G == 8 && V == 4) MOE_SEQ_GROUP(8, 4);
    else if (G == 8 && V == 8) MOE_SEQ_GROUP(8, 8);
    else if (G == 8) MOE_SEQ_GROUP(8, 16);
    else if (V == 4) MOE_SEQ_GROUP(16, 4);
    else if (V == 8) MOE_SEQ_GROUP(16, 8);
    else MOE_SEQ_GROUP(16, 16);
#undef MOE_SEQ_GROUP
  } else {
    MOE_DISPATCH_NV_B(E, seq_stats_kernel, grid, 64 * kWaves, 0, st>>>(layers, dtype, S, chunk, E,
                                                                      K, pc, ps));
  }
}

// Gradient of the sequence-wise loss of nl layers; every tensor 16-byte
// aligned (vec) takes the group kernel where E fills the lanes.
void launch_seq_bwd(const Layers& layers, int nl, bool vec, int dtype, const double* coef,
                    const float* grad, int64_t T, int E, int B, hipStream_t st) {
  const int64_t S = T / B;
  // 256 tokens per block; 64 while that leaves the chip short of blocks
  const int chunk = (S + 255) / 256 * B * nl >= 1024 ? 256 : 64;
  const dim3 grid((unsigned)((S + chunk - 1) / chunk), B, nl);
#define MOE_SEQ_BWD(G_, V_)                                                                     \
  seq_aux_bwd_group_kernel<G_, V_><<<grid, 64 * kWaves, 0, st>>>(layers, dtype, coef, grad, S, \
                                                                 chunk)
  if (vec && B < 65536 && E == 128) MOE_SEQ_BWD(8, 16);
  else if (vec && B < 65536 && E == 64) MOE_SEQ_BWD(8, 8);
  else if (vec && B < 65536 && E == 32) MOE_SEQ_BWD(8, 4);
  else if (vec && B < 65536 && E == 256) MOE_SEQ_BWD(16, 16);
  else {
    int64_t nb = (T + kWaves * 8 - 1) / (kWaves * 8);
    if (nb > 4096) nb = 4096;
    MOE_DISPATCH_NV_B(E, seq_aux_bwd_kernel, dim3((unsigned)nb, nl), 64 * kWaves, 0,
                      st>>>(layers, dtype, coef, grad, T, S, E));
  }
#undef MOE_SEQ_BWD
}

bool group_lanes(int E, int K) {  // the kernels with G lanes per token
  int G, V;
  group_shape(E, K, G, V);
  return G != 0;
}

// Tokens per block of the whole-model sequence statistics: 256 (a block's
// combine costs as much as 100 tokens), 64 while that leaves the chip short of
// blocks, and with a wave per token, which adds its 16 tokens of them in fp32.
int seq_loss_chunk(int L, int64_t S, int B, int E, int K) {
  return group_lanes(E, K) && (S + 255) / 256 * B * L >= 1024 ? 256 : kSeqChunk;
}
// Blocks per layer of the whole-model top-k statistics: what fills the chip,
// and at most 16 tokens per lane group (16 groups or more per block).
int switch_blocks(int L, int64_t T, int E, int K) {
  if (!group_lanes(E, K)) return stats_blocks(T);
  const int64_t nb = stats_blocks(T), few = (T + 255) / 256;
  const int64_t most = 2048 / L > few ? 2048 / L : few;
  return (int)(nb < most ? nb : most);
}

}  // namespace
}  // namespace moe

using namespace moe;

extern "C" size_t moe_amd_topk_stats_workspace_size(int64_t T, int E) {
  if (T < 0 || E < 1) return 0;
  const size_t nb = (size_t)stats_blocks(T);
  return align_up(nb * (size_t)E * 2 * sizeof(double), 16) + nb * 2 * sizeof(double);
}

extern "C" int moe_amd_topk_stats(const void* probs, int probs_dtype, const float* token_weights,
                                  int64_t T, int E, int K, void* workspace,
                                  size_t workspace_bytes, double* counts, double* prob_sums,
                                  double* margin, void* stream) {
  const char* who = "topk_stats";
  int rc = check_stats_shape(T, E, K, probs_dtype, who);
  if (rc) return rc;
  MOE_REQUIRE(counts && prob_sums && margin && (T == 0 || probs), MOE_ERR_ARG,
              "%s: null pointer", who);
  const size_t need = moe_amd_topk_stats_workspace_size(T, E);
  MOE_REQUIRE(workspace && workspace_bytes >= need, MOE_ERR_WORKSPACE,
              "%s: workspace of %zu bytes needed", who, need);
  MOE_REQUIRE(((uintptr_t)workspace & 15) == 0, MOE_ERR_ALIGN, "%s: workspace alignment", who);
  hipStream_t st = (hipStream_t)stream;
  const int nb = stats_blocks(T);
  double* pc = (double*)workspace;
  double* ps = pc + (size_t)nb * E;
  double* pm = (double*)((char*)workspace + align_up((size_t)nb * E * 2 * sizeof(double), 16));
  if (T == 0) {
    topk_stats_finalize_kernel<<<E + 1, 64, 0, st>>>(pc, ps, pm, 0, E, counts, prob_sums, margin);
    return check_launch(who);
  }
  Layers layers{};
  layers.in[0] = probs;
  launch_topk_stats(layers, 1, probs_dtype, token_weights, T, E, K, nb, pc, ps, pm, st);
  topk_stats_finalize_kernel<<<E + 1, 64, 0, st>>>(pc, ps, pm, nb, E, counts, prob_sums, margin);
  return check_launch(who);
}

extern "C" size_t moe_amd_seq_stats_workspace_size(int64_t T, int E, int B) {
  if (T < 0 || E < 1 || B < 1 || T % B) return 0;
  return (size_t)B * seq_chunks(T / B) * (size_t)E * 2 * sizeof(double);
}

extern "C" int moe_amd_seq_stats(const void* scores, int scores_dtype,
                                 const int64_t* selected, int64_t T, int E, int K, int B,
                                 void* workspace, size_t workspace_bytes, double* counts,
                                 double* mean_scores, void* stream) {
  const char* who = "seq_stats";
  int rc = check_stats_shape(T, E, K, scores_dtype, who);
  if (rc) return rc;
  MOE_REQUIRE(B >= 1 && T % B == 0 && T > 0, MOE_ERR_ARG,
              "%s: T=%lld must be a positive multiple of the batch size %d", who, (long long)T,
              B);
  MOE_REQUIRE(scores && counts && mean_scores, MOE_ERR_ARG, "%s: null pointer", who);
  const size_t need = moe_amd_seq_stats_workspace_size(T, E, B);
  MOE_REQUIRE(workspace && workspace_bytes >= need, MOE_ERR_WORKSPACE,
              "%s: workspace of %zu bytes needed", who, need);
  const int64_t S = T / B;
  const int nc = (int)seq_chunks(S);
  MOE_REQUIRE(nc < 65536 && B < 65536 && (int64_t)B * E < ((int64_t)1 << 31), MOE_ERR_UNSUPPORTED,
              "%s: grid too large", who);
  hipStream_t st = (hipStream_t)stream;
  double* pc = (double*)workspace;
  double* ps = pc + (size_t)B * nc * E;
  Layers layers{};
  layers.in[0] = scores;
  layers.sel[0] = selected;
  launch_seq_stats(layers, 1, scores_dtype, S, B, nc, kSeqChunk, E, K, pc, ps, st);
  seq_stats_finalize_kernel<<<(unsigned)((int64_t)B * E), 64, 0, st>>>(pc, ps, nc, B, E, S,
                                                                        counts, mean_scores);
  return check_launch(who);
}

extern "C" int moe_amd_seq_aux_backward(const void* scores, int scores_dtype,
                                        const double* coef, int64_t T, int E, int B,
                                        void* d_scores, void* stream) {
  const char* who = "seq_aux_backward";
  int rc = check_stats_shape(T, E, 1, scores_dtype, who);
  if (rc) return rc;
  MOE_REQUIRE(B >= 1 && T % B == 0, MOE_ERR_ARG, "%s: T must be a multiple of B", who);
  MOE_REQUIRE(T == 0 || (scores && coef && d_scores), MOE_ERR_ARG, "%s: null pointer", who);
  if (T == 0) return MOE_OK;
  Layers layers{};
  layers.in[0] = scores;
  layers.out[0] = d_scores;
  launch_seq_bwd(layers, 1, al16(scores) && al16(d_scores), scores_dtype, coef, nullptr, T, E, B,
                 (hipStream_t)stream);
  return check_launch(who);
}

extern "C" int moe_amd_switch_aux_backward(const double* coef, const float* token_weights,
                                           int64_t T, int E, int grad_dtype, void* grad,
                                           void* stream) {
  const char* who = "switch_aux_backward";
  MOE_REQUIRE(T >= 0 && E >= 1, MOE_ERR_ARG, "%s: bad sizes", who);
  MOE_REQUIRE(grad_dtype == MOE_DTYPE_F32 || grad_dtype == MOE_DTYPE_BF16, MOE_ERR_DTYPE,
              "%s: dtype %d", who, grad_dtype);
  MOE_REQUIRE(T == 0 || (coef && grad), MOE_ERR_ARG, "%s: null pointer", who);
  if (T == 0) return MOE_OK;
  int64_t nb = (T * (int64_t)E + 255) / 256;
  if (nb > 8192) nb = 8192;
  switch_aux_bwd_kernel<<<(unsigned)nb, 256, 0, (hipStream_t)stream>>>(coef, nullptr, token_weights,
                                                                      T, E, grad_dtype, grad);
  return check_launch(who);
}

extern "C" size_t moe_amd_seq_aux_loss_workspace_size(int L, int64_t T, int E, int B) {
  if (L < 1 || T < 1 || E < 1 || B < 1 || T % B) return 0;
  const size_t parts = (size_t)L * B * seq_chunks(T / B) * E;  // the most, whatever K
  return align_up(parts * 2 * sizeof(double), 16) + ((size_t)L * B + 1) * sizeof(double);
}

extern "C" int moe_amd_seq_aux_loss(const void* const* scores, const int64_t* const* selected,
                                    int L, int scores_dtype, int64_t T, int E, int K, int B,
                                    double f_scale, double coef_scale, double loss_scale,
                                    void* workspace, size_t workspace_bytes, double* coef,
                                    double* loss64, float* loss, void* stream) {
  const char* who = "seq_aux_loss";
  int rc = check_stats_shape(T, E, K, scores_dtype, who);
  if (rc) return rc;
  MOE_REQUIRE(L >= 1 && B >= 1 && T > 0 && T % B == 0, MOE_ERR_ARG,
              "%s: L=%d layers, T=%lld must be a positive multiple of the batch size %d", who, L,
              (long long)T, B);
  MOE_REQUIRE(scores && coef && loss64 && loss, MOE_ERR_ARG, "%s: null pointer", who);
  for (int l = 0; l < L; ++l) MOE_REQUIRE(scores[l], MOE_ERR_ARG, "%s: layer %d is null", who, l);
  const size_t need = moe_amd_seq_aux_loss_workspace_size(L, T, E, B);
  MOE_REQUIRE(workspace && workspace_bytes >= need, MOE_ERR_WORKSPACE,
              "%s: workspace of %zu bytes needed", who, need);
  MOE_REQUIRE(((uintptr_t)workspace & 15) == 0, MOE_ERR_ALIGN, "%s: workspace alignment", who);
  const int64_t S = T / B;
  const int chunk = seq_loss_chunk(L, S, B, E, K);
  const int64_t nc64 = (S + chunk - 1) / chunk;
  MOE_REQUIRE(nc64 < 65536 && B < 65536 && L < 65536, MOE_ERR_UNSUPPORTED, "%s: grid too large",
              who);
  const int nc = (int)nc64;
  hipStream_t st = (hipStream_t)stream;
  const size_t per_layer = (size_t)B * nc * E;
  double* pc = (double*)workspace;
  double* ps = pc + (size_t)L * per_layer;
  double* parts = (double*)((char*)workspace + align_up((size_t)L * per_layer * 2 * sizeof(double), 16));
  for (int l0 = 0; l0 < L; l0 += kMaxLayers) {
    const int nl = L - l0 < kMaxLayers ? L - l0 : kMaxLayers;
    Layers layers{};
    for (int l = 0; l < nl; ++l) {
      layers.in[l] = scores[l0 + l];
      layers.sel[l] = selected ? selected[l0 + l] : nullptr;
    }
    launch_seq_stats(layers, nl, scores_dtype, S, B, nc, chunk, E, K, pc + l0 * per_layer,
                     ps + l0 * per_layer, st);
  }
  seq_loss_finalize_kernel<<<dim3(B, L), 256, 0, st>>>(pc, ps, nc, E, S, f_scale, coef_scale, coef,
                                                       parts);
  loss_sum_kernel<<<1, 256, 0, st>>>(parts, L * B, loss_scale, loss64, loss);
  return check_launch(who);
}

extern "C" int moe_amd_seq_aux_loss_backward(const void* const* scores, int L, int scores_dtype,
                                             const double* coef, const float* d_loss, int64_t T,
                                             int E, int B, void* const* d_scores, void* stream) {
  const char* who = "seq_aux_loss_backward";
  int rc = check_stats_shape(T, E, 1, scores_dtype, who);
  if (rc) return rc;
  MOE_REQUIRE(L >= 1 && B >= 1 && T % B == 0, MOE_ERR_ARG, "%s: T must be a multiple of B", who);
  if (T == 0) return MOE_OK;
  MOE_REQUIRE(scores && coef && d_loss && d_scores, MOE_ERR_ARG, "%s: null pointer", who);
  for (int l0 = 0; l0 < L; l0 += kMaxLayers) {
    const int nl = L - l0 < kMaxLayers ? L - l0 : kMaxLayers;
    Layers layers{};
    bool vec = true;
    for (int l = 0; l < nl; ++l) {
      MOE_REQUIRE(scores[l0 + l] && d_scores[l0 + l], MOE_ERR_ARG, "%s: layer %d is null", who,
                  l0 + l);
      layers.in[l] = scores[l0 + l];
      layers.out[l] = d_scores[l0 + l];
      vec = vec && al16(layers.in[l]) && al16(layers.out[l]);
    }
    launch_seq_bwd(layers, nl, vec, scores_dtype, coef + (size_t)l0 * B * E, d_loss, T, E, B,
                   (hipStream_t)stream);
  }
  return check_launch(who);
}

extern "C" size_t moe_amd_switch_aux_loss_workspace_size(int L, int64_t T, int E) {
  if (L < 1 || T < 1 || E < 1) return 0;
  // the most blocks, whatever K
  return align_up((size_t)L * stats_blocks(T) * E * 2 * sizeof(double), 16) +
         (size_t)L * 2 * E * sizeof(double);
}

extern "C" int moe_amd_switch_aux_loss(const void* const* probs, int L, int probs_dtype,
                                       const float* token_weights, int64_t T, int E, int K,
                                       double num_experts, double denom, const double* denom_dev,
                                       void* workspace, size_t workspace_bytes, double* coef,
                                       double* loss, void* stream) {
  const char* who = "switch_aux_loss";
  int rc = check_stats_shape(T, E, K, probs_dtype, who);
  if (rc) return rc;
  MOE_REQUIRE(L >= 1 && L < 65536 && T > 0, MOE_ERR_ARG, "%s: L=%d layers of T=%lld tokens", who, L,
              (long long)T);
  MOE_REQUIRE(probs && coef && loss, MOE_ERR_ARG, "%s: null pointer", who);
  for (int l = 0; l < L; ++l) MOE_REQUIRE(probs[l], MOE_ERR_ARG, "%s: layer %d is null", who, l);
  const size_t need = moe_amd_switch_aux_loss_workspace_size(L, T, E);
  MOE_REQUIRE(workspace && workspace_bytes >= need, MOE_ERR_WORKSPACE,
              "%s: workspace of %zu bytes needed", who, need);
  MOE_REQUIRE(((uintptr_t)workspace & 15) == 0, MOE_ERR_ALIGN, "%s: workspace alignment", who);
  hipStream_t st = (hipStream_t)stream;
  const int nb = switch_blocks(L, T, E, K);
  const size_t per_layer = (size_t)nb * E;
  double* pc = (double*)workspace;
  double* ps = pc + L * per_layer;
  double* sums = (double*)((char*)workspace + align_up(L * per_layer * 2 * sizeof(double), 16));
  for (int l0 = 0; l0 < L; l0 += kMaxLayers) {
    const int nl = L - l0 < kMaxLayers ? L - l0 : kMaxLayers;
    Layers layers{};
    for (int l = 0; l < nl; ++l) layers.in[l] = probs[l0 + l];
    launch_topk_stats(layers, nl, probs_dtype, token_weights, T, E, K, nb, pc + l0 * per_layer,
                      ps + l0 * per_layer, nullptr, st);
  }
  switch_layer_sums_kernel<<<dim3(L, (E + 63) / 64), 1024, 0, st>>>(pc, ps, nb, E, sums);
  switch_loss_kernel<<<1, 1024, 0, st>>>(sums, L, E, num_experts, denom, denom_dev, coef, loss);
  return check_launch(who);
}

extern "C" int moe_amd_switch_aux_loss_backward(const double* coef, const float* d_loss,
                                                const float* token_weights, int L, int64_t T,
                                                int E, int grad_dtype, void* const* grads,
                                                void* stream) {
  const char* who = "switch_aux_loss_backward";
  MOE_REQUIRE(T >= 0 && E >= 1 && L >= 1, MOE_ERR_ARG, "%s: bad sizes", who);
  MOE_REQUIRE(grad_dtype == MOE_DTYPE_F32 || grad_dtype == MOE_DTYPE_BF16, MOE_ERR_DTYPE,
              "%s: dtype %d", who, grad_dtype);
  if (T == 0) return MOE_OK;
  MOE_REQUIRE(coef && d_loss && grads, MOE_ERR_ARG, "%s: null pointer", who);
  hipStream_t st = (hipStream_t)stream;
  for (int l0 = 0; l0 < L; l0 += kMaxLayers) {
    const int nl = L - l0 < kMaxLayers ? L - l0 : kMaxLayers;
    Layers layers{};
    bool vec = E % 4 == 0;
    for (int l = 0; l < nl; ++l) {
      MOE_REQUIRE(grads[l0 + l], MOE_ERR_ARG, "%s: layer %d is null", who, l0 + l);
      layers.out[l] = grads[l0 + l];
      vec = vec && al16(layers.out[l]);
    }
    int64_t nb = (T * (int64_t)E + 1023) / 1024;
    const int64_t most = 8192 / nl;
    if (nb > most) nb = most;
    if (vec) {
      switch_aux_bwd_vec_kernel<<<dim3((unsigned)nb, nl), 256, 0, st>>>(layers, coef, d_loss,
                                                                       token_weights, T, E,
                                                                       grad_dtype);
    } else {
      for (int l = 0; l < nl; ++l)
        switch_aux_bwd_kernel<<<(unsigned)nb, 256, 0, st>>>(coef, d_loss, token_weights, T, E,
                                                            grad_dtype, layers.out[l]);
    }
  }
  return check_launch(who);
}

extern "C" int moe_amd_update_expert_biases(float* const* counts, float* const* biases, int L,
                                            int E, float update_rate, int is_global,
                                            double alpha, double* stats, void* stream) {
  const char* who = "update_expert_biases";
  MOE_REQUIRE(L >= 1 && E >= 1 && (int64_t)L * E < ((int64_t)1 << 30), MOE_ERR_ARG,
              "%s: L=%d E=%d", who, L, E);
  MOE_REQUIRE(counts && biases && stats, MOE_ERR_ARG, "%s: null pointer", who);
  const size_t shm = (size_t)(L + 1 + E) * sizeof(float);
  MOE_REQUIRE(shm <= 56 * 1024, MOE_ERR_ARG, "%s: L + E too large", who);
  update_biases_kernel<<<1, 1024, shm, (hipStream_t)stream>>>(
      counts, biases, L, E, update_rate, is_global, (float)alpha, (float)(1.0 - alpha), stats);
  return check_launch(who);
}
