// Token permutation: a stable counting sort of the S = T*K routed entries by
// expert id, the GPU form of transformers' sort + histc + cumsum
// (transformers/integrations/moe.py:389-403), and the tile plan of the GEMMs.
//
// All of it is latency: a few MB move, and every launch costs about 5 us in
// the chain.  So there are two forms.
//
// Small (S <= kSmallRows, LDS for the counters and ids): one launch of three
// workgroups that share nothing.  Each counts the ids itself (16 waves, one
// contiguous run of entries each, LDS counters per wave and expert); then
// block 0 scans them into offsets and scatters within LDS, block 1 writes the
// tile tables, block 2 the dW schedule.  6 us at S = 32 and 8 us at S = 2664,
// where seven launches (a fill, histogram, two scans, tables, schedule,
// scatter) took 21 and 26; past kSmallRows the one workgroup's scatter is
// slower than the general form's many (S = 32760: 50 us against 18 us with
// scattered stores from one workgroup).
//
// General, three launches (23 us at S = 524288, E = 128, where seven took 41;
// 18 against 35 us at S = 32760):
//   hist        one wave per 256-entry chunk, LDS atomics -> per-chunk
//               counts, stored expert-major [E+1][nchunks]
//   scan        per-expert exclusive scan over chunks (one block per expert)
//   tail        by block: the dW schedule; offsets, tile prefixes and one
//               height's tile table of 64 experts; the scatter of four chunks.  Every block
//               forms the prefixes it needs from the expert totals itself (a
//               last-block-done prefix pass in the scan costs an agent-scope
//               fence per expert: 50 us at E = 1792).
//
// The scatter (both forms) takes 64 entries at a time; one ballot per bit of
// the expert id groups the lanes by expert (multi-split), the in-wave rank is
// the popcount of lower peers, and a per-wave LDS counter carries the rank
// across rounds -> stable order.
// Ids outside [0,E) land in bin E (sentinels), after every real expert.
// Every byte of the plan is written, padding included.
#include <atomic>

#include "common.h"

namespace moe {
namespace {

constexpr int kChunk = 256;        // entries per wave of hist and scatter
constexpr int kWaves = 4;          // waves per block of hist and tail

__device__ __forceinline__ int bin_of(int64_t id, int E) {
  return (id >= 0 && id < E) ? (int)id : E;
}

__global__ __launch_bounds__(64 * kWaves) void hist_kernel(const int64_t* __restrict__ ids,
                                                           int64_t S, int E, int64_t nch,
                                                           int* __restrict__ chunk_hist) {
  extern __shared__ int lds[];  // [kWaves][E+1]
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  const int64_t c = (int64_t)blockIdx.x * kWaves + wid;
  int* h = lds + wid * (E + 1);
  for (int e = lane; e <= E; e += 64) h[e] = 0;
  __builtin_amdgcn_wave_barrier();
  if (c < nch) {
    const int64_t beg = c * kChunk;
#pragma unroll
    for (int i = 0; i < kChunk / 64; ++i) {
      int64_t s = beg + i * 64 + lane;
      if (s < S) atomicAdd(&h[bin_of(ids[s], E)], 1);
    }
  }
  __builtin_amdgcn_wave_barrier();
  __syncthreads();
  if (c < nch)
    for (int e = lane; e <= E; e += 64) chunk_hist[(int64_t)e * nch + c] = h[e];
}

// Inclusive scan across one wave.
__device__ __forceinline__ int wave_incl_scan(int v, int lane) {
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    int u = __shfl_up(v, o, 64);
    if (lane >= o) v += u;
  }
  return v;
}

// Exclusive scan across the block (blockDim.x multiple of 64, <= 1024).
// Returns the exclusive prefix; *total receives the block sum.
__device__ int block_excl_scan(int v, int* tmp /* >= 16 ints */, int* total) {
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6, nw = blockDim.x >> 6;
  int inc = wave_incl_scan(v, lane);
  if (lane == 63) tmp[wid] = inc;
  __syncthreads();
  if (wid == 0) {
    int w = lane < nw ? tmp[lane] : 0;
    int wi = wave_incl_scan(w, lane);
    if (lane < nw) tmp[lane] = wi - w;
    if (lane == nw - 1) tmp[16] = wi;
  }
  __syncthreads();
  int res = inc - v + tmp[wid];
  *total = tmp[16];
  __syncthreads();
  return res;
}

// The row-tile height of the token-grouped GEMMs from the three tile counts:
// the least rows plus weight columns streamed, tiles x (BM + 256) (the larger
// height on ties), written behind the tile prefixes with the zero padding up
// to the first tile table.
__device__ __forceinline__ void write_row_tile(const int (&nt)[MOE_NUM_TILE_SIZES], int E,
                                               int* __restrict__ tile_starts) {
  int best = MOE_NUM_TILE_SIZES - 1;
  int64_t best_cost = (int64_t)nt[best] * (kTileSizes[best] + 256);
  for (int b = MOE_NUM_TILE_SIZES - 2; b >= 0; --b) {
    const int64_t c = (int64_t)nt[b] * (kTileSizes[b] + 256);
    if (c < best_cost) {
      best = b;
      best_cost = c;
    }
  }
  int* const rt = tile_starts + MOE_NUM_TILE_SIZES * (E + 1);
  *rt = best;
  for (int i = 1; (MOE_NUM_TILE_SIZES * (E + 1) + i) & 3; ++i) rt[i] = 0;
}

// One block per bin e: exclusive scan of chunk_hist[e][0..nch) in place.
__global__ __launch_bounds__(1024) void scan_kernel(int* __restrict__ chunk_hist, int64_t nch,
                                                   int* __restrict__ totals) {
  __shared__ int tmp[17];
  const int e = blockIdx.x;
  int* col = chunk_hist + (int64_t)e * nch;
  int carry = 0;
  for (int64_t base = 0; base < nch; base += blockDim.x) {
    int64_t i = base + threadIdx.x;
    int v = i < nch ? col[i] : 0;
    int tot;
    int ex = block_excl_scan(v, tmp, &tot);
    if (i < nch) col[i] = carry + ex;
    carry += tot;
  }
  if (threadIdx.x == 0) totals[e] = carry;
}

// The row tiles of expert e (rows r0..r1) for height kTileSizes[b], its
// entries t0..t1 of the table, written by threads i0, i0 + step, ...
__device__ __forceinline__ void write_tiles(int4* info, int e, int b, int t0, int t1, int r0,
                                            int r1, int i0, int step) {
  for (int t = t0 + i0; t < t1; t += step)
    info[t] = make_int4(e, r0 + (t - t0) * kTileSizes[b], r1, 0);
}

// The dW-GEMM schedule, by one block of NT threads.  Experts are sorted by
// an estimate of their dW tile cost (rows + a fixed epilogue cost, in 63
// log-spaced buckets, heaviest first, and the experts without rows in a
// 64th, last; by expert id within a bucket), then dealt to the 8 XCDs in
// serpentine order (0..7, 7..0, ...), which balances the XCDs' sums.  Each
// XCD's list therefore ends with its experts without rows; xnz[x] counts
// the others (the accumulating dW GEMMs claim only those).  Also zeroes the
// GEMMs' queue counters and the plan's last padding.  scratch: 64 + NT ints
// of LDS.
template <int NT, typename F>
__device__ void dw_schedule(F&& count_of, int E, int* __restrict__ sched, int* scratch) {
  int* const hist = scratch;
  // per-wave per-bucket counts of the current NT experts
  int(*const wcnt)[64] = (int(*)[64])(scratch + 64);
  int* const queue = sched;
  int* const xstart = sched + kSchedQueueInts;
  int* const xorder = sched + kSchedQueueInts + kSchedStartInts;
  const int tid = threadIdx.x;
  if (tid < kSchedQueueInts) queue[tid] = 0;
  if (tid < 64) hist[tid] = 0;
  // Experts per XCD under serpentine dealing depend on E only.
  if (tid < kSchedXnz) {
    const int rounds = E / 8, rem = E % 8;
    int acc = 0;
    for (int x = 0; x < 8 && x < tid; ++x) {
      const int lane = (rounds & 1) ? 7 - x : x;  // lane of XCD x in the last round
      acc += rounds + (lane < rem ? 1 : 0);
    }
    xstart[tid] = tid <= 8 ? acc : E;
  } else if (tid >= kSchedXnz + 8 && tid < kSchedStartInts) {
    xstart[tid] = 0;
  }
  if (tid < 4 && E + tid < (E + 3) / 4 * 4) xorder[E + tid] = 0;
  __syncthreads();
  auto bucket = [](int n) {
    if (n == 0) return 63;             // no rows: last
    const float c = (float)n + 192.f;  // rows, plus about three k-steps of epilogue
    const int b = (int)(8.f * __log2f(c * (1.f / 192.f)));
    return 62 - min(62, max(0, b));  // 0 = heaviest
  };
  for (int e = tid; e < E; e += NT) atomicAdd(&hist[bucket(count_of(e))], 1);
  __syncthreads();
  if (tid < 64) {  // bucket starts: an exclusive scan by the first wave
    const int n = hist[tid];
    hist[tid] = wave_incl_scan(n, tid) - n;
  }
  __syncthreads();
  // The nnz experts with rows take ranks 0..nnz-1; under the serpentine
  // dealing XCD x receives nnz/8 of them, plus one if its lane in the last,
  // partial round is below nnz % 8.
  if (tid < 8) {
    const int nnz = hist[63], rz = nnz / 8, mz = nnz % 8;
    const int lane = (rz & 1) ? 7 - tid : tid;
    xstart[kSchedXnz + tid] = rz + (lane < mz ? 1 : 0);
  }
  __syncthreads();  // hist[63] moves below
  // Rank of each expert, heaviest bucket first: its bucket's start plus the
  // number of lower-id experts in the same bucket -- a stable counting sort,
  // so every call writes the same schedule.  Experts go NT at a time (one
  // per thread); inside a wave the lanes that share a bucket are found by
  // one ballot per bucket bit, and the waves' per-bucket counts are added
  // in wave order.
  const int lane = tid & 63, wid = tid >> 6;
  const uint64_t lt_mask = lane == 0 ? 0ull : (~0ull >> (64 - lane));
  const int rounds = E / 8, rem = E % 8;
  for (int base = 0; base < E; base += NT) {
    wcnt[wid][lane] = 0;
    __builtin_amdgcn_wave_barrier();
    const int e = base + tid;
    const bool valid = e < E;
    const int b = valid ? bucket(count_of(e)) : 0;
    uint64_t peers = __ballot(valid);
    for (int bit = 0; bit < 6; ++bit) {
      const uint64_t m = __ballot((b >> bit) & 1);
      peers &= ((b >> bit) & 1) ? m : ~m;
    }
    if (valid && (peers >> lane) == 1ull) wcnt[wid][b] = __popcll(peers);  // highest peer
    __syncthreads();
    int pos = 0;
    if (valid) {
      pos = hist[b] + __popcll(peers & lt_mask);
      for (int w = 0; w < wid; ++w) pos += wcnt[w][b];
    }
    if (valid) {
      const int r = pos / 8, l = pos % 8;
      const int x = (r & 1) ? 7 - l : l;
      int start = 0;
      for (int y = 0; y < x; ++y) {
        const int ly = (rounds & 1) ? 7 - y : y;
        start += rounds + (ly < rem ? 1 : 0);
      }
      xorder[start + r] = e;
    }
    if (base + NT >= E) break;
    __syncthreads();  // every rank is formed before the bucket starts move on
    if (tid < 64) {
      int tot = 0;
      for (int w = 0; w < NT / 64; ++w) tot += wcnt[w][tid];
      hist[tid] += tot;
    }
    __syncthreads();
  }
}

// One wave places 64 entries: lane's bin `key` (any value where !valid).
// Returns the bin's counter in cnt (LDS, this wave's) plus the number of lower
// lanes of the same bin, and advances the counter past the bin's lanes.
__device__ __forceinline__ int place64(int key, bool valid, int key_bits, int lane, int* cnt) {
  const uint64_t lt_mask = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
  // Lanes sharing this lane's key (multi-split by ballots): one ballot per
  // key bit, each lane keeps the lanes that agree with it on that bit.
  uint64_t peers = __ballot(valid);
  for (int b = 0; b < key_bits; ++b) {
    const uint64_t m = __ballot((key >> b) & 1);
    peers &= ((key >> b) & 1) ? m : ~m;
  }
  int before = 0;
  if (valid) before = cnt[key];
  __builtin_amdgcn_wave_barrier();
  // Highest peer bumps the counter once for the whole group.
  if (valid && (peers >> lane) == 1ull) cnt[key] = before + __popcll(peers);
  __builtin_amdgcn_wave_barrier();
  return before + __popcll(peers & lt_mask);
}

__device__ __forceinline__ int bits_of(int v) {  // of the largest key, E (sentinel bin)
  int n = 1;
  while ((v >> n) != 0) ++n;
  return n;
}

// General form, last launch.  Block 0: the dW schedule.  Blocks 1..3 n_seg:
// for 64 experts and one tile height, the tile prefixes and the tile table
// (and, at the first height, offsets and counts); the last segment's blocks
// also the ends and the table's unused entries (zeroed).  The others: the
// scatter.
__global__ __launch_bounds__(64 * kWaves) void tail_kernel(
    const int64_t* __restrict__ ids, int64_t S, int E, int64_t nch,
    const int* __restrict__ chunk_off, const int* __restrict__ totals, int* __restrict__ counts,
    int* __restrict__ offsets, int* __restrict__ tile_starts, int4* __restrict__ info0,
    int4* __restrict__ info1, int4* __restrict__ info2, int* __restrict__ sched, int n_seg,
    int* __restrict__ row_src, int* __restrict__ slot) {
  // LDS (tail_lds(E) bytes): scatter [kWaves][E+1] running counters; the other
  // blocks their scratch.
  extern __shared__ int lds[];
  constexpr int NT = 64 * kWaves;
  const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
  if (blockIdx.x == 0) {
    dw_schedule<NT>([&](int e) { return totals[e]; }, E, sched, lds);
    return;
  }
  if ((int)blockIdx.x <= 3 * n_seg) {
    const int seg = ((int)blockIdx.x - 1) / 3, hb = ((int)blockIdx.x - 1) % 3;
    const int e0 = seg * 64, ne = min(64, E - e0);
    const bool last = seg == n_seg - 1;
    int* const row_of = lds;         // [65] first row of the block's experts
    int* const tile_of = lds + 65;   // [65] ... and first tile
    int* const sums = lds + 2 * 65;  // [kWaves][4] rows and the three heights' tiles before e0
    int* const ends = sums + 4 * kWaves;  // [4] ... past the block's experts
    int acc[4] = {0, 0, 0, 0};
    auto add = [&](int n) {
      acc[0] += n;
#pragma unroll
      for (int b = 0; b < 3; ++b) acc[1 + b] += (n + kTileSizes[b] - 1) / kTileSizes[b];
    };
    for (int e = tid; e < e0; e += NT) add(totals[e]);
    const int n = wid == 0 && lane < ne ? totals[e0 + lane] : 0;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int v = wave_incl_scan(acc[q], lane);
      if (lane == 63) sums[wid * 4 + q] = v;
    }
    __syncthreads();
    if (wid == 0) {
#pragma unroll
      for (int q = 0; q < 4; ++q) acc[q] = 0;
      add(n);
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        int before = 0;
        for (int w = 0; w < kWaves; ++w) before += sums[w * 4 + q];
        const int inc = before + wave_incl_scan(acc[q], lane), ex = inc - acc[q];
        if (q == 0) {
          row_of[lane] = ex;
          if (lane == 63) row_of[64] = inc;
          if (hb == 0 && lane < ne) {
            offsets[e0 + lane] = ex;
            counts[e0 + lane] = n;
          }
        } else if (q == 1 + hb) {
          tile_of[lane] = ex;
          if (lane == 63) tile_of[64] = inc;
          if (lane < ne) tile_starts[hb * (E + 1) + e0 + lane] = ex;
        }
        if (lane == 63) ends[q] = inc;
      }
    }
    __syncthreads();
    int4* const info = hb == 0 ? info0 : (hb == 1 ? info1 : info2);
    for (int t = tile_of[0] + tid; t < tile_of[64]; t += NT) {
      int e = 0;  // the last expert whose first tile is at or before t
#pragma unroll
      for (int step = 32; step > 0; step >>= 1)
        if (tile_of[e + step] <= t) e += step;
      info[t] = make_int4(e0 + e, row_of[e] + (t - tile_of[e]) * kTileSizes[hb], row_of[e + 1], 0);
    }
    if (!last) return;
    const int64_t m = (S + kTileSizes[hb] - 1) / kTileSizes[hb] + E;
    for (int64_t t = tile_of[64] + tid; t < m; t += NT) info[t] = make_int4(0, 0, 0, 0);
    if (tid == 0) {
      tile_starts[hb * (E + 1) + E] = tile_of[64];
      if (hb == 0) {
        offsets[E] = row_of[64];
        const int nt[MOE_NUM_TILE_SIZES] = {ends[1], ends[2], ends[3]};
        write_row_tile(nt, E, tile_starts);
      }
    }
    return;
  }
  // The wave's four rounds of ids and their chunk prefixes are loaded first:
  // the offsets' scan below runs under their latency.
  constexpr int NR = kChunk / 64;
  const int64_t c = ((int64_t)blockIdx.x - 1 - 3 * n_seg) * kWaves + wid;
  int key[NR], before[NR];
#pragma unroll
  for (int i = 0; i < NR; ++i) {
    const int64_t s = c * kChunk + i * 64 + lane;
    key[i] = s < S ? bin_of(ids[s], E) : -1;
  }
#pragma unroll
  for (int i = 0; i < NR; ++i) before[i] = key[i] >= 0 ? chunk_off[(int64_t)key[i] * nch + c] : 0;
  // Every wave's counter of a bin starts at the bin's offset.  The block
  // scan's scratch lies in the last wave's counters, filled after it.
  int* const cnt = lds + wid * (E + 1);
  int* const tmp = lds + (kWaves - 1) * (E + 1);
  int carry = 0;
  for (int base = 0; base <= E; base += NT) {
    const int e = base + tid;
    const int n = e <= E ? totals[e] : 0;
    int tot;
    const int ex = carry + block_excl_scan(n, tmp, &tot);
    if (e <= E)
      for (int w = 0; w + 1 < kWaves; ++w) lds[w * (E + 1) + e] = ex;
    carry += tot;
  }
  __syncthreads();
  for (int e = tid; e <= E; e += NT) tmp[e] = lds[e];
  __syncthreads();
  const int key_bits = bits_of(E);
#pragma unroll
  for (int i = 0; i < NR; ++i) {
    const int64_t s = c * kChunk + i * 64 + lane;
    const bool valid = key[i] >= 0;
    const int dest = before[i] + place64(key[i], valid, key_bits, lane, cnt);
    if (valid) {
      row_src[dest] = (int)s;
      slot[s] = dest;
    }
  }
}

// The small form: 3 blocks of 1024 threads, see the head of the file.  LDS:
// counters [waves][E+1] ((w, e) at w * (E + 1) + e), totals / offsets [E+1],
// the sorted rows [S] and the entries' bins [S] (16 bits: E < 65536).
constexpr int kSmallWaves = 16;
__global__ __launch_bounds__(1024) void small_kernel(
    const int64_t* __restrict__ ids, int S, int E, int* __restrict__ counts,
    int* __restrict__ offsets, int* __restrict__ row_src, int* __restrict__ slot,
    int* __restrict__ tile_starts, int4* __restrict__ info0, int4* __restrict__ info1,
    int4* __restrict__ info2, int* __restrict__ sched) {
  extern __shared__ int lds[];
  __shared__ int tmp[17];
  __shared__ int sched_scratch[64 + 1024];
  const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6, n = E + 1;
  const int rows = blockIdx.x == 0 ? kSmallWaves : 1;
  for (int i = tid; i < rows * n; i += 1024) lds[i] = 0;
  __syncthreads();
  int* const tot = lds + kSmallWaves * n;
  int* const sorted = tot + n;
  uint16_t* const bins = (uint16_t*)(sorted + S);
  // each wave's contiguous run of entries, a multiple of 64
  const int per = (S + kSmallWaves * 64 - 1) / (kSmallWaves * 64) * 64;
  const int beg = min(wid * per, S), end = min(beg + per, S);
  int* const mine = blockIdx.x == 0 ? lds + wid * n : lds;
#pragma unroll 4
  for (int s = beg + lane; s < end; s += 64) {
    const int key = bin_of(ids[s], E);
    atomicAdd(&mine[key], 1);
    if (blockIdx.x == 0) bins[s] = (uint16_t)key;
  }
  __syncthreads();
  if (blockIdx.x == 2) {
    dw_schedule<1024>([&](int e) { return lds[e]; }, E, sched, sched_scratch);
    return;
  }
  if (blockIdx.x == 1) {
    int carry[1 + MOE_NUM_TILE_SIZES] = {0, 0, 0, 0};
    for (int base = 0; base <= E; base += 1024) {
      const int e = base + tid;
      const int c = e < E ? lds[e] : 0;
      int t;
      const int r0 = carry[0] + block_excl_scan(c, tmp, &t);
      carry[0] += t;
#pragma unroll
      for (int b = 0; b < MOE_NUM_TILE_SIZES; ++b) {
        const int nt = (c + kTileSizes[b] - 1) / kTileSizes[b];
        const int t0 = carry[1 + b] + block_excl_scan(nt, tmp, &t);
        carry[1 + b] += t;
        if (e <= E) tile_starts[b * n + e] = t0;
        write_tiles(b == 0 ? info0 : (b == 1 ? info1 : info2), e, b, t0, t0 + nt, r0, r0 + c, 0, 1);
      }
    }
    if (tid == 0) {
      const int nt[MOE_NUM_TILE_SIZES] = {carry[1], carry[2], carry[3]};
      write_row_tile(nt, E, tile_starts);
    }
#pragma unroll
    for (int b = 0; b < MOE_NUM_TILE_SIZES; ++b) {
      int4* const info = b == 0 ? info0 : (b == 1 ? info1 : info2);
      const int m = (S + kTileSizes[b] - 1) / kTileSizes[b] + E;
      for (int t = carry[1 + b] + tid; t < m; t += 1024) info[t] = make_int4(0, 0, 0, 0);
    }
    return;
  }
  // block 0: each bin's exclusive scan over the waves
  for (int e = tid; e < n; e += 1024) {
    int acc = 0;
#pragma unroll
    for (int w = 0; w < kSmallWaves; ++w) {
      const int c = lds[w * n + e];
      lds[w * n + e] = acc;
      acc += c;
    }
    tot[e] = acc;
  }
  __syncthreads();
  int carry = 0;
  for (int base = 0; base < n; base += 1024) {
    const int e = base + tid;
    const int c = e < n ? tot[e] : 0;
    int t;
    const int ex = carry + block_excl_scan(c, tmp, &t);
    carry += t;
    if (e < n) {
      offsets[e] = ex;
      tot[e] = ex;
      if (e < E) counts[e] = c;
    }
  }
  __syncthreads();
  const int key_bits = bits_of(E);
  for (int at = beg; at < end; at += 64) {
    const int s = at + lane;
    const bool valid = s < end;
    const int key = valid ? bins[s] : -1;
    const int pos = place64(key, valid, key_bits, lane, mine);
    if (valid) {
      const int dest = tot[key] + pos;
      sorted[dest] = s;
      slot[s] = dest;
    }
  }
  __syncthreads();
  for (int s = tid; s < S; s += 1024) row_src[s] = sorted[s];
}

// LDS that tail_kernel needs whatever E: the schedule's scratch, the segment
// blocks' and the block scan's 17 ints behind 3 (E + 1).
constexpr size_t kTailScratch = 512 * sizeof(int);

// Rows up to which the small form is taken, and the LDS it needs.
constexpr int kSmallRows = 8192;
constexpr int kSmallLds = 152 * 1024;
size_t small_lds(int64_t S, int E) {
  return (size_t)(kSmallWaves + 1) * (E + 1) * sizeof(int) + (size_t)S * 6;
}

size_t permute_ws_bytes(int64_t S, int E) {
  int64_t nch = (S + kChunk - 1) / kChunk;
  return align_up(((size_t)(E + 1) * (size_t)nch + (size_t)(E + 1)) * sizeof(int), 256);
}

}  // namespace
}  // namespace moe

using namespace moe;

extern "C" size_t moe_amd_permute_workspace_size(int64_t S, int E) {
  if (S < 0 || E < 1) return 0;
  return permute_ws_bytes(S, E);
}

extern "C" size_t moe_amd_tile_plan_size(int64_t S, int E) {
  if (S < 0 || E < 1) return 0;
  return plan_bytes(S, E);
}

namespace moe {
namespace {

// The permutation proper: validation, then the kernels on `stream`, with
// `workspace` as the general form's histogram / scan scratch.
int permute_run(const int64_t* topk_index, int64_t S, int E, void* workspace,
                size_t workspace_bytes, int32_t* counts, int32_t* offsets, int32_t* row_src,
                int32_t* slot, void* tile_plan, size_t tile_plan_bytes, void* stream,
                const char* who) {
  MOE_REQUIRE(S >= 0 && S < (int64_t)1 << 31, MOE_ERR_ARG, "%s: S=%lld out of range", who,
              (long long)S);
  MOE_REQUIRE(E >= 1 && E <= 16384, MOE_ERR_ARG, "%s: E=%d out of range", who, E);
  MOE_REQUIRE(counts && offsets && tile_plan, MOE_ERR_ARG, "%s: null output", who);
  MOE_REQUIRE(tile_plan_bytes >= plan_bytes(S, E) && ((uintptr_t)tile_plan & 15) == 0,
              MOE_ERR_WORKSPACE, "%s: tile plan needs %zu bytes, 16-byte aligned", who,
              plan_bytes(S, E));
  MOE_REQUIRE(S == 0 || (topk_index && row_src && slot), MOE_ERR_ARG, "%s: null pointer", who);
  const size_t need = permute_ws_bytes(S, E);
  MOE_REQUIRE(workspace && workspace_bytes >= need, MOE_ERR_WORKSPACE,
              "%s: workspace %zu bytes < %zu needed", who, workspace_bytes, need);
  const size_t lds = (size_t)kWaves * (E + 1) * sizeof(int);
  MOE_REQUIRE(lds <= 160 * 1024, MOE_ERR_ARG, "%s: E=%d needs too much LDS", who, E);
  const size_t tail_lds = lds > kTailScratch ? lds : kTailScratch;
  hipStream_t st = (hipStream_t)stream;
  int* tile_starts = (int*)tile_plan;
  char* pb = (char*)tile_plan;
  int4* const info0 = (int4*)(pb + plan_info_offset(S, E, 0));
  int4* const info1 = (int4*)(pb + plan_info_offset(S, E, 1));
  int4* const info2 = (int4*)(pb + plan_info_offset(S, E, 2));
  int* sched = (int*)(pb + plan_sched_offset(S, E));
  if (S <= kSmallRows && small_lds(S, E) <= kSmallLds) {
    static std::atomic<int> lds_done[64];
    hipError_t err = set_dynamic_lds_once(lds_done, (const void*)small_kernel, kSmallLds);
    MOE_REQUIRE(err == hipSuccess, MOE_ERR_HIP, "%s: hipFuncSetAttribute failed: %s", who,
                hipGetErrorString(err));
    small_kernel<<<3, 1024, small_lds(S, E), st>>>(topk_index, (int)S, E, counts, offsets, row_src,
                                                   slot, tile_starts, info0, info1, info2, sched);
    return check_launch(who);
  }
  const int64_t nch = (S + kChunk - 1) / kChunk;
  int* chunk_hist = (int*)workspace;
  int* totals = chunk_hist + (size_t)(E + 1) * nch;
  const int blocks = (int)((nch + kWaves - 1) / kWaves);
  if (nch > 0)
    hist_kernel<<<blocks, 64 * kWaves, lds, st>>>(topk_index, S, E, nch, chunk_hist);
  scan_kernel<<<E + 1, 1024, 0, st>>>(chunk_hist, nch, totals);
  const int n_seg = (E + 63) / 64;
  tail_kernel<<<1 + 3 * n_seg + blocks, 64 * kWaves, tail_lds, st>>>(
      topk_index, S, E, nch, chunk_hist, totals, counts, offsets, tile_starts, info0, info1, info2,
      sched, n_seg, row_src, slot);
  return check_launch(who);
}

}  // namespace
}  // namespace moe

extern "C" int moe_amd_permute(const int64_t* topk_index, int64_t S, int E, void* workspace,
                               size_t workspace_bytes, int32_t* counts, int32_t* offsets,
                               int32_t* row_src, int32_t* slot, void* tile_plan,
                               size_t tile_plan_bytes, void* stream) {
  return permute_run(topk_index, S, E, workspace, workspace_bytes, counts, offsets, row_src,
                     slot, tile_plan, tile_plan_bytes, stream, "permute");
}

// ---------------------------------------------------------------------------
// Allocation-free variant.  Its scratch is this file-scope device array (one
// copy per GPU, in the code object's global segment, held until the process
// ends).  In host code `scratch` names a host-side stand-in, not a device
// address: the device address of each GPU's copy comes from
// hipGetSymbolAddress, taken once per device (with that device current) on
// the entry point's first call there, and only that address is passed to the
// kernels.  The permutation's scratch is fully rewritten by every call (the
// per-chunk histograms by hist_kernel, the totals by scan_kernel), so
// nothing in it has to start at zero; calls that overlap on one GPU share the
// array and race.
static __device__ __align__(256) char scratch[MOE_PERMUTE_NOALLOC_SCRATCH_BYTES];

namespace {

std::atomic<void*> g_scratch_dev[64];  // device address of `scratch`, per device

int scratch_address(void** out, const char* who) {
  int dev = 0;
  hipError_t err = hipGetDevice(&dev);
  MOE_REQUIRE(err == hipSuccess, MOE_ERR_HIP, "%s: hipGetDevice failed: %s", who,
              hipGetErrorString(err));
  MOE_REQUIRE(dev >= 0 && dev < 64, MOE_ERR_UNSUPPORTED, "%s: device %d out of range", who, dev);
  void* p = g_scratch_dev[dev].load(std::memory_order_acquire);
  if (!p) {
    err = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    MOE_REQUIRE(err == hipSuccess && p, MOE_ERR_HIP, "%s: hipGetSymbolAddress failed: %s", who,
                hipGetErrorString(err));
    g_scratch_dev[dev].store(p, std::memory_order_release);
  }
  *out = p;
  return MOE_OK;
}

}  // namespace

extern "C" int moe_amd_permute_noalloc(const int64_t* topk_index, int64_t S, int E,
                                       int32_t* counts, int32_t* offsets, int32_t* row_src,
                                       int32_t* slot, void* tile_plan, size_t tile_plan_bytes,
                                       void* stream) {
  const char* who = "permute_noalloc";
  MOE_REQUIRE(S >= 0 && S < (int64_t)1 << 31 && E >= 1 && E <= 16384, MOE_ERR_ARG,
              "%s: S=%lld or E=%d out of range", who, (long long)S, E);
  const size_t need = permute_ws_bytes(S, E);
  MOE_REQUIRE(need <= (size_t)MOE_PERMUTE_NOALLOC_SCRATCH_BYTES, MOE_ERR_UNSUPPORTED,
              "%s: S=%lld, E=%d need %zu bytes of scratch, more than the %d-byte static array "
              "(use moe_amd_permute with a workspace)", who, (long long)S, E, need,
              MOE_PERMUTE_NOALLOC_SCRATCH_BYTES);
  void* ws = nullptr;
  int rc = scratch_address(&ws, who);
  if (rc) return rc;
  return permute_run(topk_index, S, E, ws, MOE_PERMUTE_NOALLOC_SCRATCH_BYTES, counts, offsets,
                     row_src, slot, tile_plan, tile_plan_bytes, stream, who);
}
