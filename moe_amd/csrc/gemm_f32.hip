// fp32 grouped GEMMs of the expert layer on gfx950, on the bf16 matrix cores
// with fp32 precision (three-term split, v_mfma_f32_32x32x16_bf16).
//
// The fp32 configurations of the reference (its CPU-runnable XS standard
// layer) run the experts in fp32: F.grouped_mm on fp32 operands with fp32
// accumulation and no intermediate rounding (transformers/integrations/
// moe.py:439-459 forward, :226-242 backward formulas).  This file is that
// path: the same six GEMMs as the bf16 kernels, unfused backward (the
// combine backward and the gather backward run as their own kernels).
//
//   mode  C [rows x cols]          rows (operand)                 cols (operand)              k
//   F1    gate_up -> act           routed rows (x gathered, kc)   [gate 64 | up 64] (W1, kc)  H
//   F2    y                        routed rows (act, kc)          H (W2[e], kc)               I
//   FDX2  d_act -> d_gate_up       routed rows (dy, kc)           I (W2[e], km)               H
//   FDX1  d_xs                     routed rows (d_gate_up, kc)    H (W1[e], km)               2I
//   FDW2  d_down_proj[e]           H (dy rows of e, km)           I (act rows of e, km)       rows of e
//   FDW1  d_gate_up_proj[e]        2I (d_gate_up rows, km)        H (x gathered, km)          rows of e
//
// (kc: the operand's k index is contiguous in memory; km: its feature index
// is, k strides by rows.)
//
// Products: the fp32 MFMA peaks at 157 TFLOP/s, the bf16 MFMA at 2500, so an
// fp32 product made of six bf16 ones has 2.6 times the room.  Every operand
// value is split into three bf16 terms x = hi + mid + lo (each the
// round-to-nearest of what is left: 8 bits plus a sign per term, so the sum
// is exact), and a product is
// summed as hi*hi + hi*mid + mid*hi + hi*lo + lo*hi + mid*mid; the three
// products left out are at most 2^-24 of |x*y| together.  hi*hi has its own
// fp32 accumulators and the five small products share others, added once at
// the end: in one accumulator all six MFMAs of 16 k would round at the sum's
// scale, where the fp32 MFMA rounds once for 2 k, and a row with few terms
// other than zero came out up to twice as far from 64 bits as there.  2-norm
// errors, fp32 MFMA / one accumulator / two: 1 nonzero term 2.5e-8 / 3.4e-8 /
// 2.6e-8, 4 terms 4.1e-8 / 7.6e-8 / 2.7e-8, 64 terms 1.4e-7 / 2.7e-7 / 5.6e-8,
// 768 terms 4.9e-7 / 4.2e-7 / 1.6e-7.  A weight gradient over at most 32 rows
// (one stage) also sums mid*lo and lo*mid, so that the one product of a single
// row is rounded as the fp32 MFMA's: 2.53e-8 both, 3.46e-8 before.
// Both operands are multiplied by 2^16 on their way, and the sums by
// 2^-32 at the end (exact in normal range): the last bit of the smallest fp32
// subnormal then lies at the smallest bf16 one, so that no term underflows
// (without it a value below 2^-110 lost its third term, then its second: 2.2e-6
// at 2^-116, 5.6e-4 at 2^-124; now 9e-8 down to 2^-128, as at 1).
// A value that is not finite, or overflows (from 2^112 on, sums from 2^96 on),
// makes every element it touches non-finite here; a workgroup that finds such
// an element in its tile computes the tile again with the fp32 MFMA
// (v_mfma_f32_32x32x2_f32), whose infinities and NaNs are the plain fp32 ones,
// and takes those elements from it.  The others keep their bits: an element
// depends on its own row and column only, whatever else is in the tile.
//
// Workgroup: 256 threads = 4 waves as 2 x 2, a 128 x 128 tile of C, each wave
// a 64 x 64 block of 2 x 2 MFMA sub-tiles (64 fp32 accumulators per lane for
// hi*hi, 64 for the small products).
// A k-stage is 32 deep: both operands are loaded global -> registers (16
// bytes per load, coalesced along the contiguous index), split in registers
// and written to LDS as three bf16 planes of [feature][32 k] (64-byte rows,
// lds_at()'s swizzle makes the fragment reads and both operands' writes
// bank-conflict free); the loads of stage s+1 are in flight while stage s is
// multiplied.  One stage buffer of 48 KB and 128 accumulators: two workgroups
// share a CU, one splits while the other multiplies.  (With one accumulator
// per element three workgroups fit: the six GEMMs below took 2436 us, with two
// 2585, with the operands' scaling 2673.)
// Per stage a wave issues 48 MFMAs (1536 cycles) and about 280 VALU
// instructions (1100 cycles, mostly the split).  Kernel times at S = 32768
// rows, H = 1024, E = 16, I = 768, with the fp32 MFMA -> with the split: F1 899 ->
// 596, F2 467 -> 298, FDX2 645 -> 361, FDX1 1195 -> 577, FDW2 792 -> 287, FDW1
// 1448 -> 556 us (173, 173, 143, 179, 180, 185 TFLOP/s).  That is 1.1 PFLOP/s of
// bf16 products, what the board's power leaves the bf16 grouped GEMMs too.
// An operand's loads go out as soon as its registers are free, no barrier
// waits for them and multiplying waves have priority (2% over the six).
// Output: register 4q+c of a lane holds (tile row L % 32, tile column 8q + 4(L/32) + c)
// of the sub-tile (the column operand is MFMA's "A").  Epilogue: 64 rows at a
// time are staged in LDS (reusing the stage buffer) and written out row by row
// with 16-byte lanes, applying the SwiGLU / dSwiGLU tail in fp32.
//
// Token-grouped tiles come from the permutation's row-tile table for 128-row
// tiles ({expert, first row, end row} per tile, device-side); dW tiles are
// (expert, row tile, column tile), their k range the expert's rows.  Each XCD
// takes a contiguous eighth of the tiles, so its L2 holds the rows and the
// weights that neighbouring tiles share.
#include <cmath>
#include <type_traits>

#include "common.h"
#include "gemm_f32.h"

namespace moe {
namespace {

constexpr int FBM = 128;          // tile rows
constexpr int FBN = 128;          // tile columns
constexpr int FBK = 32;           // k per stage
constexpr int FLD = FBK + 4;      // floats per feature row of an fp32 stage in LDS
constexpr int FSTG = FBN + 4;     // floats per row of the epilogue staging tile
constexpr int FNT = 256;          // threads per workgroup
constexpr int FTILE_TABLE = 1;    // the permutation's 128-row tile table
constexpr int kPlane = FBM * FBK * 2;          // bytes of one split plane of one operand
constexpr int kOperand = 3 * kPlane;           // ... of the three planes of one operand
constexpr size_t kLdsBytes = 2 * kOperand;
static_assert((size_t)(FBM + FBN) * FLD * 4 <= kLdsBytes, "fp32 stage fits");
static_assert((size_t)(FBM / 2) * FSTG * 4 <= kLdsBytes, "staging fits");

enum FMode { F1 = 0, F2 = 1, FDX2 = 2, FDX1 = 3, FDW2 = 4, FDW1 = 5 };

struct FArgs {
  const float* x;         // hidden_states [T,H]
  const float* w;         // gate_up_proj [E,2I,H] or down_proj [E,H,I]
  const float* a0;        // act [S,I] (F2) | dy [S,H] (FDX2, FDW2) | d_gate_up [S,2I] (FDX1, FDW1)
  const float* a1;        // gate_up [S,2I] (FDX2) | act [S,I] (FDW2)
  const int* row_src;     // [S]
  const int* offsets;     // [E+1]
  const int* tile_count;  // token modes: number of 128-row tiles
  const int4* tile_info;  // token modes: {expert, first row, end row, 0} per row tile
  float* out;
  float* out2;            // F1: gate_up [S,2I] (may be null)
  int64_t T, S;
  int E, H, I, topk;
  int n_ct, n_rt;         // column tiles; dW modes: row tiles per expert
  int n_tiles;            // dW modes: E * n_rt * n_ct
  uint32_t tok_mul;       // n / topk == (n * tok_mul) >> tok_shift for 0 <= n < 2^31
  int tok_shift;
};

__device__ __forceinline__ f32x4 ld4(const float* p) { return *(const f32x4*)p; }

// Byte offset of (feature f, 16-byte chunk c of its 32 k) in a split plane:
// 64-byte rows, four to the 256 bytes that the LDS banks span.  The chunk is
// XORed with the row's place among 16 so that 16 lanes reading one chunk of
// 16 consecutive features cover all banks; the row's low bits are XORed with
// f >> 4 so that the lanes writing features 4l + j (a k-major operand) do too.
__device__ __forceinline__ uint32_t lds_at(int f, int c) {
  return (uint32_t)((f ^ ((f >> 4) & 3)) * 64 + ((c ^ ((f >> 2) & 3)) << 4));
}

constexpr float kScale = 65536.f;  // on both operands: see the head of the file

// Two fp32 values -> the three bf16 terms of kScale times each, packed in pairs.
__device__ __forceinline__ void split_pair(float x0, float x1, uint32_t& hi, uint32_t& mid,
                                           uint32_t& lo) {
  x0 *= kScale;
  x1 *= kScale;
  hi = pack_bf2(x0, x1);
  const float r0 = x0 - bf_lo(hi), r1 = x1 - bf_hi(hi);
  mid = pack_bf2(r0, r1);
  lo = pack_bf2(r0 - bf_lo(mid), r1 - bf_hi(mid));
}

template <int MODE>
__global__ __launch_bounds__(FNT, 2) void f32_gemm_kernel(FArgs p) {
  constexpr bool TOKEN = MODE == F1 || MODE == F2 || MODE == FDX2 || MODE == FDX1;
  constexpr bool COL_KM = MODE != F1 && MODE != F2;
  constexpr bool ROW_KM = MODE == FDW2 || MODE == FDW1;
  extern __shared__ __attribute__((aligned(16))) float fsm[];
  char* const planes = (char*)fsm;  // row operand's hi, mid, lo planes, then the column operand's

  const int tid = threadIdx.x, lane = tid & 63;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wr = wid >> 1, wc = wid & 1;
  const int l32 = lane & 31, hl = lane >> 5;
  const int H = p.H, I = p.I, I2 = 2 * p.I;

  // ------------------------------------------------------------ the tile
  // XCD b % 8 (workgroups are dealt round-robin) walks a contiguous eighth.
  int e, row0 = 0, row_end = 0, ct, rt = 0, kbeg = 0, kend = 0;
  const int n_tiles = TOKEN ? *p.tile_count * p.n_ct : p.n_tiles;
  const int per_xcd = (n_tiles + 7) >> 3;
  const int tile = (int)(blockIdx.x & 7) * per_xcd + (int)(blockIdx.x >> 3);
  if ((int)(blockIdx.x >> 3) >= per_xcd || tile >= n_tiles) return;
  if constexpr (TOKEN) {
    const int rtile = tile / p.n_ct;
    ct = tile % p.n_ct;
    const int4 ti = p.tile_info[rtile];
    e = ti.x;
    row0 = ti.y;
    row_end = ti.z;
  } else {
    const int per_e = p.n_rt * p.n_ct;
    e = tile / per_e;
    const int rem = tile % per_e;
    rt = rem / p.n_ct;
    ct = rem % p.n_ct;
    kbeg = p.offsets[e];
    kend = p.offsets[e + 1];
  }
  int K_len;
  if constexpr (MODE == F1 || MODE == FDX2) K_len = H;
  else if constexpr (MODE == F2) K_len = I;
  else if constexpr (MODE == FDX1) K_len = I2;
  else K_len = kend - kbeg;
  const int nk = (K_len + FBK - 1) / FBK;

  // ------------------------------------------------------ operand loads
  // kc operand: thread t loads features t/8 + 32i (i = 0..3), k 4(t%8)..+3.
  // km operand: a thread loads four consecutive k rows (km_k + i) of four
  // features, so that the four k of a feature are written as one 8-byte
  // piece per plane; lanes l and l + 8 hold the two halves of a chunk, so
  // 16 lanes write 128 bytes of distinct banks.
  const int kc_f = tid >> 3, kc_k = (tid & 7) * 4;
  const int km_k = (wid * 2 + ((lane >> 3) & 1)) * 4;
  const int km_f = ((lane & 7) | ((lane >> 4) << 3)) * 4;

  auto div_topk = [&](int n) {  // row_src / topk by multiply-shift
    return (int)(((uint64_t)(uint32_t)n * p.tok_mul) >> p.tok_shift);
  };
  // Operands are read through buffer descriptors rebased to each stage in
  // scalar registers (64-bit base, extent capped at 4 GB), so that a lane
  // keeps 32-bit offsets only and reads past an operand return zero: the
  // ragged k range of the dW modes.  Rows past a token tile's end and weight
  // rows past H repeat the last one, and features of a km operand past its
  // width read what lies there: all of that only reaches elements of C that
  // are not stored.  Gathered token rows (F1's rows, FDW1's columns) keep
  // 64-bit addresses, since hidden_states may hold more than 4 GB.
  const int l_end = TOKEN ? min(row_end - row0, FBM) - 1 : 0;  // last row of the tile
  const char* rptr = nullptr;
  const char* cptr = nullptr;
  const char* cptr2 = nullptr;  // F1: the up rows
  uint64_t rleft = 0, cleft = 0;
  uint32_t rstep = FBK * 4, cstep = FBK * 4;
  uint32_t roff[4], coff[4];
  const float* xrow[4];
  if constexpr (MODE == F1) {
#pragma unroll
    for (int i = 0; i < 4; ++i)
      xrow[i] = p.x + (int64_t)div_topk(p.row_src[row0 + min(kc_f + 32 * i, l_end)]) * H + kc_k;
  } else if constexpr (TOKEN) {
    const int ld = MODE == F2 ? I : (MODE == FDX2 ? H : I2);
    rptr = (const char*)(p.a0 + (int64_t)row0 * ld);
    rleft = (uint64_t)(l_end + 1) * ld * 4;
#pragma unroll
    for (int i = 0; i < 4; ++i)
      roff[i] = (uint32_t)min(kc_f + 32 * i, l_end) * (uint32_t)(ld * 4) + kc_k * 4;
  } else {
    const int nf = MODE == FDW2 ? H : I2;  // features of the row operand
    rptr = (const char*)(p.a0 + (int64_t)kbeg * nf + rt * FBM);
    rleft = ((uint64_t)K_len * nf - rt * FBM) * 4;
    rstep = (uint32_t)FBK * nf * 4;
#pragma unroll
    for (int i = 0; i < 4; ++i) roff[i] = (uint32_t)(km_k + i) * (uint32_t)(nf * 4) + km_f * 4;
  }
  if constexpr (MODE == F1) {
    // tile columns: gate features ct*64 .. +63, then their up features
    cptr = (const char*)(p.w + ((int64_t)e * I2 + ct * 64) * H);
    cptr2 = cptr + (int64_t)I * H * 4;
    cleft = (uint64_t)64 * H * 4;  // I is a multiple of 64
#pragma unroll
    for (int i = 0; i < 4; ++i)
      coff[i] = (uint32_t)((kc_f + 32 * i) & 63) * (uint32_t)(H * 4) + kc_k * 4;
  } else if constexpr (MODE == F2) {
    cptr = (const char*)(p.w + ((int64_t)e * H + ct * FBN) * I);
    const int last = min(H - ct * FBN, FBN) - 1;
    cleft = (uint64_t)(last + 1) * I * 4;
#pragma unroll
    for (int i = 0; i < 4; ++i)
      coff[i] = (uint32_t)min(kc_f + 32 * i, last) * (uint32_t)(I * 4) + kc_k * 4;
  } else if constexpr (MODE == FDW1) {
    coff[0] = (uint32_t)(ct * FBN + km_f);  // hidden_states feature
  } else {
    // FDX2: down_proj[e] [H][I], k = h; FDX1: gate_up_proj[e] [2I][H], k = j;
    // FDW2: act rows of e [rows][I]
    const int nf = MODE == FDX1 ? H : I;
    cptr = (const char*)((MODE == FDW2 ? p.a1 + (int64_t)kbeg * I
                                       : p.w + (int64_t)e * (MODE == FDX1 ? I2 : H) * nf) +
                         ct * FBN);
    cleft = ((uint64_t)K_len * nf - ct * FBN) * 4;
    cstep = (uint32_t)FBK * nf * 4;
#pragma unroll
    for (int i = 0; i < 4; ++i) coff[i] = (uint32_t)(km_k + i) * (uint32_t)(nf * 4) + km_f * 4;
  }
  auto stage_rsrc = [&](const char* ptr, uint64_t bytes, uint32_t step, int s) {
    const uint64_t adv = (uint64_t)(uint32_t)s * step;
    const uint64_t left = adv < bytes ? bytes - adv : 0ull;
    return make_rsrc(ptr + adv, __builtin_amdgcn_readfirstlane(
                                    (uint32_t)(left < 0xfffff000ull ? left : 0xfffff000ull)));
  };
  auto buf4 = [](__amdgpu_buffer_rsrc_t r, uint32_t off) {
    return __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 0));
  };

  f32x4 rv[4], cv[4];
  const f32x4 zero4 = {0.f, 0.f, 0.f, 0.f};
  // FDW1: row_src of the four k rows of the next stage to be loaded, read a
  // stage ahead of the rows themselves.
  int src[4];
  auto load_src = [&](int s) {
    if constexpr (MODE == FDW1) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int k = s * FBK + km_k + i;
        src[i] = k < K_len ? p.row_src[kbeg + k] : 0;
      }
    }
  };
  auto load_rows = [&](int s) {
    if constexpr (MODE == F1) {
#pragma unroll
      for (int i = 0; i < 4; ++i) rv[i] = ld4(xrow[i] + min(s, nk - 1) * FBK);
    } else {
      const auto rr = stage_rsrc(rptr, rleft, rstep, s);
#pragma unroll
      for (int i = 0; i < 4; ++i) rv[i] = buf4(rr, roff[i]);
    }
  };
  auto load_cols = [&](int s) {
    if constexpr (MODE == FDW1) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const bool ok = (int)coff[0] < H && s * FBK + km_k + i < K_len;
        cv[i] = ok ? ld4(p.x + (int64_t)div_topk(src[i]) * H + coff[0]) : zero4;
      }
      load_src(s + 1);
    } else {
      const auto rc = stage_rsrc(cptr, cleft, cstep, s);
      const auto rc2 = MODE == F1 ? stage_rsrc(cptr2, cleft, cstep, s) : rc;
#pragma unroll
      for (int i = 0; i < 4; ++i) cv[i] = buf4(MODE == F1 && i >= 2 ? rc2 : rc, coff[i]);
    }
  };
  // Splits a loaded operand into its three planes at `base`.
  auto store_operand = [&](const f32x4 (&v)[4], char* base, auto km) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      float x[4];
      uint32_t at;
      if constexpr (decltype(km)::value) {  // k km_k..+3 of feature km_f + i
#pragma unroll
        for (int j = 0; j < 4; ++j) x[j] = v[j][i];
        at = lds_at(km_f + i, km_k >> 3) + ((km_k >> 2) & 1) * 8;
      } else {  // k kc_k..+3 of feature kc_f + 32 i
#pragma unroll
        for (int j = 0; j < 4; ++j) x[j] = v[i][j];
        at = lds_at(kc_f + 32 * i, kc_k >> 3) + ((kc_k >> 2) & 1) * 8;
      }
      u32x2 hi, mid, lo;
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        uint32_t a, b, c;
        split_pair(x[2 * h], x[2 * h + 1], a, b, c);
        hi[h] = a;
        mid[h] = b;
        lo[h] = c;
      }
      *(u32x2*)(base + at) = hi;
      *(u32x2*)(base + kPlane + at) = mid;
      *(u32x2*)(base + 2 * kPlane + at) = lo;
    }
  };

  // Workgroup barrier over LDS accesses only: __syncthreads would also wait
  // for the next stage's global loads.
  auto sync_lds = [] {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
  };
  f32x16 acc[2][2], low[2][2];  // hi*hi; the small products
  auto zero = [](f32x16 (&v)[2][2]) {
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r) v[i][j][r] = 0.f;
  };
  zero(acc);
  zero(low);

  if (nk > 0) {
    // fragment addresses of k sub-step 0 (sub-step 1: chunk ^ 2)
    uint32_t fa[2], fb[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      fa[i] = (uint32_t)kOperand + lds_at(wc * 64 + i * 32 + l32, hl);
      fb[i] = lds_at(wr * 64 + i * 32 + l32, hl);
    }
    load_src(0);
    load_rows(0);
    load_cols(0);
    // dW of an expert with few rows: eight products (see the head of the file)
    const bool few = ROW_KM && nk == 1;
    for (int s = 0; s < nk; ++s) {
      constexpr int TA[8] = {2, 1, 2, 0, 1, 1, 0, 0}, TB[8] = {1, 2, 0, 2, 1, 0, 1, 0};
      // An operand's next loads go out as soon as its registers are free, so
      // they have a barrier, the MFMAs and the other operand's split to land.
      // (Unconditionally, since a branch would make every wait a full one: what
      // lies past the last stage is not used.  A k-major operand's descriptor
      // is empty there, a k-contiguous one reads on within the tile's rows, or
      // zeros past them, and F1 reads its last rows again.)
      __builtin_amdgcn_s_setprio(0);
      store_operand(rv, planes, std::integral_constant<bool, ROW_KM>{});
      __builtin_amdgcn_sched_barrier(0);
      load_rows(s + 1);
      __builtin_amdgcn_sched_barrier(0);
      store_operand(cv, planes + kOperand, std::integral_constant<bool, COL_KM>{});
      __builtin_amdgcn_sched_barrier(0);
      load_cols(s + 1);
      __builtin_amdgcn_sched_barrier(0);
      __builtin_amdgcn_s_setprio(1);  // multiplying waves issue first (1%)
      sync_lds();
#pragma unroll
      for (int kk = 0; kk < 2; ++kk) {
        bf16x8 a[3][2], b[3][2];
#pragma unroll
        for (int t = 0; t < 3; ++t)
#pragma unroll
          for (int i = 0; i < 2; ++i) {
            a[t][i] = *(const bf16x8*)(planes + t * kPlane + (fa[i] ^ (kk * 32)));
            b[t][i] = *(const bf16x8*)(planes + t * kPlane + (fb[i] ^ (kk * 32)));
          }
        auto product = [&](int t) {  // small ones first
#pragma unroll
          for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j) {
              f32x16& c = t < 7 ? low[i][j] : acc[i][j];
              c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[TA[t]][i], b[TB[t]][j], c, 0, 0, 0);
            }
        };
        if (few) {
          product(0);
          product(1);
        }
#pragma unroll
        for (int t = 2; t < 8; ++t) product(t);
      }
      sync_lds();  // the stage is read: the next one may be written
    }
    // Non-finite elements: the tile again on the fp32 MFMA (into `low`, which is
    // free by now), from which only they are taken.
    bool bad = false;
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          acc[i][j][r] = (acc[i][j][r] + low[i][j][r]) * (1.f / kScale / kScale);
          bad |= !(fabsf(acc[i][j][r]) < INFINITY);
        }
    if (__syncthreads_or(bad)) {
      zero(low);
      float* const R = fsm;
      float* const C = fsm + FBM * FLD;
      load_src(0);
      for (int s = 0; s < nk; ++s) {
        load_rows(s);
        load_cols(s);
        __syncthreads();  // the previous stage is read
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          if constexpr (!ROW_KM) {
            *(f32x4*)(R + (kc_f + 32 * i) * FLD + kc_k) = rv[i];
          } else {
#pragma unroll
            for (int j = 0; j < 4; ++j) R[(km_f + j) * FLD + km_k + i] = rv[i][j];
          }
          if constexpr (!COL_KM) {
            *(f32x4*)(C + (kc_f + 32 * i) * FLD + kc_k) = cv[i];
          } else {
#pragma unroll
            for (int j = 0; j < 4; ++j) C[(km_f + j) * FLD + km_k + i] = cv[i][j];
          }
        }
        __syncthreads();
        // lane L supplies feature L % 32 at k 8kk + 4(L/32) + q, q = 0..3
        for (int kk = 0; kk < FBK / 8; ++kk) {
          f32x4 a[2], b[2];
#pragma unroll
          for (int i = 0; i < 2; ++i) {
            a[i] = ld4(C + (wc * 64 + i * 32 + l32) * FLD + kk * 8 + 4 * hl);
            b[i] = ld4(R + (wr * 64 + i * 32 + l32) * FLD + kk * 8 + 4 * hl);
          }
#pragma unroll
          for (int q = 0; q < 4; ++q)
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
              for (int j = 0; j < 2; ++j)
                low[i][j] =
                    __builtin_amdgcn_mfma_f32_32x32x2f32(a[i][q], b[j][q], low[i][j], 0, 0, 0);
        }
      }
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
          for (int r = 0; r < 16; ++r)
            acc[i][j][r] = fabsf(acc[i][j][r]) < INFINITY ? acc[i][j][r] : low[i][j][r];
    }
  }

  // ------------------------------------------------------------ epilogue
  // Sub-tile j of both row halves at a time: staging row wr*32 + l32 is tile
  // row wr*64 + j*32 + l32.
  float* stg = fsm;  // [FBM / 2][FSTG]
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    __syncthreads();  // the stage buffer or the previous half is read
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int col = wc * 64 + i * 32 + 8 * q + 4 * hl;
        const f32x4 v = {acc[i][j][4 * q + 0], acc[i][j][4 * q + 1], acc[i][j][4 * q + 2],
                         acc[i][j][4 * q + 3]};
        *(f32x4*)(stg + (wr * 32 + l32) * FSTG + col) = v;
      }
    __syncthreads();
    auto tile_row = [&](int sr) { return (sr >> 5) * 64 + j * 32 + (sr & 31); };
    if constexpr (MODE == F1) {
      // act = silu(gate) * up, silu(g) = g / (1 + exp(-g)) as torch evaluates it
      const int f4 = (tid & 15) * 4;
      const int feat = ct * 64 + f4;
      for (int sr = tid >> 4; sr < FBM / 2; sr += FNT / 16) {
        const int r = row0 + tile_row(sr);
        if (r >= row_end || feat >= I) continue;
        const f32x4 g = ld4(stg + sr * FSTG + f4);
        const f32x4 u = ld4(stg + sr * FSTG + 64 + f4);
        f32x4 a;
#pragma unroll
        for (int c = 0; c < 4; ++c) a[c] = g[c] / (1.0f + expf(-g[c])) * u[c];
        *(f32x4*)(p.out + (int64_t)r * I + feat) = a;
        if (p.out2) {
          *(f32x4*)(p.out2 + (int64_t)r * I2 + feat) = g;
          *(f32x4*)(p.out2 + (int64_t)r * I2 + I + feat) = u;
        }
      }
    } else if constexpr (MODE == FDX2) {
      // d_act -> d_gate = d_act * up * sigmoid(g) * (1 + g * (1 - sigmoid(g))),
      //          d_up = d_act * silu(g)   (autograd of silu(gate) * up)
      const int c4 = (tid & 31) * 4;
      const int i0 = ct * FBN + c4;
      for (int sr = tid >> 5; sr < FBM / 2; sr += FNT / 32) {
        const int r = row0 + tile_row(sr);
        if (r >= row_end || i0 >= I) continue;
        const f32x4 da = ld4(stg + sr * FSTG + c4);
        const f32x4 g = ld4(p.a1 + (int64_t)r * I2 + i0);
        const f32x4 u = ld4(p.a1 + (int64_t)r * I2 + I + i0);
        f32x4 dg, du;
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          const float sg = 1.0f / (1.0f + expf(-g[c]));
          const float sl = g[c] / (1.0f + expf(-g[c]));
          du[c] = da[c] * sl;
          dg[c] = da[c] * u[c] * (sg * (1.0f + g[c] * (1.0f - sg)));
        }
        *(f32x4*)(p.out + (int64_t)r * I2 + i0) = dg;
        *(f32x4*)(p.out + (int64_t)r * I2 + I + i0) = du;
      }
    } else {
      // Plain tile: y (F2), d_xs (FDX1), d_down_proj[e] (FDW2), d_gate_up_proj[e] (FDW1).
      const int c4 = (tid & 31) * 4;
      int nrows, ncols, rbeg;
      int64_t ld;
      float* ob;
      if constexpr (TOKEN) {
        nrows = row_end;
        rbeg = row0;
        ncols = H;
        ld = H;
        ob = p.out;
      } else {
        nrows = MODE == FDW2 ? H : I2;
        rbeg = rt * FBM;
        ncols = MODE == FDW2 ? I : H;
        ld = ncols;
        ob = p.out + (int64_t)e * nrows * ncols;
      }
      const int col = ct * FBN + c4;
      for (int sr = tid >> 5; sr < FBM / 2; sr += FNT / 32) {
        const int r = rbeg + tile_row(sr);
        if (r < nrows && col < ncols)
          *(f32x4*)(ob + (int64_t)r * ld + col) = ld4(stg + sr * FSTG + c4);
      }
    }
  }
}

// The multiply-shift of row_src / topk (Granlund and Montgomery, "Division by
// invariant integers using multiplication", 1994).
void set_topk_f32(FArgs& a, int top_k) {
  a.topk = top_k;
  int sh = 0;
  while ((1 << sh) < top_k) ++sh;
  a.tok_shift = 31 + sh;
  a.tok_mul = (uint32_t)((((uint64_t)1 << (31 + sh)) + (uint64_t)top_k - 1) / (uint64_t)top_k);
}

template <int MODE>
int launch_f32(const FArgs& a, int64_t blocks, hipStream_t st, const char* who) {
  if (blocks <= 0) return MOE_OK;
  blocks = (blocks + 7) / 8 * 8;  // the XCDs' eighths are rounded up
  MOE_REQUIRE(blocks < ((int64_t)1 << 31), MOE_ERR_UNSUPPORTED, "%s: too many tiles", who);
  static std::atomic<int> lds_done[64];
  hipError_t err = set_dynamic_lds_once(lds_done, (const void*)f32_gemm_kernel<MODE>, (int)kLdsBytes);
  if (err != hipSuccess) {
    set_error("%s: hipFuncSetAttribute failed: %s", who, hipGetErrorString(err));
    return MOE_ERR_HIP;
  }
  f32_gemm_kernel<MODE><<<(unsigned)blocks, FNT, kLdsBytes, st>>>(a);
  return check_launch(who);
}

int check_f32(int64_t S, int E, int H, int I, const char* who) {
  MOE_REQUIRE(S >= 0 && E >= 1 && H > 0 && I > 0, MOE_ERR_ARG, "%s: bad sizes", who);
  MOE_REQUIRE(H % 64 == 0 && I % 64 == 0, MOE_ERR_ARG,
              "%s: H=%d and I=%d must be multiples of 64", who, H, I);
  MOE_REQUIRE(S < ((int64_t)1 << 31), MOE_ERR_UNSUPPORTED, "%s: S out of range", who);
  return MOE_OK;
}

bool al16f(const void* p) { return ((uintptr_t)p & 15) == 0; }

#define F32_ALIGNED(ptr, who) \
  MOE_REQUIRE(al16f(ptr), MOE_ERR_ALIGN, "%s: pointer %s not 16-byte aligned", who, #ptr)

// Token-grouped launch: one workgroup per (128-row tile, column tile); the
// row-tile count is on the device, so the grid covers the most tiles the
// plan can hold and surplus workgroups return at once.
template <int MODE>
int launch_f32_token(FArgs a, const void* tile_plan, int ncols_per_tile, int ncols,
                     hipStream_t st, const char* who) {
  const char* pb = (const char*)tile_plan;
  a.tile_count = (const int*)pb + (size_t)FTILE_TABLE * (a.E + 1) + a.E;
  a.tile_info = (const int4*)(pb + plan_info_offset(a.S, a.E, FTILE_TABLE));
  a.n_ct = (ncols + ncols_per_tile - 1) / ncols_per_tile;
  return launch_f32<MODE>(a, plan_max_tiles(a.S, a.E, FTILE_TABLE) * a.n_ct, st, who);
}

}  // namespace

int f32_gate_up_swiglu(const float* x, const int32_t* row_src, int top_k, const int32_t* offsets,
                       const void* tile_plan, const float* w1, int64_t T, int64_t S, int E, int H,
                       int I, float* gate_up, float* act, hipStream_t st) {
  const char* who = "gemm_gate_up_swiglu (fp32)";
  int rc = check_f32(S, E, H, I, who);
  if (rc) return rc;
  MOE_REQUIRE(top_k >= 1 && S == T * top_k, MOE_ERR_ARG, "%s: S != T*top_k", who);
  MOE_REQUIRE(offsets && tile_plan && w1 && (S == 0 || (x && row_src && act)), MOE_ERR_ARG,
              "%s: null pointer", who);
  F32_ALIGNED(x, who);
  F32_ALIGNED(w1, who);
  F32_ALIGNED(act, who);
  F32_ALIGNED(gate_up, who);
  if (S == 0) return MOE_OK;
  FArgs a{};
  a.x = x; a.w = w1; a.row_src = row_src; a.offsets = offsets; a.out = act; a.out2 = gate_up;
  a.T = T; a.S = S; a.E = E; a.H = H; a.I = I; set_topk_f32(a, top_k);
  return launch_f32_token<F1>(a, tile_plan, 64, I, st, who);
}

int f32_down(const float* act, const int32_t* offsets, const void* tile_plan, const float* w2,
             int64_t S, int E, int H, int I, float* y, hipStream_t st) {
  const char* who = "gemm_down (fp32)";
  int rc = check_f32(S, E, H, I, who);
  if (rc) return rc;
  MOE_REQUIRE(offsets && tile_plan && w2 && (S == 0 || (act && y)), MOE_ERR_ARG,
              "%s: null pointer", who);
  F32_ALIGNED(act, who);
  F32_ALIGNED(w2, who);
  F32_ALIGNED(y, who);
  if (S == 0) return MOE_OK;
  FArgs a{};
  a.w = w2; a.a0 = act; a.offsets = offsets; a.out = y;
  a.S = S; a.E = E; a.H = H; a.I = I;
  return launch_f32_token<F2>(a, tile_plan, FBN, H, st, who);
}

int f32_down_dx_dswiglu(const float* dy, const int32_t* offsets, const void* tile_plan,
                        const float* w2, const float* gate_up, int64_t S, int E, int H, int I,
                        float* d_gate_up, hipStream_t st) {
  const char* who = "gemm_down_backward_dx_dswiglu (fp32)";
  int rc = check_f32(S, E, H, I, who);
  if (rc) return rc;
  MOE_REQUIRE(offsets && tile_plan && w2 && (S == 0 || (dy && gate_up && d_gate_up)),
              MOE_ERR_ARG, "%s: null pointer", who);
  F32_ALIGNED(dy, who);
  F32_ALIGNED(w2, who);
  F32_ALIGNED(gate_up, who);
  F32_ALIGNED(d_gate_up, who);
  if (S == 0) return MOE_OK;
  FArgs a{};
  a.w = w2; a.a0 = dy; a.a1 = gate_up; a.offsets = offsets; a.out = d_gate_up;
  a.S = S; a.E = E; a.H = H; a.I = I;
  return launch_f32_token<FDX2>(a, tile_plan, FBN, I, st, who);
}

int f32_gate_up_dx(const float* dgu, const int32_t* offsets, const void* tile_plan,
                   const float* w1, int64_t S, int E, int H, int I, float* d_xs,
                   hipStream_t st) {
  const char* who = "gemm_gate_up_backward_dx (fp32)";
  int rc = check_f32(S, E, H, I, who);
  if (rc) return rc;
  MOE_REQUIRE(offsets && tile_plan && w1 && (S == 0 || (dgu && d_xs)), MOE_ERR_ARG,
              "%s: null pointer", who);
  F32_ALIGNED(dgu, who);
  F32_ALIGNED(w1, who);
  F32_ALIGNED(d_xs, who);
  if (S == 0) return MOE_OK;
  FArgs a{};
  a.w = w1; a.a0 = dgu; a.offsets = offsets; a.out = d_xs;
  a.S = S; a.E = E; a.H = H; a.I = I;
  return launch_f32_token<FDX1>(a, tile_plan, FBN, H, st, who);
}

int f32_down_dw(const float* dy, const float* act, const int32_t* offsets, int64_t S, int E,
                int H, int I, float* d_w2, hipStream_t st) {
  const char* who = "gemm_down_backward_dw (fp32)";
  int rc = check_f32(S, E, H, I, who);
  if (rc) return rc;
  MOE_REQUIRE(offsets && d_w2 && (S == 0 || (dy && act)), MOE_ERR_ARG, "%s: null pointer", who);
  F32_ALIGNED(dy, who);
  F32_ALIGNED(act, who);
  F32_ALIGNED(d_w2, who);
  FArgs a{};
  a.a0 = dy; a.a1 = act; a.offsets = offsets; a.out = d_w2;
  a.S = S; a.E = E; a.H = H; a.I = I;
  a.n_rt = (H + FBM - 1) / FBM;
  a.n_ct = (I + FBN - 1) / FBN;
  a.n_tiles = E * a.n_rt * a.n_ct;
  // every expert's tiles are written (zeros for an expert without rows)
  return launch_f32<FDW2>(a, (int64_t)E * a.n_rt * a.n_ct, st, who);
}

int f32_gate_up_dw(const float* dgu, const float* x, const int32_t* row_src, int top_k,
                   const int32_t* offsets, int64_t T, int64_t S, int E, int H, int I,
                   float* d_w1, hipStream_t st) {
  const char* who = "gemm_gate_up_backward_dw (fp32)";
  int rc = check_f32(S, E, H, I, who);
  if (rc) return rc;
  MOE_REQUIRE(top_k >= 1 && S == T * top_k, MOE_ERR_ARG, "%s: S != T*top_k", who);
  MOE_REQUIRE(offsets && d_w1 && (S == 0 || (dgu && x && row_src)), MOE_ERR_ARG,
              "%s: null pointer", who);
  F32_ALIGNED(dgu, who);
  F32_ALIGNED(x, who);
  F32_ALIGNED(d_w1, who);
  FArgs a{};
  a.x = x; a.a0 = dgu; a.row_src = row_src; a.offsets = offsets; a.out = d_w1;
  a.T = T; a.S = S; a.E = E; a.H = H; a.I = I; set_topk_f32(a, top_k);
  a.n_rt = (2 * I + FBM - 1) / FBM;
  a.n_ct = (H + FBN - 1) / FBN;
  a.n_tiles = E * a.n_rt * a.n_ct;
  return launch_f32<FDW1>(a, (int64_t)E * a.n_rt * a.n_ct, st, who);
}

}  // namespace moe
