// int2 QAT LM head: the reference's logits producer
// (src/webgpu/decode-lm-head.ts:262-340, weights src/model/gemma-output-
// weights.ts:72-81), restated from its CPU definition cpuQatLinear
// (src/reference/qat-linear.ts:78-148):
//   logits[m][r] = srq(scale[r] * sum_k (code[r][k] - 2) * srq(x[m][k], in_scale), out_scale)
// with srq(v, s) = v for s = 0, else clamp(rint(v / s), -128, 127) * s
// rounded to float. Each lane owns one vocabulary row and sums its products
// in column order in binary64: a product of a small integer and a float is
// exact there, so the fused multiply-add rounds exactly where the reference's
// sequential binary64 sum does, and the logits equal cpuQatLinear's bit for
// bit. (The reference's WGSL kernel sums in binary32 in a subgroup order;
// its test allows 5e-4.)
//
// Weights: 2-bit codes, code k of a row at bits 2k..2k+1 of word k / 16
// (packInt2Rows). Row-major: word w of row r at r * (D / 16) + w, the
// checkpoint's order. Block-major: the 4-word block b of row r at
// (b * V + r) * 4, the reference's GPU order, where a wave's 64 lanes read
// 1 KiB in one coalesced load per block.
//
// HBM: V * D / 4 bytes of codes (96 MiB at V 262144, D 1536) + 4 V of scales
// + 4 M V of logits per call; the activations (M x D) are staged in LDS as
// binary64. Work: one bit-field extract, one conversion and one fused
// multiply-add per weight and row of x. qat_lmhead_kernel does so for widths
// past 2048 and for little work (launch_qat_lmhead).
//
// Exact integer path (widths up to 2048). Every activation a_k is a binary32 value, an integer multiple of its
// granule 2^g_k; with E the smallest granule of a row (nonzero a_k), every
// product (code - 2) a_k and every partial sum is an integer multiple of 2^E
// no larger than 2 sum |a_k|. When that bound is below 2^(E + 53), no partial
// sum rounds: the sequential binary64 sum is the exact sum, and so is
//   2^E (sum_k code_k A_k - 2 sum_k A_k),   A_k = a_k / 2^E (integers).
// qat_tile_kernel (one or two rows, widths a multiple of 256, V a multiple of
// 16) and qat_gemm_kernel (groups of 16 rows, any width and V) check the
// bound per row of x, write A_k as up to 7 balanced
// base-256 digits (int8 limbs), multiply the codes (0..3, int8) by the
// limbs on v_mfma_i32_16x16x64_i8 (exact int32 sums), combine the limbs in
// wrapping 64-bit arithmetic (exact: the total fits in 53 bits) and apply
// the same epilogue, so the logits equal the binary64 path's bit for bit.
// Rows that fail the bound (a huge exponent range, subnormals, non-finite
// values) take the binary64 path in the same launch.
#include "gs_internal.h"

namespace gs {
namespace {

constexpr int kQatThreads = 256;
constexpr int kQatLdsDoubles = 4096;  // activations staged: one row of width 4096 or two of 2048
constexpr int64_t kQatSmall = 60000000;  // products of one or two rows

struct QatArgs {
  const float* x;         // [M][D]
  const uint32_t* words;  // packed codes
  const float* scales;    // [V]
  float* out;             // [M][V]
  int32_t D, V, M;
  int32_t block_major;
  double in_scale, out_scale;
};

__device__ __forceinline__ double srq(double v, double s) {
  if (s == 0) return v;
  // the reference's floor-based rounding (qat-linear.ts:142-148) returns +0
  // for ratios in [-1/2, 0), where rint gives -0, and keeps a ratio of -0
  // (floor(-0) is -0): a zero from rint becomes the ratio itself when that
  // is a zero, else +0
  const double r = v / s;
  double q = __builtin_rint(r);
  if (q == 0.0) q = r == 0.0 ? r : 0.0;
  q = q < -128.0 ? -128.0 : (q > 127.0 ? 127.0 : q);
  return (double)(float)(q * s);
}

// srq with r = 1 / s rounded to nearest (0 where s lies outside 2^+-100: the
// division): v / s in three operations, exactly rounded (Markstein; |v| is 0
// or within 2^-300 .. 2^320 here, so nothing under- or overflows).
__device__ __forceinline__ double srq_reciprocal(double s) { return s >= 0x1p-100 && s <= 0x1p100 ? 1.0 / s : 0.0; }
__device__ __forceinline__ double srq(double v, double s, double r) {
  if (r == 0) return srq(v, s);
  const double q0 = v * r;
  double ratio = __builtin_fma(__builtin_fma(-q0, s, v), r, q0);
  ratio = v == 0 || v - v != 0 ? v : ratio;  // a zero keeps its sign; infinities and NaN
  double q = __builtin_rint(ratio);
  if (q == 0.0) q = ratio == 0.0 ? ratio : 0.0;
  q = q < -128.0 ? -128.0 : (q > 127.0 ? 127.0 : q);
  return (double)(float)(q * s);
}

// The activations of kRows rows of x from m0 (those below M) into act,
// after the input SRQ, in binary64 (the whole block calls it).
template <int kRows, int kThreads = kQatThreads>
__device__ __forceinline__ void qat_stage_act(const QatArgs& a, int32_t m0, double* act) {
  const int D = a.D;
  const int rows = a.M - m0 < kRows ? a.M - m0 : kRows;
  for (int i = threadIdx.x; i < kRows * D; i += kThreads) {
    const int m = i / D;
    act[i] = m < rows ? srq((double)a.x[(int64_t)(m0 + m) * D + (i - m * D)], a.in_scale) : 0.0;
  }
  __syncthreads();
}

// Logits of the staged rows (those below M and not skipped) at vocabulary
// row r < V.
template <int kRows>
__device__ __forceinline__ void qat_row_binary64(const QatArgs& a, int32_t m0, const bool (&skip)[kRows],
                                                 const double* act, int64_t r) {
  const int D = a.D;
  const int rows = a.M - m0 < kRows ? a.M - m0 : kRows;
  double acc[kRows];
#pragma unroll
  for (int m = 0; m < kRows; ++m) acc[m] = 0.0;
  const int blocks = D / 64;
  const uint4* w4 = (const uint4*)a.words;
  for (int b = 0; b < blocks; ++b) {
    const uint4 w = load_nt16(a.block_major ? w4 + (int64_t)b * a.V + r : w4 + r * blocks + b);
    const uint32_t q[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      // code ^ 2 read as a signed 2-bit field is code - 2
      const uint32_t flipped = q[j] ^ 0xAAAAAAAAu;
#pragma unroll
      for (int f = 0; f < 16; ++f) {
        const double wt = (double)(int)__builtin_amdgcn_sbfe((int)flipped, 2 * f, 2);
        const int k = b * 64 + j * 16 + f;
#pragma unroll
        for (int m = 0; m < kRows; ++m) acc[m] = __builtin_fma(wt, act[m * D + k], acc[m]);
      }
    }
  }
  const double scale = (double)a.scales[r];
#pragma unroll
  for (int m = 0; m < kRows; ++m) {
    if (m < rows && !skip[m]) a.out[(int64_t)(m0 + m) * a.V + r] = (float)srq(acc[m] * scale, a.out_scale);
  }
}

// kRows rows of x per pass (m0 .. m0 + kRows - 1, those below M)
template <int kRows>
__global__ __launch_bounds__(kQatThreads) void qat_lmhead_kernel(QatArgs a, int32_t m0) {
  __shared__ double act[kQatLdsDoubles];
  bool skip[kRows];
#pragma unroll
  for (int m = 0; m < kRows; ++m) skip[m] = false;
  qat_stage_act<kRows>(a, m0, act);
  const int64_t r = (int64_t)blockIdx.x * kQatThreads + threadIdx.x;
  if (r < a.V) qat_row_binary64<kRows>(a, m0, skip, act, r);
}

// ---- the exact integer path
typedef int i32x4 __attribute__((ext_vector_type(4)));
constexpr int kQatLimbs = 7;                   // balanced base-256 digits of |A_k| < 2^52
constexpr uint64_t kQatSumBound = 1ull << 52;  // sum |A_k| below it: every partial sum exact

// Operand layout of the integer path: MFMA step s takes 64 codes of a row,
// lane row + 16 g of a 16-row tile holding 16 of them as 4 dwords, byte i of
// dword t being code 16 W + 4 i + t of word W = 16 q + 4 g + t' (s = 4 q + t').
// The tile kernel expands a code word into bytes in that order and writes
// the activations' limbs at the same positions; the dot product does not
// depend on the order of k.
// The activation's integer significand and granule exponent (the value is
// sig 2^g); false for a non-finite value.
__device__ __forceinline__ bool act_parts(float f, uint32_t* sig, int* g) {
  const uint32_t bits = __builtin_bit_cast(uint32_t, f);
  const uint32_t ex = (bits >> 23) & 0xFFu;
  if (ex == 0xFFu) return false;
  *sig = ex ? (bits & 0x7FFFFFu) | 0x800000u : bits & 0x7FFFFFu;
  *g = ex ? (int)ex - 150 : -149;
  return true;
}

// Per-row constants of a tile's two rows of x, reduced in LDS.
struct QatTileRows {
  int emin[2];                  // smallest granule exponent of the nonzero activations
  uint32_t bad[2];              // a non-finite activation, or a magnitude past the bound
  unsigned long long sabs[2];   // sum |A_k|
  unsigned long long ssum[2];   // sum A_k (wrapping; exact when the check passes)
};

constexpr int kQatMaxSteps = 2048 / 64;
constexpr int kQatTileThreads = 1024;
constexpr int kQatTileWaves = kQatTileThreads / 64;
constexpr int32_t kQatNT = 2;        // non-temporal cache policy of the code stream
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

// One or two rows of x, one workgroup per compute unit over a contiguous run
// of 16-row vocabulary tiles. Each workgroup checks the rows and writes their
// limbs into LDS as a 16-row operand tile (rows 8 r + limb, limb 7 zero; one
// thread per code word of 16 activations); its 16 waves then take the run's
// tiles in turn, the next tile's codes loading while the current one
// multiplies. A row the check refused takes the binary64 path over the same
// vocabulary rows afterwards. (Four 256-thread workgroups per compute unit,
// each repeating the check and the limbs, took 25.3 us instead of 24.4 at
// V 262144, D 1536; reducing the check's sums through an LDS array by one wave
// per row instead of LDS atomics, 24.9 us instead of 24.0.)
__global__ __launch_bounds__(kQatTileThreads) void qat_tile_kernel(QatArgs a) {
  __shared__ union __attribute__((aligned(16))) {
    i32x4 op[kQatMaxSteps][64];   // the integer path's operand tile
    double act[2 * 2048];         // the binary64 path's activations
  } L;
  __shared__ QatTileRows R;
  const int tid = threadIdx.x;
  const int D = a.D, words = D / 16, quads = D / 256;
  const int lane = tid & 63, wave = tid >> 6, j = lane & 15, g = lane >> 4;
  const int n_tiles = a.V / 16;
  const int t_lo = (int)((int64_t)blockIdx.x * n_tiles / gridDim.x);
  const int t_hi = (int)((int64_t)(blockIdx.x + 1) * n_tiles / gridDim.x);
  // Every global access below is a buffer access with no branch around it:
  // codes of tiles past the run or of quads past the width, activations past
  // the rows and logits a lane does not own take an out-of-range offset (zeros, no memory request; stores
  // dropped). Loads and stores share one in-order wait counter, and a branch
  // around either made the compiler wait for every access in flight.
  const __amdgpu_buffer_rsrc_t cr =
      __builtin_amdgcn_make_buffer_rsrc((void*)a.words, (short)0, a.V * words * 4, kBufferWord3);
  const __amdgpu_buffer_rsrc_t sr = __builtin_amdgcn_make_buffer_rsrc((void*)a.scales, (short)0, a.V * 4, kBufferWord3);
  const __amdgpu_buffer_rsrc_t xr = __builtin_amdgcn_make_buffer_rsrc((void*)a.x, (short)0, a.M * D * 4, kBufferWord3);
  const __amdgpu_buffer_rsrc_t orr =
      __builtin_amdgcn_make_buffer_rsrc((void*)a.out, (short)0, a.M * a.V * 4, kBufferWord3);
  // words 16 q + 4 g .. + 3 of vocabulary row n (block 4 q + g in block-major
  // order) and the row's scale
  auto load = [&](int vt, u32x4 (&cw)[kQatMaxSteps / 4], float& sc) __attribute__((always_inline)) {
    const bool live = vt < t_hi;
    const uint32_t n = (uint32_t)vt * 16u + (uint32_t)j;
#pragma unroll
    for (int q = 0; q < kQatMaxSteps / 4; ++q) {
      const uint32_t off = a.block_major ? ((uint32_t)(4 * q + g) * (uint32_t)a.V + n) * 16u
                                         : (n * (uint32_t)words + (uint32_t)(16 * q + 4 * g)) * 4u;
      cw[q] = __builtin_amdgcn_raw_buffer_load_b128(cr, live && q < quads ? off : kBufferOutOfRange, 0, kQatNT);
    }
    sc = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(sr, live ? n * 4u : kBufferOutOfRange, 0, 0));
  };

  // the check: this thread's word W of row rr (activations 16 W .. 16 W + 15)
  const int rr = tid / words, W = tid - rr * words;
  const bool mine = tid < 2 * words;
  u32x4 xv[4];
#pragma unroll
  for (int v = 0; v < 4; ++v)
    xv[v] = __builtin_amdgcn_raw_buffer_load_b128(xr, mine ? (uint32_t)((rr * D + 16 * W) * 4 + 16 * v) : kBufferOutOfRange,
                                                  0, 0);
  if (tid < 2) { R.emin[tid] = 0x7FFFFFFF; R.bad[tid] = 0; R.sabs[tid] = 0; R.ssum[tid] = 0; }
  __syncthreads();
  // activations of rows past M, and of threads past the words, read zeros
  float f[16];
#pragma unroll
  for (int v = 0; v < 4; ++v) {
    // the elements as scalars first: a bit cast of a vector element
    // subscript reads element 0 here
    const uint32_t xs[4] = {xv[v].x, xv[v].y, xv[v].z, xv[v].w};
#pragma unroll
    for (int e = 0; e < 4; ++e) f[4 * v + e] = (float)srq((double)__builtin_bit_cast(float, xs[e]), a.in_scale);
  }
  // An integer workgroup's first codes load while the rest of the check runs.
  // They go out once the activations are in: issued at the start, the whole
  // grid's first tiles (24 MB at D 1536) queued ahead of the activations' own
  // misses and tripled their latency.
  __builtin_amdgcn_sched_barrier(0);
  u32x4 b0[kQatMaxSteps / 4], b1[kQatMaxSteps / 4];
  float s0, s1;
  int vt = t_lo + wave;
  load(vt, b0, s0);
  __builtin_amdgcn_sched_barrier(0);
  int gmin = 0x7FFFFFFF;
  bool bad = false;
#pragma unroll
  for (int e = 0; e < 16; ++e) {
    uint32_t sig;
    int g;
    if (!act_parts(f[e], &sig, &g)) bad = true;
    else if (sig) gmin = g < gmin ? g : gmin;
  }
  if (mine && gmin != 0x7FFFFFFF) atomicMin(&R.emin[rr], gmin);
  __syncthreads();
  const int E = mine && R.emin[rr] != 0x7FFFFFFF ? R.emin[rr] : 0;
  int64_t A[16];
  uint64_t sabs = 0, ssum = 0;
#pragma unroll
  for (int e = 0; e < 16; ++e) {
    A[e] = 0;
    uint32_t sig = 0;
    int g = 0;
    if (!act_parts(f[e], &sig, &g) || !sig) continue;
    const int sh = g - E;
    if (sh > 62 - 24) { bad = true; continue; }
    const uint64_t mag = (uint64_t)sig << sh;
    if (mag >= kQatSumBound) { bad = true; continue; }
    A[e] = f[e] < 0.0f ? -(int64_t)mag : (int64_t)mag;
    sabs += mag;
    ssum += (uint64_t)A[e];
  }
  if (mine) {
    // (magnitudes below 2^52, at most 2048 of them: the sums do not wrap
    // unless the check fails anyway)
    atomicAdd(&R.sabs[rr], (unsigned long long)sabs);
    atomicAdd(&R.ssum[rr], (unsigned long long)ssum);
    if (bad) atomicOr(&R.bad[rr], 1u);
  }
  __syncthreads();
  bool ok[2];
#pragma unroll
  for (int q = 0; q < 2; ++q) ok[q] = q < a.M && !R.bad[q] && R.sabs[q] < kQatSumBound;

  const bool any_ok = ok[0] || ok[1];
  // the limbs: tile row 8 rr + l, balanced base-256 digits of A (zeros for a
  // row the check refused), at the operand positions of word W. With
  // K = sum_l 128 256^l (l < 7) and |A| < 2^52, u = A + K has the base-256
  // digits c_l = d_l + 128 in [0, 255]; the int8 digit d_l = c_l - 128 is
  // byte l of u ^ K (byte 7 is zero).
  if (mine && any_ok) {
    const int q = W >> 4, gw = (W >> 2) & 3, tp = W & 3;
    const int step = 4 * q + tp;
    constexpr uint64_t kK = 0x0080808080808080ull;
    static_assert(kQatLimbs == 7, "K holds one 0x80 byte per limb");
    uint32_t* op_words = (uint32_t*)&L.op[step][0];
    // dword t of a limb's operand holds activations 4 i + t (byte i)
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      uint32_t lo[4], hi[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const uint64_t u = ((uint64_t)(ok[rr] ? A[4 * i + t] : 0) + kK) ^ kK;
        lo[i] = (uint32_t)u;
        hi[i] = (uint32_t)(u >> 32);
      }
#pragma unroll
      for (int l = 0; l < 8; ++l) {
        uint32_t dw = 0u;
#pragma unroll
        for (int i = 0; i < 4; ++i) dw |= (((l < 4 ? lo[i] : hi[i]) >> (8 * (l & 3))) & 0xFFu) << (8 * i);
        op_words[(8 * rr + l + 16 * gw) * 4 + t] = dw;
      }
    }
  }
  __syncthreads();

  auto multiply = [&](int vt, const u32x4 (&cw)[kQatMaxSteps / 4], float sc) __attribute__((always_inline)) {
    i32x4 acc = {0, 0, 0, 0};
#pragma unroll
    for (int q = 0; q < kQatMaxSteps / 4; ++q) {
      if (q < quads) {
        const uint32_t wq[4] = {cw[q].x, cw[q].y, cw[q].z, cw[q].w};
#pragma unroll
        for (int tp = 0; tp < 4; ++tp) {
          const uint32_t w = wq[tp];
          constexpr uint32_t kLow = 0x03030303u;
          const i32x4 b = {(int)(w & kLow), (int)((w >> 2) & kLow), (int)((w >> 4) & kLow), (int)((w >> 6) & kLow)};
          acc = __builtin_amdgcn_mfma_i32_16x16x64_i8(L.op[4 * q + tp][lane], b, acc, 0, 0, 0);
        }
      }
    }
    // lane (j, g) holds tile rows 4 g .. 4 g + 3: row g / 2, limbs
    // 4 (g & 1) .. + 3; the limbs combine in wrapping 64-bit arithmetic (the
    // total is below 2^53 in magnitude, so the wrapped sum is exact)
    uint64_t p = 0;
#pragma unroll
    for (int e = 0; e < 4; ++e) p += (uint64_t)(int64_t)acc[e] << (8 * (4 * (g & 1) + e));
    p += shfl_xor_u64(p, 16);
    const int r = g >> 1;
    const uint32_t n = (uint32_t)vt * 16u + (uint32_t)j;
    const int64_t T = (int64_t)(p - 2 * (uint64_t)R.ssum[r]);
    const double dot = __builtin_ldexp((double)T, R.emin[r] != 0x7FFFFFFF ? R.emin[r] : 0);
    const float y = (float)srq(dot * (double)sc, a.out_scale);
    const bool st = (g & 1) == 0 && ok[r] && vt < t_hi;
    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, y), orr,
                                          st ? ((uint32_t)r * (uint32_t)a.V + n) * 4u : kBufferOutOfRange, 0, 0);
  };
  // two register buffers with fixed roles: tile t multiplies from one while
  // tile t + 16 loads into the other (the first load went out with the
  // check); tiles past the run read zeros and store nothing
  if (any_ok) {
    for (; vt < t_hi; vt += 2 * kQatTileWaves) {
      load(vt + kQatTileWaves, b1, s1);
      multiply(vt, b0, s0);
      load(vt + 2 * kQatTileWaves, b0, s0);
      multiply(vt + kQatTileWaves, b1, s1);
    }
  }
  // rows the check refused: the binary64 path over this run's vocabulary
  // rows, the activations staged where the operand tile was
  const bool skip[2] = {ok[0], ok[1]};
  if (!(skip[0] && (skip[1] || a.M < 2))) {
    __syncthreads();
    qat_stage_act<2, kQatTileThreads>(a, 0, L.act);
    for (int64_t r = (int64_t)t_lo * 16 + tid; r < (int64_t)t_hi * 16; r += kQatTileThreads)
      qat_row_binary64<2>(a, 0, skip, L.act, r);
  }
}

// ---- the exact integer path for batches and for every width up to 2048
//
// Rows of x in groups of 16, a group's limbs resident in LDS for the whole
// width: operand tile t holds the group's rows (kRows 16: limb t of each) or
// limbs 2t and 2t + 1 of eight of them (kRows 8, where 16 rows' limbs take
// more than 144 KB). A workgroup takes a run of 32-row vocabulary
// pairs, a pair per wave: each code word is expanded once and multiplied by
// every tile, and each limb tile read from LDS serves two vocabulary tiles
// (64 lanes x 16 bytes per 32 cycles of a CU's matrix cores). Only as many
// limbs are multiplied as the group's largest |A_k| has: 5 for activations of
// an input SRQ, 5 or 6 for normal ones. The groups of one run are on one XCD,
// so its codes come from HBM once. V 262144, D 1536, input SRQ: 3 rows
// 40 us, 16 rows 59, 32 rows 81, 48 rows 106 (714 in launches of
// qat_tile_kernel for two rows each), 64 rows 129; D 2048 without SRQ, 48 rows (eight at a time)
// 194. Bound by the limbs read from LDS and the matrix cores (38 us each at
// 48 rows); the check and the limbs take about 10 us a workgroup.
constexpr int kQatGemmThreads = 512;
constexpr int kQatGemmWaves = kQatGemmThreads / 64;
constexpr int kQatGroup = 16;
constexpr int kQatMinTiles = 3;         // limb tiles multiplied at least
constexpr int kQatOpBytes = 144 * 1024; // operand tiles in LDS

struct QatGroupRows {
  int emin[kQatGroup];                  // smallest granule exponent of the nonzero activations
  uint32_t bad[kQatGroup];
  unsigned long long sabs[kQatGroup];   // sum |A_k|
  unsigned long long ssum[kQatGroup];   // sum A_k
  uint32_t limbs;                       // of the group's largest |A_k|
};

union __attribute__((aligned(16))) QatGemmOp {
  i32x4 op[kQatOpBytes / 16];  // [tile][step][lane]
  float4 f[kQatGroup * 2048 / 4];  // the group's activations after the input SRQ, before
  double act[2 * 2048];        // the binary64 path's activations
};

// Bytes i of the four words into dword i (byte k of it from word k).
__device__ __forceinline__ void transpose_bytes(const uint32_t (&w)[4], uint32_t (&d)[4]) {
  const uint32_t a = __builtin_amdgcn_perm(w[1], w[0], 0x05010400u), b = __builtin_amdgcn_perm(w[1], w[0], 0x07030602u);
  const uint32_t c = __builtin_amdgcn_perm(w[3], w[2], 0x05010400u), e = __builtin_amdgcn_perm(w[3], w[2], 0x07030602u);
  d[0] = __builtin_amdgcn_perm(c, a, 0x05040100u);
  d[1] = __builtin_amdgcn_perm(c, a, 0x07060302u);
  d[2] = __builtin_amdgcn_perm(e, b, 0x05040100u);
  d[3] = __builtin_amdgcn_perm(e, b, 0x07060302u);
}

// The first `limbs` limbs of 16 integers (below 2^52), word W of row o of the
// group (row o of eight for kRows 8), at their operand positions (see above).
template <int kRows>
__device__ __forceinline__ void qat_store_limbs(i32x4* op, int steps, int limbs, int o, int W, const double (&A)[16]) {
  constexpr uint64_t kK = 0x0080808080808080ull;
  const int step = 4 * (W >> 4) + (W & 3), gw = (W >> 2) & 3;
  uint32_t dw[8][4];
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    uint32_t lo[4], hi[4], d[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      // the integer's two halves: whole numbers, each step exact
      const double h = __builtin_floor(A[4 * i + t] * 0x1p-32);
      const uint64_t v = ((uint64_t)(uint32_t)(int)h << 32) | (uint32_t)__builtin_fma(h, -0x1p32, A[4 * i + t]);
      const uint64_t u = (v + kK) ^ kK;
      lo[i] = (uint32_t)u;
      hi[i] = (uint32_t)(u >> 32);
    }
    transpose_bytes(lo, d);
#pragma unroll
    for (int l = 0; l < 4; ++l) dw[l][t] = d[l];
    transpose_bytes(hi, d);
#pragma unroll
    for (int l = 0; l < 4; ++l) dw[4 + l][t] = d[l];
  }
#pragma unroll
  for (int l = 0; l < 8; ++l) {
    if (l >= limbs) break;
    const int tile = kRows == 16 ? l : l >> 1, at = kRows == 16 ? o : 8 * (l & 1) + o;
    op[(tile * steps + step) * 64 + at + 16 * gw] = i32x4{(int)dw[l][0], (int)dw[l][1], (int)dw[l][2], (int)dw[l][3]};
  }
}

// The run's vocabulary pairs [p_lo, p_hi) against rows r0 .. r0 + kRows - 1 of
// the group at m0, its limbs in op.
template <int kTiles, int kRows>
__device__ __forceinline__ void qat_gemm_run(const QatArgs& a, const QatGroupRows& R, const i32x4* op, int m0, int r0,
                                             int rows_here, uint32_t ok_rows, int p_lo, int p_hi) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, j = lane & 15, g = lane >> 4;
  const int D = a.D, words = D / 16, blocks = D / 64, quads = (D + 255) / 256, steps = 4 * quads;
  const __amdgpu_buffer_rsrc_t cr =
      __builtin_amdgcn_make_buffer_rsrc((void*)a.words, (short)0, a.V * words * 4, kBufferWord3);
  const __amdgpu_buffer_rsrc_t sr = __builtin_amdgcn_make_buffer_rsrc((void*)a.scales, (short)0, a.V * 4, kBufferWord3);
  const __amdgpu_buffer_rsrc_t orr = __builtin_amdgcn_make_buffer_rsrc((void*)(a.out + (int64_t)m0 * a.V), (short)0,
                                                                       rows_here * a.V * 4, kBufferWord3);
  const double r_out = srq_reciprocal(a.out_scale);
  constexpr int kQuads = kQatMaxSteps / 4;
  u32x4 cw[2][kQuads];
  // block 4 q + g of vocabulary row n; rows past V, blocks past the width and
  // pairs past the run read zeros without a request
  auto fetch = [&](int p, int v, int q) __attribute__((always_inline)) {
    const uint32_t n = (uint32_t)p * 32u + (uint32_t)(16 * v + j);
    const bool live = p < p_hi && n < (uint32_t)a.V && 4 * q + g < blocks;
    const uint32_t off = a.block_major ? ((uint32_t)(4 * q + g) * (uint32_t)a.V + n) * 16u
                                       : (n * (uint32_t)words + (uint32_t)(16 * q + 4 * g)) * 4u;
    cw[v][q] = __builtin_amdgcn_raw_buffer_load_b128(cr, live ? off : kBufferOutOfRange, 0, 0);
  };
  // no branch around a load (see above): quads past the width read zeros
  int p = p_lo + wave;
#pragma unroll
  for (int q = 0; q < kQuads; ++q) { fetch(p, 0, q); fetch(p, 1, q); }
  // a step's limbs are read while the step before multiplies
  i32x4 limb[2][kTiles];
  auto read = [&](int step, i32x4 (&d)[kTiles]) __attribute__((always_inline)) {
#pragma unroll
    for (int t = 0; t < kTiles; ++t) d[t] = op[(t * steps + step) * 64 + lane];
  };
  read(0, limb[0]);
  for (; p < p_hi; p += kQatGemmWaves) {
    const uint32_t n0 = (uint32_t)p * 32u + (uint32_t)j;
    float sc[2];
#pragma unroll
    for (int v = 0; v < 2; ++v)
      sc[v] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(
                                            sr, n0 + 16u * v < (uint32_t)a.V ? (n0 + 16u * v) * 4u : kBufferOutOfRange, 0, 0));
    i32x4 acc[kTiles][2];
#pragma unroll
    for (int t = 0; t < kTiles; ++t) acc[t][0] = acc[t][1] = i32x4{0, 0, 0, 0};
#pragma unroll
    for (int q = 0; q < kQuads; ++q) {
      const uint32_t w0[4] = {cw[0][q].x, cw[0][q].y, cw[0][q].z, cw[0][q].w};
      const uint32_t w1[4] = {cw[1][q].x, cw[1][q].y, cw[1][q].z, cw[1][q].w};
      if (q < quads) {
#pragma unroll
        for (int tp = 0; tp < 4; ++tp) {
          const int step = 4 * q + tp;
          read(step + 1 < steps ? step + 1 : 0, limb[(tp + 1) & 1]);
          constexpr uint32_t kLow = 0x03030303u;
          const uint32_t x = w0[tp], y = w1[tp];
          const i32x4 b0 = {(int)(x & kLow), (int)((x >> 2) & kLow), (int)((x >> 4) & kLow), (int)((x >> 6) & kLow)};
          const i32x4 b1 = {(int)(y & kLow), (int)((y >> 2) & kLow), (int)((y >> 4) & kLow), (int)((y >> 6) & kLow)};
#pragma unroll
          for (int t = 0; t < kTiles; ++t) {
            acc[t][0] = __builtin_amdgcn_mfma_i32_16x16x64_i8(limb[tp & 1][t], b0, acc[t][0], 0, 0, 0);
            acc[t][1] = __builtin_amdgcn_mfma_i32_16x16x64_i8(limb[tp & 1][t], b1, acc[t][1], 0, 0, 0);
          }
          // (the limb reads of later steps hoisted over these spill registers)
          __builtin_amdgcn_sched_barrier(0);
        }
      }
      // the next pair's codes into the registers these leave
      fetch(p + kQatGemmWaves, 0, q);
      fetch(p + kQatGemmWaves, 1, q);
    }
    // lane (j, g) holds rows 4 g .. 4 g + 3 of every tile; the limbs combine
    // in wrapping 64-bit arithmetic (the totals are below 2^53)
#pragma unroll
    for (int v = 0; v < 2; ++v) {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        uint64_t s = 0;
        if constexpr (kRows == 16) {
#pragma unroll
          for (int t = 0; t < kTiles; ++t) s += (uint64_t)(int64_t)acc[t][v][e] << (8 * t);
        } else {
#pragma unroll
          for (int t = 0; t < kTiles; ++t) s += (uint64_t)(int64_t)acc[t][v][e] << (8 * (2 * t + (g >> 1)));
          s += shfl_xor_u64(s, 32);
        }
        const int r = r0 + (kRows == 16 ? 4 * g + e : 4 * (g & 1) + e);
        const int64_t T = (int64_t)(s - 2 * (uint64_t)R.ssum[r]);
        const double dot = __builtin_ldexp((double)T, R.emin[r] != 0x7FFFFFFF ? R.emin[r] : 0);
        const float y = (float)srq(dot * (double)sc[v], a.out_scale, r_out);
        const uint32_t n = n0 + 16u * v;
        const bool st = (ok_rows >> r & 1u) != 0 && n < (uint32_t)a.V && (kRows == 16 || g < 2);
        __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, y), orr,
                                              st ? ((uint32_t)r * (uint32_t)a.V + n) * 4u : kBufferOutOfRange, 0, 0);
      }
    }
  }
}

__global__ __launch_bounds__(kQatGemmThreads) void qat_gemm_kernel(QatArgs a, int32_t n_groups, int32_t n_runs) {
  __shared__ QatGemmOp L;
  __shared__ QatGroupRows R;
  const int tid = threadIdx.x;
  const int D = a.D, words = D / 16, quads = (D + 255) / 256, steps = 4 * quads;
  // runs 8 i .. 8 i + 7 of every group follow each other: run k is on XCD k % 8
  const int band = blockIdx.x / (8 * n_groups), in_band = blockIdx.x % (8 * n_groups);
  const int group = in_band / 8, run = 8 * band + in_band % 8;
  if (run >= n_runs) return;
  const int m0 = kQatGroup * group;
  const double r_in = srq_reciprocal(a.in_scale);
  const int rows_here = a.M - m0 < kQatGroup ? a.M - m0 : kQatGroup;
  const int n_pairs = (a.V + 31) / 32;
  const int p_lo = (int)((int64_t)run * n_pairs / n_runs), p_hi = (int)((int64_t)(run + 1) * n_pairs / n_runs);
  if (tid < kQatGroup) { R.emin[tid] = 0x7FFFFFFF; R.bad[tid] = 0; R.sabs[tid] = 0; R.ssum[tid] = 0; }
  if (tid == 0) R.limbs = 0;
  __syncthreads();
  // The check: a row's activations after the input SRQ into LDS with their
  // smallest granule, then the integers' sums. A row is one wave's, or
  // several waves' when the rows are few; values are reduced in the wave (LDS
  // atomics of every lane on one address took 20 us for 16 rows).
  const float4* x = (const float4*)(a.x + (int64_t)m0 * D);
  const int lane = tid & 63, wave = tid >> 6;
  const int per_row = rows_here > 4 ? 1 : (rows_here > 2 ? 2 : (rows_here > 1 ? 4 : 8));
  const int part = wave % per_row, row_step = kQatGemmWaves / per_row;
#pragma unroll 1
  for (int o = wave / per_row; o < rows_here; o += row_step) {
    int gmin = 0x7FFFFFFF;
    bool bad = false;
#pragma unroll 1
    for (int W = 64 * part + lane; W < words; W += 64 * per_row) {
      const int k = o * words + W;
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const float4 q = x[4 * k + v];
        float e[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          e[i] = (float)srq((double)e[i], a.in_scale, r_in);
          uint32_t sig;
          int g;
          if (!act_parts(e[i], &sig, &g)) bad = true;
          else if (sig) gmin = g < gmin ? g : gmin;
        }
        L.f[4 * k + v] = make_float4(e[0], e[1], e[2], e[3]);
      }
    }
    // (granules are above -256: offset, they are unsigned, below "none")
    const uint32_t least = wave_min_u32(gmin == 0x7FFFFFFF ? 0x7FFFFFFFu : (uint32_t)(gmin + 256));
    const bool any_bad = __ballot(bad) != 0;
    if (lane == 0) {
      if (least != 0x7FFFFFFFu) atomicMin(&R.emin[o], (int)least - 256);
      if (any_bad) atomicOr(&R.bad[o], 1u);
    }
  }
  __syncthreads();
#pragma unroll 1
  for (int o = wave / per_row; o < rows_here; o += row_step) {
    // The integers A_k = a_k / 2^E and their sums in binary64: whole numbers,
    // exact below 2^53, and a sum that leaves that range stays out of it (an
    // infinity or a NaN among them too).
    double sabs = 0.0, ssum = 0.0, largest = 0.0;
    const int E = R.emin[o] != 0x7FFFFFFF ? R.emin[o] : 0;
#pragma unroll 1
    for (int W = 64 * part + lane; W < words; W += 64 * per_row) {
      const int k = o * words + W;
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const float4 q = L.f[4 * k + v];
        const float e[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const double A = __builtin_ldexp((double)e[i], -E);
          sabs += fabs(A);
          ssum += A;
          largest = fmax(largest, fabs(A));
        }
      }
    }
    sabs = wave_sum_f64_dpp(sabs);
    ssum = wave_sum_f64_dpp(ssum);
    const bool fits = sabs < (double)kQatSumBound;
    const uint64_t most = wave_max_u64(fits ? (uint64_t)largest : 0ull);
    if (lane == 0) {
      // n limbs hold |A| up to 0x7F7F .. 7F (n bytes)
      uint32_t limbs = 1;
      for (int n = 1; n < kQatLimbs; ++n) limbs += most > (0x007F7F7F7F7F7F7Full >> (8 * (kQatLimbs - n))) ? 1u : 0u;
      atomicAdd(&R.sabs[o], (unsigned long long)(fits ? sabs : 0.0));
      atomicAdd(&R.ssum[o], (unsigned long long)(int64_t)(fits ? ssum : 0.0));
      if (!fits) atomicOr(&R.bad[o], 1u);
      atomicMax(&R.limbs, limbs);
    }
  }
  __syncthreads();
  uint32_t ok_rows = 0;
  for (int o = 0; o < rows_here; ++o) ok_rows |= !R.bad[o] && R.sabs[o] < kQatSumBound ? 1u << o : 0u;
  const int limbs = (int)R.limbs < kQatMinTiles ? kQatMinTiles : (int)R.limbs;

  // The limbs take the activations' place in LDS, so these are read again.
  // A refused row's limbs are zeros.
  auto word = [&](int o, int W, double (&A)[16]) __attribute__((always_inline)) {
    const int E = R.emin[o] != 0x7FFFFFFF ? R.emin[o] : 0;
    const bool ok = (ok_rows >> o & 1u) != 0;
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const float4 q = x[4 * (o * words + W) + v];
      const float e[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
      for (int i = 0; i < 4; ++i)
        A[4 * v + i] = ok ? __builtin_ldexp((double)(float)srq((double)e[i], a.in_scale, r_in), -E) : 0.0;
    }
  };
  if (ok_rows == 0) {
    // nothing for the integer path
  } else if (limbs * steps * 1024 <= kQatOpBytes) {
    __syncthreads();
#pragma unroll 1
    // (lanes along the rows: their 16-byte pieces are neighbours in LDS)
    for (int k = tid; k < rows_here * words; k += kQatGemmThreads) {
      const int o = k % rows_here, W = k / rows_here;
      double A[16];
      word(o, W, A);
      qat_store_limbs<16>(L.op, steps, limbs, o, W, A);
    }
    __syncthreads();
    switch (limbs) {
      case 3: qat_gemm_run<3, 16>(a, R, L.op, m0, 0, rows_here, ok_rows, p_lo, p_hi); break;
      case 4: qat_gemm_run<4, 16>(a, R, L.op, m0, 0, rows_here, ok_rows, p_lo, p_hi); break;
      case 5: qat_gemm_run<5, 16>(a, R, L.op, m0, 0, rows_here, ok_rows, p_lo, p_hi); break;
      case 6: qat_gemm_run<6, 16>(a, R, L.op, m0, 0, rows_here, ok_rows, p_lo, p_hi); break;
      default: qat_gemm_run<7, 16>(a, R, L.op, m0, 0, rows_here, ok_rows, p_lo, p_hi); break;
    }
  } else {
    // eight rows at a time, all limbs (4 tiles: 128 KB at width 2048)
#pragma unroll 1
    for (int r0 = 0; r0 < rows_here; r0 += 8) {
      __syncthreads();
#pragma unroll 1
      for (int k = tid; k < 8 * words; k += kQatGemmThreads) {
        const int o = k & 7, W = k / 8;
        if (r0 + o >= rows_here) continue;
        double A[16];
        word(r0 + o, W, A);
        qat_store_limbs<8>(L.op, steps, 8, o, W, A);
      }
      __syncthreads();
      if (limbs <= 6) qat_gemm_run<3, 8>(a, R, L.op, m0, r0, rows_here, ok_rows, p_lo, p_hi);
      else qat_gemm_run<4, 8>(a, R, L.op, m0, r0, rows_here, ok_rows, p_lo, p_hi);
    }
  }
  // rows the check refused: the binary64 path over this run's vocabulary rows
  for (int r0 = 0; r0 < rows_here; r0 += 2) {
    const uint32_t two = rows_here - r0 >= 2 ? 3u : 1u, ok = ok_rows >> r0 & two;
    if (ok == two) continue;
    const bool skip[2] = {(ok & 1u) != 0, (ok & 2u) != 0};
    __syncthreads();
    qat_stage_act<2, kQatGemmThreads>(a, m0 + r0, L.act);
    const int64_t end = (int64_t)p_hi * 32 < a.V ? (int64_t)p_hi * 32 : a.V;
    for (int64_t r = (int64_t)p_lo * 32 + tid; r < end; r += kQatGemmThreads)
      qat_row_binary64<2>(a, m0 + r0, skip, L.act, r);
  }
}

}  // namespace

void launch_qat_lmhead(const float* x, int32_t M, int32_t D, const uint32_t* words, int32_t block_major,
                       const float* scales, int32_t V, double in_scale, double out_scale, float* out,
                       int32_t cu_count, hipStream_t s, LaunchEvents ev) {
  QatArgs a{x, words, scales, out, D, V, M, block_major, in_scale, out_scale};
  const int cus = cu_count > 0 ? cu_count : 256;
  if (D % 256 == 0 && D <= 2048 && V % 16 == 0 && M <= 2) {
    // one or two rows: one workgroup per compute unit, the codes streamed past
    // eight limb rows (24 us at V 262144, D 1536; qat_gemm_kernel 36)
    hipExtLaunchKernelGGL(qat_tile_kernel, dim3(cus), dim3(kQatTileThreads), 0, s, ev.start, ev.stop, 0, a);
    return;
  }
  const dim3 grid((unsigned)((V + kQatThreads - 1) / kQatThreads));
  if (D <= 640 && M <= 2 && (int64_t)V * D * M <= kQatSmall) {
    // little work: the check and the limbs would take longer (one row of
    // V 32000, D 320 6 us, qat_gemm_kernel 11; of V 100003, D 576 14 and 16; of
    // V 32001, D 1088 15 and 13)
    if (M == 1) hipExtLaunchKernelGGL(qat_lmhead_kernel<1>, grid, dim3(kQatThreads), 0, s, ev.start, ev.stop, 0, a, 0);
    else hipExtLaunchKernelGGL(qat_lmhead_kernel<2>, grid, dim3(kQatThreads), 0, s, ev.start, ev.stop, 0, a, 0);
    return;
  }
  if (D <= 2048) {
    // groups of 16 rows, about one workgroup per compute unit in all (3 rows of
    // V 262144, D 1536 take 40 us, two launches of the kernel above 48)
    const int groups = (M + kQatGroup - 1) / kQatGroup;
    const int pairs = (V + 31) / 32;
    // as many runs as each XCD's compute units take at once: one workgroup
    // more on some of them doubled the time (48 rows in 85 runs 235 us)
    int runs = 8 * (cus / 8 / groups);
    runs = runs < 8 ? 8 : (runs > pairs ? pairs : runs);
    hipExtLaunchKernelGGL(qat_gemm_kernel, dim3(((runs + 7) / 8) * 8 * groups), dim3(kQatGemmThreads), 0, s, ev.start,
                          ev.stop, 0, a, groups, runs);
    return;
  }
  // wider: a launch per row
  for (int32_t m = 0; m < M; ++m)
    hipExtLaunchKernelGGL(qat_lmhead_kernel<1>, grid, dim3(kQatThreads), 0, s, m == 0 ? ev.start : nullptr,
                          m == M - 1 ? ev.stop : nullptr, 0, a, m);
}

}  // namespace gs
