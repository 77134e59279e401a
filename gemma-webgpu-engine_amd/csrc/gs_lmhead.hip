// lm_head logits producer: logits[m][v] = cap * tanh((H[m] . W[v]) / cap)
// (cap <= 0: no cap), bf16 inputs, f32 accumulate, on gfx950 MFMA.
//
// The reference's producer is an int2 QAT GEMV (src/webgpu/decode-lm-head.ts:
// 187-340); this is the bf16 tied-embedding variant the sampler consumes.
// Two kernels, one order of sums: the K steps of a row (32 wide) fall into
// eight ranges, each summed by v_mfma_f32_16x16x32_bf16 in K order, and the
// ranges are added one by one in binary32, so a logit is the same bits
// whichever kernel and batch it comes from (and about half the rounding error
// of one chain over K: 1.1e-7 against 2.0e-7 relative at D 2048).
//   * up to 64 rows, widths up to 2048: lmhead_resident_kernel, H in registers;
//   * anything else: lmhead_gemm_kernel, tiles of 128 vocabulary rows (64 for
//     narrow heads of odd vocabularies, launch_lmhead) by up to 128 rows of H. W is read from HBM once whatever M is (an XCD takes the
//     row blocks of a slab of W one after another). At D 2048, V 262144:
//     M 128 takes 220 us (5.5 TB/s), M 256 350, M 512 665 (830 TFLOP/s);
//     the resident kernel, launched once per 64 rows, took 399, 793 and 1582.
//     At M 12, D 3840, V 151643 226 us (5.2 TB/s) against 281 for a kernel
//     that held the rows of W it multiplied in registers.
// What bounds the GEMM: memory up to about 160 rows; past that the operand
// traffic of the tiles (12 TB/s from the L2s at M 512), the matrix cores 42%
// busy. The totals of the ranges take the registers that a larger tile would.
#include "gs_internal.h"

namespace gs {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

// The K range (of eight) that the sums of vocabulary row v start with. Rows
// of a multiple of 1024 bytes all start on the same few memory channels, and
// every workgroup reads its rows' lines in the order of its sums: the slabs
// of 128 rows start at different ranges, which spreads the chip's reads at
// any time over the channels (M 128, D 2048, V 262144: 265 us with one start
// for all, 230 so; widths off such strides measure the same either way).
__device__ __forceinline__ int lmhead_first_range(int64_t v, int D) { return D % 512 == 0 ? (int)((v >> 7) & 7) : 0; }

// cap tanh(x / cap) of kN values of each lane. Below 5/8 tanh q is
// q + q^3 P(q^2), P of degree 5 fitted over that range (relative error of the
// fit 2^-32; at most 0.70 ulp with its roundings); a wave whose values all lie
// there evaluates them side by side, where a tanhf a value, each behind its
// own branch, was one long chain (60 of 690 us at M 512, D 2048, V 262144).
// Their x / cap rounded to nearest takes two fused multiply-adds from
// r = 1 / cap rounded to nearest (Markstein: the remainder of q0 = x r is
// exact, and its share r completes the quotient). Every value takes the same
// formula in either branch. r = 0 (cap outside 2^+-60): always the division.
constexpr float kTanhSmall = 0.625f;
__device__ __forceinline__ float tanh_small(float q) {
  const float s = q * q;
  float p = 0x1.197b58p-9f;
  p = __builtin_fmaf(p, s, -0x1.0c213cp-7f);
  p = __builtin_fmaf(p, s, 0x1.6394d6p-6f);
  p = __builtin_fmaf(p, s, -0x1.b9ef7cp-5f);
  p = __builtin_fmaf(p, s, 0x1.11106cp-3f);
  p = __builtin_fmaf(p, s, -0x1.555554p-2f);
  return __builtin_fmaf(q * s, p, q);
}
__device__ __forceinline__ float reciprocal_of_cap(float cap) {
  return cap >= 0x1p-60f && cap <= 0x1p60f ? 1.0f / cap : 0.0f;
}
template <int kN>
__device__ __forceinline__ void lmhead_cap(float (&x)[kN], float cap, float r) {
  float q[kN];
  bool small = r != 0.0f;
#pragma unroll
  for (int e = 0; e < kN; ++e) {
    const float q0 = x[e] * r;
    q[e] = __builtin_fmaf(__builtin_fmaf(-q0, cap, x[e]), r, q0);
    small = small && __builtin_fabsf(q[e]) < kTanhSmall;  // (false for a NaN)
  }
  if (__all(small)) {
#pragma unroll
    for (int e = 0; e < kN; ++e) x[e] = cap * tanh_small(q[e]);
  } else {
#pragma unroll
    for (int e = 0; e < kN; ++e) {
      const float v = x[e] / cap;
      x[e] = cap * (__builtin_fabsf(v) < kTanhSmall ? tanh_small(v) : tanhf(v));
    }
  }
}

constexpr int kGemmThreads = 256;  // 2 x 2 waves over (V, M)
constexpr int kGemmK = 64;         // K block: one 128-byte line of every row
constexpr int kGemmChunks = 8;     // K ranges summed one by one, as the resident kernel's waves do

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) void* LdsPtr;

// One K block's rows into LDS by the memory pipe alone (no registers): wave
// instruction i of this wave takes 8 rows (lane / 8) of 128 bytes. Row r's
// 16-byte chunk c lands at position c ^ (r & 7), so that the 8 lanes of an
// operand read that go together hit 8 different 16-byte columns of the banks.
template <int kInstr, typename Rsrc>
__device__ __forceinline__ void gemm_fetch(Rsrc r, char* lds, const uint32_t (&off)[kInstr], uint32_t k) {
#ifdef __HIP_DEVICE_COMPILE__  // (the host pass refuses the 16-byte size)
#pragma unroll
  for (int i = 0; i < kInstr; ++i)
    __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (LdsPtr)(lds + 1024 * i), 16, off[i], k, 0, 0);
#endif
}

// The running tiles into the totals, at the end of a range of K.
template <int kVT, int kMT>
__device__ __forceinline__ void gemm_flush(f32x4 (&acc)[kVT][kMT], f32x4 (&total)[kVT][kMT]) {
#pragma unroll
  for (int a = 0; a < kVT; ++a) {
#pragma unroll
    for (int b = 0; b < kMT; ++b) {
      total[a][b] += acc[a][b];
      acc[a][b] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    }
  }
}

// One K block: the next fetches go out, then two K-32 steps of this wave's
// kVT x kMT tiles; a range ends (uniform) after the second step or, with
// kHalf, also after the first. The buffers are distinct objects, so the
// compiler's own waits before the reads cover nothing that is still being
// fetched.
template <int kVT, int kMT, bool kHalf, typename Rsrc>
__device__ __forceinline__ void gemm_block(const char* __restrict__ w, const char* __restrict__ h,
                                           char* __restrict__ w_next, char* __restrict__ h_next,
                                           Rsrc wr, Rsrc hr,
                                           const uint32_t (&w_off)[kVT], const uint32_t (&h_off)[kMT], uint32_t w_k,
                                           uint32_t h_k, const uint32_t (&pos)[2], bool half_flush, bool flush,
                                           f32x4 (&acc)[kVT][kMT], f32x4 (&total)[kVT][kMT]) {
  gemm_fetch<kMT>(hr, h_next, h_off, h_k);
  asm volatile("" ::: "memory");  // W's fetches stay the last kVT issued
  gemm_fetch<kVT>(wr, w_next, w_off, w_k);
  bf16x8 wf[2][kVT], hf[2][kMT];
#pragma unroll
  for (int s = 0; s < 2; ++s) {
#pragma unroll
    for (int a = 0; a < kVT; ++a) wf[s][a] = *(const bf16x8*)(w + pos[s] + 2048 * a);
#pragma unroll
    for (int b = 0; b < kMT; ++b) hf[s][b] = *(const bf16x8*)(h + pos[s] + 2048 * b);
  }
#pragma unroll
  for (int s = 0; s < 2; ++s) {
#pragma unroll
    for (int a = 0; a < kVT; ++a) {
#pragma unroll
      for (int b = 0; b < kMT; ++b)
        acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[s][a], hf[s][b], acc[a][b], 0, 0, 0);
    }
    if (kHalf && s == 0 && half_flush) gemm_flush<kVT, kMT>(acc, total);
  }
  if (flush) gemm_flush<kVT, kMT>(acc, total);
}

// kVT, kMT: 16-row tiles of W and H per wave (32 kVT vocabulary rows and
// 32 kMT rows of H per workgroup). kHalf: the resident kernel's ranges at
// widths off 512, which may end within a K block; where that kernel never runs
// they end with blocks (the flush between a block's steps costs up to 3%, and
// ranges of whole blocks would cost the resident kernel up to 6% there:
// V 32000, D 576, one row 15.9 us | 15.0).
template <int kVT, int kMT, bool kHalf>
__global__ __launch_bounds__(kGemmThreads, kVT == 2 ? 4 : 2) void lmhead_gemm_kernel(
    const uint16_t* __restrict__ H, const uint16_t* __restrict__ W, int M, int D, int V, int m_blocks, int wide,
    float cap, float* __restrict__ out) {
  constexpr int kGemmV = 32 * kVT, kRows = 32 * kMT;
  constexpr int kGemmStride = kGemmV + 4;  // LDS floats per staged output row
  constexpr int kWBytes = kGemmV * kGemmK * 2, kHBytes = kRows * kGemmK * 2;
  // three blocks of W and two of H; the staged outputs take their place
  __shared__ __attribute__((aligned(16))) char lds[3 * kWBytes + 2 * kHBytes];
  static_assert(kRows * kGemmStride * 4 <= sizeof(lds), "the staged outputs fit where the operands were");
  char *sw0 = lds, *sw1 = lds + kWBytes, *sw2 = lds + 2 * kWBytes, *sh0 = lds + 3 * kWBytes, *sh1 = sh0 + kHBytes;
  // consecutive workgroups go to the XCDs in turn: an XCD takes the row
  // blocks of one slab of W one after another, so W comes from HBM once and
  // from that XCD's L2 for the other row blocks
  const int xcd = blockIdx.x & 7, local = blockIdx.x >> 3;
  const int vt = (local / m_blocks) * 8 + xcd;
  const int64_t v0 = (int64_t)vt * kGemmV, m0 = (int64_t)(local % m_blocks) * kRows;
  if (v0 >= V) return;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int j = lane & 15, g = lane >> 4, wv = wave & 1, wm = wave >> 1;
  const int v_rows = V - v0 < kGemmV ? (int)(V - v0) : kGemmV;
  const int m_rows = M - m0 < kRows ? (int)(M - m0) : kRows;
  // rows past V or M read zeros
  const __amdgpu_buffer_rsrc_t wr =
      __builtin_amdgcn_make_buffer_rsrc((void*)(W + (size_t)v0 * D), (short)0, v_rows * D * 2, kBufferWord3);
  const __amdgpu_buffer_rsrc_t hr =
      __builtin_amdgcn_make_buffer_rsrc((void*)(H + (size_t)m0 * D), (short)0, m_rows * D * 2, kBufferWord3);
  // this wave fetches rows 8 kVT wave .. of W's block and 8 kMT wave .. of H's
  const int lr = lane >> 3, lc = ((lane & 7) ^ lr) * 16;
  uint32_t w_off[kVT], h_off[kMT];
#pragma unroll
  for (int i = 0; i < kVT; ++i) w_off[i] = (uint32_t)((8 * kVT * wave + 8 * i + lr) * D * 2 + lc);
#pragma unroll
  for (int i = 0; i < kMT; ++i) h_off[i] = (uint32_t)((8 * kMT * wave + 8 * i + lr) * D * 2 + lc);
  const int w_dst = 8 * kVT * wave * 128, h_dst = 8 * kMT * wave * 128;
  // operand reads: lane (j, g) holds k = 32 s + 8 g .. + 7 of row j of a tile
  uint32_t pos[2];
#pragma unroll
  for (int s = 0; s < 2; ++s) pos[s] = (uint32_t)(j * 128 + (((4 * s + g) ^ (j & 7)) * 16));
  const int w_src = 16 * kVT * wv * 128, h_src = 16 * kMT * wm * 128;

  f32x4 acc[kVT][kMT], total[kVT][kMT];
#pragma unroll
  for (int a = 0; a < kVT; ++a) {
#pragma unroll
    for (int b = 0; b < kMT; ++b) {
      acc[a][b] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
      total[a][b] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    }
  }
  const int nk = D / kGemmK;
  int range = 0, bound = 0;  // `bound`: the K step that ends the current range (empty ranges are passed over)
  auto next_bound = [&]() __attribute__((always_inline)) {
    const int done = bound;
    do {
      ++range;
      bound = kHalf ? range * 2 * nk / kGemmChunks : 2 * (range * nk / kGemmChunks);
    } while (bound == done && range < kGemmChunks);
  };
  next_bound();
  const int first = lmhead_first_range(v0, D) * (nk / kGemmChunks);  // blocks wrap around after the last
  auto at = [&](int kb) __attribute__((always_inline)) {
    const int k = (kb < nk ? kb : nk - 1) + first;
    return (uint32_t)((k < nk ? k : k - nk) * kGemmK * 2);
  };
  auto block = [&](int kb, char* w, char* h, char* wn, char* hn) __attribute__((always_inline)) {
    // block kb's rows have landed for every wave (W's block kb + 1, fetched
    // after them, may still be under way), and every wave has read block kb - 1
    if constexpr (kVT == 4) asm volatile("s_waitcnt vmcnt(4) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    else asm volatile("s_waitcnt vmcnt(2) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    const bool half_flush = kHalf && 2 * kb + 1 == bound;
    if (half_flush) next_bound();
    const bool flush = 2 * kb + 2 == bound;
    if (flush) next_bound();
    gemm_block<kVT, kMT, kHalf>(w + w_src, h + h_src, wn + w_dst, hn + h_dst, wr, hr, w_off, h_off, at(kb + 2), at(kb + 1),
                           pos, half_flush, flush, acc, total);
  };
  gemm_fetch<kVT>(wr, sw0 + w_dst, w_off, at(0));
  gemm_fetch<kMT>(hr, sh0 + h_dst, h_off, at(0));
  asm volatile("" ::: "memory");
  gemm_fetch<kVT>(wr, sw1 + w_dst, w_off, at(1));
  // blocks past the last are fetched as the last one again, and not read
  for (int kb = 0;; kb += 6) {
    block(kb, sw0, sh0, sw2, sh1);
    if (kb + 1 >= nk) break;
    block(kb + 1, sw1, sh1, sw0, sh0);
    if (kb + 2 >= nk) break;
    block(kb + 2, sw2, sh0, sw1, sh1);
    if (kb + 3 >= nk) break;
    block(kb + 3, sw0, sh1, sw2, sh0);
    if (kb + 4 >= nk) break;
    block(kb + 4, sw1, sh0, sw0, sh1);
    if (kb + 5 >= nk) break;
    block(kb + 5, sw2, sh1, sw1, sh0);
    if (kb + 6 >= nk) break;
  }
  // nothing is in flight to or from LDS before the outputs take its place
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");

  // the cap, then the tile [m][v] through LDS, so that rows go out in pieces
  // of 512 bytes (D layout: lane (j, g) holds column j, rows 4 g + e; the
  // column is H's row, the rows are W's)
  float* stage = (float*)lds;
  const float rcap = reciprocal_of_cap(cap);
#pragma unroll
  for (int b = 0; b < kMT; ++b) {
#pragma unroll
    for (int a = 0; a < kVT; ++a) {
      float x[4] = {total[a][b][0], total[a][b][1], total[a][b][2], total[a][b][3]};
      if (cap > 0.0f) lmhead_cap<4>(x, cap, rcap);
      *(f32x4*)&stage[(16 * (kMT * wm + b) + j) * kGemmStride + 16 * kVT * wv + 16 * a + 4 * g] = f32x4{x[0], x[1], x[2], x[3]};
    }
  }
  __syncthreads();
  float* o = out + (size_t)m0 * V + v0;
  if (wide) {  // V % 4 == 0 and 16-byte aligned logits: a piece lies within its row
#pragma unroll 4
    for (int q = tid; q < kRows * kGemmV / 4; q += kGemmThreads) {
      const int row = q / (kGemmV / 4), c = 4 * (q % (kGemmV / 4));
      if (row < m_rows && c < v_rows)
        __builtin_nontemporal_store(*(const f32x4*)&stage[row * kGemmStride + c], (f32x4*)&o[(size_t)row * V + c]);
    }
  } else {
#pragma unroll 4
    for (int q = tid; q < kRows * kGemmV; q += kGemmThreads) {
      const int row = q / kGemmV, c = q % kGemmV;
      if (row < m_rows && c < v_rows)
        __builtin_nontemporal_store(stage[row * kGemmStride + c], &o[(size_t)row * V + c]);
    }
  }
}

// Resident-H kernel for widths up to 2048: one workgroup per compute unit
// holds its 64-row block of H in registers for the whole launch and streams
// W in steps of 16 vocabulary rows, in runs of 16 steps (256 rows, 1 MB at
// D 2048) dealt round-robin to the workgroups, so the chip reads a window of
// adjacent runs at a time (199 us against 203 us for one contiguous range
// per workgroup).
//   * 8 waves split K: wave w owns the 32-wide K steps [w nS / 8, (w+1) nS / 8)
//     of the nS = D / 32, its H slice (64 rows) held as MFMA A operands
//     (v_mfma_f32_16x16x32_bf16: lane i + 16 g holds k = 32 s + 8 g .. + 7 of
//     row i of an M tile, 4 M tiles);
//   * per step a lane loads 16 bytes per K step of one vocabulary row (the
//     B operand), so the workgroup reads 16 whole rows of W (16 x 2D bytes,
//     contiguous) per step; two steps of loads are in flight per wave;
//   * the 8 waves' partial 64x16 tiles go through LDS (double-buffered), and
//     after one barrier each thread adds two outputs' partials in the order of
//     their ranges (lmhead_first_range)
//     and applies the cap into an LDS stage of 16 steps, which then goes out
//     as 1 KB runs of each logits row in 16-byte stores. At M 64, D 2048,
//     V 262144 the logits cost 73 us of 258 stored per step (64-byte pieces
//     of 64 rows 4V bytes apart), 31 us of 216 staged over 8 steps, 19 us of
//     204 over 16 (185 us without stores); spreading a double-buffered stage's
//     stores over the next run's steps took 224 us, write-back stores 237 us.
// Every global access is a buffer access with no branch around it: rows past
// V or M, K steps a wave does not own, and the steps past a workgroup's run
// take an out-of-range offset (zeros, no memory request; stores dropped). The
// compiler's wait counts then cover exactly the loads a step consumes, as
// loads and stores share one in-order counter on this part.
constexpr int kResM = 64;         // hidden rows at most
constexpr int kResWaves = 8;
constexpr int kResThreads = 64 * kResWaves;
constexpr int kResN = 16;         // vocabulary rows per step
constexpr int kResStride = 68;    // LDS floats per vocabulary row of a partial (64 + 4)
constexpr int kResMaxWidth = 2048;
constexpr int32_t kResNT = 2;     // non-temporal cache policy of the streams
constexpr int kResStage = 16;     // steps of logits staged per flush
constexpr int kResStageStride = kResStage * kResN + 4;  // LDS floats per staged row

template <int kS>  // K steps per wave, at most 8
__global__ __launch_bounds__(kResThreads) void lmhead_resident_kernel(const uint16_t* __restrict__ H,
                                                                      const uint16_t* __restrict__ W, int M, int D,
                                                                      int V, float cap, float* __restrict__ out) {
  __shared__ __attribute__((aligned(16))) float red[2][kResWaves][kResN * kResStride];
  __shared__ __attribute__((aligned(16))) float stage[64 * kResStageStride];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int j = lane & 15, g = lane >> 4;
  const int n_steps = D / 32;
  const int s_lo = wave * n_steps / kResWaves, s_hi = (wave + 1) * n_steps / kResWaves;
  const int my_steps = s_hi - s_lo;  // kS or kS - 1
  // this workgroup's steps k = 0 .. k_end - 1: run blockIdx.x + gridDim.x r
  // (r = k / kResStage), tile kResStage run + k % kResStage of 16 vocabulary
  // rows; steps on tiles past the last are empty
  const int n_tiles = (V + kResN - 1) / kResN;
  const int n_runs = (n_tiles + kResStage - 1) / kResStage;
  const int k_end = n_runs > (int)blockIdx.x ? ((n_runs - 1 - (int)blockIdx.x) / (int)gridDim.x + 1) * kResStage : 0;
  auto tile_of = [&](int k) __attribute__((always_inline)) {
    return ((int)blockIdx.x + (int)gridDim.x * (k / kResStage)) * kResStage + k % kResStage;
  };
  // byte offsets of this lane's K step s within a row of H or W
  uint32_t k_off[kS];
#pragma unroll
  for (int s = 0; s < kS; ++s) k_off[s] = s < my_steps ? (uint32_t)(64 * (s_lo + s) + 16 * g) : kBufferOutOfRange;

  // H slice: rows 16 mt + j of the M tiles (rows past M read zeros)
  const __amdgpu_buffer_rsrc_t hr =
      __builtin_amdgcn_make_buffer_rsrc((void*)H, (short)0, M * D * 2, kBufferWord3);
  bf16x8 hreg[4][kS];
#pragma unroll
  for (int mt = 0; mt < 4; ++mt) {
#pragma unroll
    for (int s = 0; s < kS; ++s) {
      const u32x4 v = __builtin_amdgcn_raw_buffer_load_b128(hr, k_off[s] + (uint32_t)((16 * mt + j) * D * 2), 0, 0);
      hreg[mt][s] = __builtin_bit_cast(bf16x8, v);
    }
  }
  u32x4 wbuf[2][kS];
  // step k's rows in a resource of their own (empty past the steps or the
  // tiles, short at V)
  auto issue = [&](int slot, int k) __attribute__((always_inline)) {
    const int t = tile_of(k);
    const bool live = k < k_end && t < n_tiles;
    const int rows = live ? (V - t * kResN < kResN ? V - t * kResN : kResN) : 0;
    const __amdgpu_buffer_rsrc_t wr = __builtin_amdgcn_make_buffer_rsrc(
        (void*)(W + (size_t)(live ? t : 0) * kResN * D), (short)0, rows * D * 2, kBufferWord3);
    const uint32_t row_off = (uint32_t)(j * D * 2);
#pragma unroll
    for (int s = 0; s < kS; ++s) wbuf[slot][s] = __builtin_amdgcn_raw_buffer_load_b128(wr, row_off + k_off[s], 0, kResNT);
  };
  // the output block: rows past M fall outside the resource
  const __amdgpu_buffer_rsrc_t orc =
      __builtin_amdgcn_make_buffer_rsrc((void*)out, (short)0, M * V * 4, kBufferWord3);
  // reduction role: outputs (m, n) = (2 (tid >> 4) + e, tid & 15), e = 0, 1
  const int rn = tid & 15, rm = 2 * (tid >> 4);
  const float rcap = reciprocal_of_cap(cap);
  auto step = [&](int k, int u) __attribute__((always_inline)) {
    const int slot = u & 1;
    f32x4 acc[4];
#pragma unroll
    for (int mt = 0; mt < 4; ++mt) acc[mt] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int s = 0; s < kS; ++s) {
      const bf16x8 b = __builtin_bit_cast(bf16x8, wbuf[slot][s]);
#pragma unroll
      for (int mt = 0; mt < 4; ++mt) acc[mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(hreg[mt][s], b, acc[mt], 0, 0, 0);
    }
    issue(slot, k + 2);
    // lane (j, g) holds rows 16 mt + 4 g + e of column j
    float* r = &red[slot][wave][j * kResStride + 4 * g];
#pragma unroll
    for (int mt = 0; mt < 4; ++mt) *(f32x4*)(r + 16 * mt) = acc[mt];
    __syncthreads();
    const int first = lmhead_first_range((int64_t)tile_of(k) * kResN, D);
    float x[2] = {0.0f, 0.0f};
#pragma unroll
    for (int i = 0; i < kResWaves; ++i) {
      const int w = (first + i) & (kResWaves - 1);
      const float2 p = *(const float2*)&red[slot][w][rn * kResStride + rm];
      x[0] += p.x;
      x[1] += p.y;
    }
    if (cap > 0.0f) lmhead_cap<2>(x, cap, rcap);
    stage[rm * kResStageStride + kResN * u + rn] = x[0];
    stage[(rm + 1) * kResStageStride + kResN * u + rn] = x[1];
  };
  // a staged run: piece q = tid + 512 i is 16 bytes of row q / 64 at column
  // 4 (q % 64), so a wave writes one row's 1 KB. Columns of tiles past the
  // last, or past V, are dropped (V % 4 == 0: a piece lies within its row).
  constexpr int kRowPieces = kResStage * kResN / 4;  // 64
  auto flush = [&](int k0) __attribute__((always_inline)) {
    const int t0 = tile_of(k0);
#pragma unroll
    for (int i = 0; i < 64 * kRowPieces / kResThreads; ++i) {
      const int q = tid + kResThreads * i, row = q / kRowPieces, c = 4 * (q % kRowPieces);
      const f32x4 v = *(const f32x4*)&stage[row * kResStageStride + c];
      const int n = t0 * kResN + c;
      const uint32_t o = t0 + c / kResN < n_tiles && n < V ? (uint32_t)(row * V + n) * 4u : kBufferOutOfRange;
      __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, v), orc, o, 0, kResNT);
    }
  };
  // Straight-line runs of kResStage steps (even, so the two load slots
  // alternate in place); steps past the tiles read zeros and drop their
  // stores. The reduction buffer of step u is u & 1: the barrier of
  // step u + 1 orders step u's reads before step u + 2's writes; the barrier
  // before a flush orders the stage's writes before its reads, and the next
  // run's first barrier its reads before the next writes.
  auto run = [&](int k0) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < kResStage; ++u) step(k0 + u, u);
    __syncthreads();
    flush(k0);
  };
  issue(0, 0);
  // keep the first step's loads ahead of the second's (waits count in issue order)
  __builtin_amdgcn_sched_barrier(0);
  issue(1, 1);
  for (int k0 = 0; k0 < k_end; k0 += kResStage) run(k0);
}

}  // namespace

void launch_lmhead(const uint16_t* hidden, const uint16_t* weight, int32_t m, int32_t width, int32_t vocab,
                   float softcap, float* out, int32_t cu_count, hipStream_t s, LaunchEvents ev) {
  const bool resident = width <= kResMaxWidth && width % 32 == 0 && vocab % 4 == 0 &&
                        (int64_t)vocab * kResM * 4 < ((int64_t)1 << 31);
  if (resident && m <= kResM && ((uintptr_t)out & 15) == 0) {
    // one workgroup per compute unit
    const int k_steps = (width / 32 + kResWaves - 1) / kResWaves;
    const dim3 grid(cu_count > 0 ? cu_count : 256), block(kResThreads);
    switch (k_steps) {
#define GS_RES_CASE(k)                                                                                               \
  case k:                                                                                                            \
    hipExtLaunchKernelGGL(lmhead_resident_kernel<k>, grid, block, 0, s, ev.start, ev.stop, 0, hidden, weight, m,     \
                          width, vocab, softcap, out);                                                               \
    break;
      GS_RES_CASE(1)
      GS_RES_CASE(2)
      GS_RES_CASE(3)
      GS_RES_CASE(4)
      GS_RES_CASE(5)
      GS_RES_CASE(6)
      GS_RES_CASE(7)
      GS_RES_CASE(8)
#undef GS_RES_CASE
    }
    return;
  }
  // blocks of at most 128 rows of H, the rows spread evenly over them
  const int m_blocks = (m + 127) / 128;
  const int tiles = ((m + m_blocks - 1) / m_blocks + 31) / 32;  // per wave: 1 .. 4
  const int half = resident && width % 512 != 0;
  // Tiles of 64 vocabulary rows, four workgroups a compute unit, where a row
  // block is small, the larger tiles would take more than one round of
  // workgroups and the weights about fit the last-level cache: the start and
  // end of a workgroup weigh there. 64 rows of V 151643, D 704 46 us (50 in
  // tiles of 128), V 200003, D 512 51 (56), V 262143, D 512 57 (67), but V 50257,
  // D 704 19 (17) and V 262143, D 576 79 (73), D 3840 436 (361).
  const int cus = cu_count > 0 ? cu_count : 256;
  const bool narrow = tiles <= 2 && !half && (vocab + 127) / 128 > 2 * cus && (int64_t)vocab * width <= 145000000;
  const int v_rows = narrow ? 64 : 128;
  const int v_tiles = (vocab + v_rows - 1) / v_rows;
  const dim3 grid((unsigned)((v_tiles + 7) / 8 * 8 * m_blocks)), block(kGemmThreads);
  const int wide = vocab % 4 == 0 && ((uintptr_t)out & 15) == 0;
  switch (narrow ? 20 + tiles : (half ? 10 + tiles : tiles)) {
#define GS_GEMM_CASE(n, vt, k, half)                                                                                   \
  case n:                                                                                                              \
    hipExtLaunchKernelGGL((lmhead_gemm_kernel<vt, k, half>), grid, block, 0, s, ev.start, ev.stop, 0, hidden, weight,  \
                          m, width, vocab, m_blocks, wide, softcap, out);                                              \
    break;
    GS_GEMM_CASE(1, 4, 1, false)
    GS_GEMM_CASE(2, 4, 2, false)
    GS_GEMM_CASE(3, 4, 3, false)
    GS_GEMM_CASE(4, 4, 4, false)
    GS_GEMM_CASE(11, 4, 1, true)
    GS_GEMM_CASE(12, 4, 2, true)
    GS_GEMM_CASE(13, 4, 3, true)
    GS_GEMM_CASE(14, 4, 4, true)
    GS_GEMM_CASE(21, 2, 1, false)
    GS_GEMM_CASE(22, 2, 2, false)
#undef GS_GEMM_CASE
  }
}

}  // namespace gs
