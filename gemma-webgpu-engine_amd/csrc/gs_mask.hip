// Constraint masker and raw-logit log-probability.
//
// walk_masks_kernel and build_masks_kernel: legalTokenIds
// (src/runtime/constraints.ts:56-92) for a byte-level DFA, as a 262144-bit
// mask per requested state. The reference walks a token-byte trie
// depth-first; here every token walks its own bytes
// (the vocab is a CSR of token byte strings), one token per lane, against a
// next-state table whose entries already fold in viability
// (src/runtime/constraints.ts:253-265, 300-322): next'[s][b] = -1 unless the
// edge exists and its target can still reach a final state. A token is legal
// from s iff it has at least one byte and no step yields -1 -- the set the
// trie DFS emits. Lanes of a wave64 cover 64 consecutive ids, so one ballot
// gives two mask words.
//
// logprob_part_kernel + logprob_join_kernel: tokenLogProbability
// (src/runtime/sampling.ts:67-80).
//
// mask_fill_kernel + mask_copy_kernel: maskConstraintLogits
// (src/runtime/constraints.ts:159-173): a row of -Infinity, then the raw
// logit copied back at every listed id inside [0, n). Listed ids may repeat
// (legal and termination lists overlap); repeats store the same value.
#include <algorithm>

#include "gs_exp2.h"
#include "gs_internal.h"

namespace gs {
namespace {

constexpr int kMaskThreads = 1024;
constexpr int kMaskWaves = kMaskThreads / 64;
constexpr int kMaskStates = 64;  // requested states walked together, a bit each
constexpr int kLdsStates = 192;  // tables up to 192 x 256 x int16 (96 KiB) stay in LDS

// A token's first 16 bytes (past its end its last one again).
__device__ __forceinline__ void token_bytes(const uint8_t* bytes, int64_t b0, int len, uint64_t* lo, uint64_t* hi) {
  *lo = *hi = 0;
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const uint64_t v = len > 0 ? bytes[b0 + (i < len ? i : len - 1)] : 0u;
    if (i < 8) *lo |= v << (8 * i);
    else *hi |= v << (8 * (i - 8));
  }
}

constexpr int kWalkThreads = 256;
constexpr int kWalkLdsStates = 96;  // tables up to 48 KiB
constexpr int kWalkLdsVocab = 196608;

// Every token walked from each requested state in turn, a wave waiting for
// its longest lane (launch_masks says where this is the faster kernel).
template <bool kInLds>
__global__ __launch_bounds__(kWalkThreads) void walk_masks_kernel(const int64_t* offsets, const uint8_t* bytes,
                                                                  int32_t vocab, const int16_t* next,
                                                                  int32_t n_states, const int32_t* states, int32_t n,
                                                                  uint32_t* masks, int32_t mask_words) {
  __shared__ uint4 s_next[kInLds ? kWalkLdsStates * 32 : 1];
  const int lane = threadIdx.x & 63;
  const int64_t t = (int64_t)blockIdx.x * kWalkThreads + threadIdx.x;
  int64_t b0 = 0, b1 = 0;
  if (t < vocab) { b0 = offsets[t]; b1 = offsets[t + 1]; }
  const int len = (int)(b1 - b0);
  uint64_t lo, hi;
  token_bytes(bytes, b0, len, &lo, &hi);
  if (kInLds) {
    for (int i = threadIdx.x; i < n_states * 32; i += kWalkThreads) s_next[i] = ((const uint4*)next)[i];
    __syncthreads();
  }
  const int16_t* table = kInLds ? (const int16_t*)s_next : next;
  const int64_t word = ((t & ~63ll) >> 5) + lane;
  for (int q = 0; q < n; ++q) {
    int32_t s = states[q];
    bool legal = len > 0 && s >= 0 && s < n_states;
    for (int i = 0; legal && i < len; ++i) {
      const uint32_t b = i < 8 ? (uint32_t)(lo >> (8 * i)) & 0xFFu
                               : (i < 16 ? (uint32_t)(hi >> (8 * (i - 8))) & 0xFFu : bytes[b0 + i]);
      s = table[s * 256 + (int)b];
      legal = s >= 0;
    }
    const uint64_t bits = __ballot(legal);
    if (lane < 2 && word < mask_words) masks[(int64_t)q * mask_words + word] = (uint32_t)(bits >> (32 * lane));
  }
}

struct MaskLds {
  int16_t next[kLdsStates * 256];
  int16_t first[256][kMaskStates + 2];       // the state after a token's first byte (rows a bank apart)
  uint16_t alive[256][kMaskStates / 16];     // bit q: that state is not dead
  uint32_t out[kMaskStates][2 * kMaskWaves]; // the workgroup's mask words
};

// kMaskStates requested states at a time. A token's first byte rules most of
// them out at once: `alive` holds, for every byte, the states that survive it,
// and each lane then walks its token from the survivors alone, one after the
// other, the next survivor's state read while this one walks. The lanes'
// bits are turned into mask words by ballots. Walking every token from every
// state, lanes waiting for the longest of 64, took 103 us for 64 states over
// 262144 tokens.
template <bool kInLds>
__global__ __launch_bounds__(kMaskThreads) void build_masks_kernel(const int64_t* offsets, const uint8_t* bytes,
                                                                   int32_t vocab, const int16_t* next,
                                                                   int32_t n_states, const int32_t* states,
                                                                   int32_t n, uint32_t* masks, int32_t mask_words) {
  __shared__ MaskLds L;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int64_t t = (int64_t)blockIdx.x * kMaskThreads + tid;
  int64_t b0 = 0, b1 = 0;
  if (t < vocab) { b0 = offsets[t]; b1 = offsets[t + 1]; }
  const int len = (int)(b1 - b0);
  if (kInLds) {
    // 512 bytes a state: whole 16-byte pieces
    for (int i = tid; i < n_states * 32; i += kMaskThreads) ((uint4*)L.next)[i] = ((const uint4*)next)[i];
  }
  // the first 16 bytes in registers, the rest read on demand
  uint64_t lo, hi;
  token_bytes(bytes, b0, len, &lo, &hi);
  __syncthreads();
  const int16_t* table = kInLds ? L.next : next;
  for (int q0 = 0; q0 < n; q0 += kMaskStates) {
    const int nq = n - q0 < kMaskStates ? n - q0 : kMaskStates;
    // thread (byte, part): 16 of the states' first steps
    {
      const int byte = tid & 255, part = tid >> 8;
      uint32_t m = 0;
#pragma unroll
      for (int k = 0; k < 16; ++k) {
        const int q = 16 * part + k;
        const int32_t s = q < nq ? states[q0 + q] : -1;
        const int16_t s1 = s >= 0 && s < n_states ? table[s * 256 + byte] : (int16_t)-1;
        L.first[byte][q] = s1;
        m |= s1 >= 0 ? 1u << k : 0u;
      }
      L.alive[byte][part] = (uint16_t)m;
    }
    __syncthreads();
    uint64_t legal = 0;
    if (len > 0) {
      const int first = (int)(lo & 0xFFu);
      uint64_t left = 0;
#pragma unroll
      for (int part = 0; part < kMaskStates / 16; ++part) left |= (uint64_t)L.alive[first][part] << (16 * part);
      if (len == 1) {
        legal = left;
      } else if (left) {
        int q = __builtin_ctzll(left), i = 1;
        int32_t s = L.first[first][q];
        left &= left - 1;
        int32_t s_next = left ? L.first[first][__builtin_ctzll(left)] : 0;
        for (;;) {
          const uint32_t b = i < 8 ? (uint32_t)(lo >> (8 * i)) & 0xFFu
                                   : (i < 16 ? (uint32_t)(hi >> (8 * (i - 8))) & 0xFFu : bytes[b0 + i]);
          s = table[s * 256 + (int)b];
          ++i;
          if (s >= 0 && i < len) continue;
          if (s >= 0) legal |= 1ull << q;
          if (!left) break;
          q = __builtin_ctzll(left);
          left &= left - 1;
          s = s_next;
          i = 1;
          if (left) s_next = L.first[first][__builtin_ctzll(left)];
        }
      }
    }
#pragma unroll 8
    for (int q = 0; q < kMaskStates; ++q) {
      const uint64_t bits = __ballot((legal >> q & 1u) != 0);
      if (lane < 2) L.out[q][2 * wave + lane] = (uint32_t)(bits >> (32 * lane));
    }
    __syncthreads();
    for (int i = tid; i < nq * 2 * kMaskWaves; i += kMaskThreads) {
      const int q = i / (2 * kMaskWaves), w = i % (2 * kMaskWaves);
      const int64_t word = (int64_t)blockIdx.x * (2 * kMaskWaves) + w;
      if (word < mask_words) masks[(int64_t)(q0 + q) * mask_words + word] = L.out[q][w];
    }
    __syncthreads();
  }
}

// ---- tokenLogProbability
//
// out = l_t - M - ln sum e^(l - M), the sum in binary64. Bound by reading the
// row once: rows are split into parts over workgroups (the chip is idle with
// one workgroup per row), every thread takes its logits as 16-byte loads, and
// keeps a running maximum and sum, so there is one pass. An exponential is 14
// binary64 operations: e^d = 2^(j/32) 2^k e^r with |r| <= ln2/64, the e^r of
// degree 6 (truncation 3.5e-18) and the 32 factors, correctly rounded, in one
// LDS bank pair each, so that random j never conflict. 128 rows of 262144 f32
// take 39 + 4 us (3.4 TB/s); one 1024-thread workgroup per row with two
// passes of 4-byte loads and fdlibm's exp took 297 us.
constexpr int kLogThreads = 256;
constexpr int kLogVecs = 4;  // 16-byte loads in flight per thread
constexpr int kLogParts = 2048;  // parts of a split call

struct LogPart {
  double sum;  // sum of e^(l - max) over the part
  float max;   // its maximum (-inf: no finite logit; NaN propagates)
  uint32_t pad;
};

// (m, s) joined with (om, os): both sums relative to the larger maximum. A
// maximum of -inf has a sum of 0, one of NaN or +inf makes the sum NaN, as
// the reference's l - M does.
__device__ __forceinline__ void join_sums(float& m, double& s, float om, double os, const double* tab) {
  const float n = __builtin_elementwise_maximum(m, om);
  if (!(n > -__builtin_inff())) {  // -inf or NaN
    s = n != n ? (double)n : 0.0;
  } else if (n == __builtin_inff()) {
    s = __builtin_nan("");
  } else {
    s = s * exp_neg((double)m - (double)n, tab) + os * exp_neg((double)om - (double)n, tab);
  }
  m = n;
}

__device__ __forceinline__ void wave_join(float& m, double& s, const double* tab) {
  for (int k = 32; k > 0; k >>= 1) {
    const float om = __builtin_bit_cast(float, shfl_xor_u32(__builtin_bit_cast(uint32_t, m), k));
    const double os = shfl_xor_f64(s, k);
    join_sums(m, s, om, os, tab);
  }
}

template <typename In>
__device__ __forceinline__ float logit_f32(In v) {
  if constexpr (sizeof(In) == 2) return __builtin_bit_cast(float, (uint32_t)v << 16);
  else return v;
}

// out for a row whose maximum and sum are known
template <typename In>
__device__ __forceinline__ double log_prob(const In* row, int32_t vocab, int32_t tok, float m, double s) {
  // M = -inf: every l - M is NaN
  if (!(m > -__builtin_inff()) || tok < 0 || tok >= vocab) return __builtin_nan("");
  return (double)logit_f32<In>(row[tok]) - (double)m - gsm::js_log(s);
}

// Part `blockIdx.x % parts` of row `blockIdx.x / parts`.
template <typename In>
__global__ __launch_bounds__(kLogThreads) void logprob_part_kernel(const In* logits, int64_t stride, int32_t vocab,
                                                                   const int32_t* tokens, int32_t parts,
                                                                   LogPart* partial, double* out) {
  constexpr int kVec = 16 / (int)sizeof(In);
  __shared__ double tab[kExpTable];
  __shared__ double s_sum[kLogThreads / 64];
  __shared__ float s_max[kLogThreads / 64];
  load_exp_table(tab);
  const int64_t row = blockIdx.x / parts;
  const int part = (int)(blockIdx.x % parts);
  const In* base = logits + row * stride;
  // the row's 16-byte aligned pieces [0, nv) start at element `head`; the few
  // elements before and after them go to part 0's first threads
  const int to_aligned = (int)((16u - ((uintptr_t)base & 15u)) & 15u) / (int)sizeof(In);
  const int head = to_aligned < vocab ? to_aligned : vocab;
  const int nv = (vocab - head) / kVec;
  const int tail = head + nv * kVec;
  const int v0 = (int)((int64_t)nv * part / parts), v1 = (int)((int64_t)nv * (part + 1) / parts);
  float m = -__builtin_inff();
  double s = 0.0;
  const int tid = threadIdx.x;
  if (part == 0) {
    if (tid < head) m = logit_f32<In>(base[tid]);
    else if (tid - head < vocab - tail) m = logit_f32<In>(base[tail + tid - head]);
    if (m > -__builtin_inff() && m < __builtin_inff()) s = 1.0;
  }
  const uint4* vecs = (const uint4*)(base + head);
  for (int v = v0 + tid; v < v1; v += kLogThreads * kLogVecs) {
    uint4 w[kLogVecs];
#pragma unroll
    for (int i = 0; i < kLogVecs; ++i) {
      const int q = v + i * kLogThreads;
      w[i] = load_nt16(vecs + (q < v1 ? q : v1 - 1));
    }
    const int wave_v = __builtin_amdgcn_readfirstlane(v);  // its first lane's: the lowest
    float x[kLogVecs][kVec];
    float n = m;
#pragma unroll
    for (int i = 0; i < kLogVecs; ++i) {
      const bool in = v + i * kLogThreads < v1;
      const uint32_t d[4] = {w[i].x, w[i].y, w[i].z, w[i].w};
#pragma unroll
      for (int j = 0; j < kVec; ++j) {
        uint32_t b;
        if constexpr (sizeof(In) == 4) b = d[j];
        else b = (j & 1) ? d[j >> 1] & 0xFFFF0000u : d[j >> 1] << 16;
        x[i][j] = in ? __builtin_bit_cast(float, b) : -__builtin_inff();
        n = __builtin_elementwise_maximum(n, x[i][j]);
      }
    }
    // a maximum that is not finite is settled where sums are joined
    const bool live = n > -__builtin_inff() && n < __builtin_inff();
    if (live && n > m) s *= exp_neg((double)m - (double)n, tab);
    m = n;
    if (live) {
#pragma unroll
      for (int i = 0; i < kLogVecs; ++i) {
        // (pieces past the part's end for the whole wave: a short row's work is its first)
        if (i > 0 && wave_v + i * kLogThreads >= v1) break;
#pragma unroll
        for (int j = 0; j < kVec; ++j) s += exp_neg((double)x[i][j] - (double)n, tab);
      }
    }
  }
  wave_join(m, s, tab);
  const int wave = tid >> 6;
  if ((tid & 63) == 0) { s_max[wave] = m; s_sum[wave] = s; }
  __syncthreads();
  if (tid != 0) return;
  for (int w = 1; w < kLogThreads / 64; ++w) join_sums(m, s, s_max[w], s_sum[w], tab);
  if (parts == 1) out[row] = log_prob<In>(base, vocab, tokens[row], m, s);
  else partial[blockIdx.x] = LogPart{s, m, 0};
}

// One wave per row joins its parts (at most 64, one per lane).
template <typename In>
__global__ __launch_bounds__(kLogThreads) void logprob_join_kernel(const In* logits, int64_t stride, int32_t vocab,
                                                                   int32_t rows, const int32_t* tokens, int32_t parts,
                                                                   const LogPart* partial, double* out) {
  __shared__ double tab[kExpTable];
  load_exp_table(tab);
  const int lane = threadIdx.x & 63;
  const int64_t row = (int64_t)blockIdx.x * (kLogThreads / 64) + (threadIdx.x >> 6);
  if (row >= rows) return;
  float m = -__builtin_inff();
  double s = 0.0;
  if (lane < parts) {
    const LogPart p = partial[row * parts + lane];
    m = p.max;
    s = p.sum;
  }
  wave_join(m, s, tab);
  if (lane == 0) out[row] = log_prob<In>(logits + row * stride, vocab, tokens[row], m, s);
}

constexpr int kFillThreads = 256;

__global__ __launch_bounds__(kFillThreads) void mask_fill_kernel(float* out, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * kFillThreads + threadIdx.x;
  if (i < n) out[i] = -__builtin_inff();
}

__global__ __launch_bounds__(kFillThreads) void mask_copy_kernel(const float* raw, int64_t n, const int32_t* ids,
                                                                 int64_t n_ids, float* out) {
  const int64_t k = (int64_t)blockIdx.x * kFillThreads + threadIdx.x;
  if (k >= n_ids) return;
  const int32_t id = ids[k];
  if (id >= 0 && id < n) out[id] = raw[id];
}

}  // namespace

void launch_mask_logits(const float* raw, int64_t n, const int32_t* ids, int64_t n_ids, float* out, hipStream_t s) {
  if (n > 0) {
    hipLaunchKernelGGL(mask_fill_kernel, dim3((unsigned)((n + kFillThreads - 1) / kFillThreads)), dim3(kFillThreads),
                       0, s, out, n);
  }
  if (n > 0 && n_ids > 0) {
    hipLaunchKernelGGL(mask_copy_kernel, dim3((unsigned)((n_ids + kFillThreads - 1) / kFillThreads)),
                       dim3(kFillThreads), 0, s, raw, n, ids, n_ids, out);
  }
}

// share: of the vocabulary, by first byte, that the requested states take on
// average. The walk of every token is the faster kernel for few states and
// where first bytes rule out little; its line depends on whether its table is
// in LDS (1.2 times the speed, up to 96 states, and a loss past about 200000
// tokens, where the 48 KiB cost resident waves). Whole calls in us, walk |
// by first bytes: 32000 tokens, 8 states, share 0.3: 25 | 30 for 8 requested,
// 67 | 64 for 64; share 0.8: 105 | 169 for 64. 262144 tokens, 300 states, share
// 0.3: 29 | 29 for 8 requested, 38 | 32 for 16; for 64 requested 168 | 141 at
// share 0.8, 177 | 217 at share 1. With one state 21 | 25 on either.
void launch_masks(const int64_t* offsets, const uint8_t* bytes, int32_t vocab, const int16_t* next,
                  const int32_t* states, int32_t n, double share, uint32_t* masks, int32_t mask_words,
                  int32_t n_states, hipStream_t s) {
#define GS_MASKS(kernel, threads)                                                                               \
  hipLaunchKernelGGL(kernel, dim3((vocab + threads - 1) / threads), dim3(threads), 0, s, offsets, bytes, vocab, \
                     next, n_states, states, n, masks, mask_words)
  const bool walk_lds = n_states <= kWalkLdsStates && vocab <= kWalkLdsVocab;
  const int few = walk_lds ? 16 : (vocab > kWalkLdsVocab ? 8 : 10);
  const double most = walk_lds ? (n_states < 32 ? 0.6 : 0.66) : 0.8;
  if (n < few || share > most) {
    if (walk_lds && n >= 4) GS_MASKS(walk_masks_kernel<true>, kWalkThreads);
    else GS_MASKS(walk_masks_kernel<false>, kWalkThreads);
  } else if (n_states <= kLdsStates) {
    GS_MASKS(build_masks_kernel<true>, kMaskThreads);
  } else {
    GS_MASKS(build_masks_kernel<false>, kMaskThreads);
  }
#undef GS_MASKS
}

template <typename In>
static void launch_logprob_as(const In* logits, int32_t rows, int64_t stride, int32_t vocab, const int32_t* tokens,
                              double* out, void* partial, int32_t cu_count, hipStream_t s) {
  // Parts per row: a power of two that keeps about 8 workgroups per compute
  // unit (more than one a row only while rows leave units idle), at most 64
  // (the join's lanes) and at least one 16-byte load per thread and part. A row
  // of one turn of a workgroup's loads stays whole: the second launch costs 3 us
  // (8 rows of 4000 f32 logits 9.0 us in two parts, 5.8 whole).
  const int64_t most = std::min<int64_t>(kLogParts, 8 * (int64_t)cu_count);
  const int64_t bytes = (int64_t)vocab * (int)sizeof(In);
  int32_t parts = 1;
  while (bytes > 16 * kLogThreads * kLogVecs && parts < 64 && (int64_t)rows * parts * 2 <= most &&
         bytes >= 16 * kLogThreads * 2 * (int64_t)parts)
    parts *= 2;
  hipLaunchKernelGGL(logprob_part_kernel<In>, dim3((unsigned)(rows * parts)), dim3(kLogThreads), 0, s, logits, stride,
                     vocab, tokens, parts, (LogPart*)partial, out);
  if (parts > 1) {
    constexpr int kRows = kLogThreads / 64;
    hipLaunchKernelGGL(logprob_join_kernel<In>, dim3((unsigned)((rows + kRows - 1) / kRows)), dim3(kLogThreads), 0, s,
                       logits, stride, vocab, rows, tokens, parts, (const LogPart*)partial, out);
  }
}

size_t logprob_bytes() { return (size_t)kLogParts * sizeof(LogPart); }

void launch_logprob(const void* logits, int32_t dtype, int32_t rows, int64_t stride, int32_t vocab,
                    const int32_t* tokens, double* out, void* partial, int32_t cu_count, hipStream_t s) {
  if (dtype == GS_BF16)
    launch_logprob_as((const uint16_t*)logits, rows, stride, vocab, tokens, out, partial, cu_count, s);
  else launch_logprob_as((const float*)logits, rows, stride, vocab, tokens, out, partial, cu_count, s);
}

}  // namespace gs
