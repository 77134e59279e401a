// Typical-p over the whole vocabulary (sampling.ts:49-55 with topK 0), one
// workgroup per row and one pass of exponentials.
//
// With x = (max - l) / T, Z = sum e^-x and c = sum x e^-x / Z, the entropy is
// log Z + c and an item's surprise |-log p - entropy| is |x - c|: the typical
// set is a window around c. So nothing is sorted but the items at its edge:
// a first pass finds the range of x, a second sums Z, c and the mass of 8192
// bins of x, prefix sums of the bins bound the window's half-width, a third
// pass gathers the items of the few bins its two edges fall in, and these,
// put in order of surprise, decide the cut. The draw then falls among them or
// in one bin of the window, which a last pass gathers. All sums are binary64.
//
// A decision that the reference's own rounding could turn (its sequential
// sums move by V 2^-53 relative) is left to the exact replay: a sum within
// `margin` of its threshold, a logit other than the cut's whose surprise lies
// within the entropy's error of it, one other than the drawn whose
// probability could round either way. So are lists of more than kTypCap
// items: more equal logits than that at the cut or in the drawn bin. The bins' sums vary in their last bits with
// the order of the LDS atomics: no decision rests on those, only, within
// 1e-15 of the margin's own edge, whether the replay takes it.
//
// Bound by the exponential pass on one CU (about 30 binary64 operations a
// logit); spreading a row over workgroups would take a launch, about 5 us, for
// each of the four steps. Whole calls: 24 rows of 151643 f32 logits 113 us (125
// before the gathers skipped waves without an item by a comparison in
// binary32), 256 rows of 262144 240 us; the replays, with three sorts and five
// one-lane sums a row, took 27.3 and 29.9 ms. Probabilities are within 4e-16 of 64-bit ones (2.4e-14).
#include "gs_exact_row.h"
#include "gs_exp2.h"

namespace gs {
namespace {

constexpr int kTypThreads = kExactThreads;
constexpr int kTypWaves = kTypThreads / 64;
constexpr int kTypBins = 8192;
constexpr int kTypCap = 4096;      // items gathered at a time
constexpr double kTypSpan = 700.0; // e^-x stays far from underflow

struct TypicalLds {
  double mass[kTypBins + 1];  // bin sums, then the mass before each bin
  uint64_t k1[kTypCap], k2[kTypCap];
  double tab[kExpTable];
  double wsum[2][kTypWaves];
  uint32_t wkey[2][kTypWaves];
  uint32_t n, flag, first;
  int32_t lo, hi;
};

template <typename In>
__device__ __forceinline__ float typ_logit(In v) {
  if constexpr (sizeof(In) == 2) return __builtin_bit_cast(float, (uint32_t)v << 16);
  else return v;
}

// visit(l, id, live) over the row's logits (softcapped when cap > 0): the
// 16-byte aligned pieces, kPieces per thread in flight, and the elements
// before and after them. Every wave calls visit with all its lanes.
template <typename In, typename F>
__device__ __forceinline__ void typ_visit(const In* base, int vocab, double cap, F&& visit) {
  constexpr int kVec = 16 / (int)sizeof(In), kPieces = 4;
  const int tid = threadIdx.x;
  const int to_aligned = (int)((16u - ((uintptr_t)base & 15u)) & 15u) / (int)sizeof(In);
  const int head = to_aligned < vocab ? to_aligned : vocab;
  const int nv = (vocab - head) / kVec, tail = head + nv * kVec;
  auto one = [&](float l, int id, bool live) __attribute__((always_inline)) {
    visit(cap > 0 ? softcap_call(l, cap) : l, (uint32_t)id, live);
  };
  {
    // fewer than 2 kVec elements: the first wave's
    const int rest = head + vocab - tail;
    if (tid < 64 && rest > 0) {
      const int id = tid < head ? tid : tail + tid - head;
      const bool live = tid < rest;
      one(typ_logit<In>(base[live ? id : 0]), id, live);
    }
  }
  const uint4* vecs = (const uint4*)(base + head);
  for (int v0 = 0; v0 < nv; v0 += kTypThreads * kPieces) {
    uint4 w[kPieces];
#pragma unroll
    for (int i = 0; i < kPieces; ++i) {
      const int q = v0 + tid + i * kTypThreads;
      w[i] = vecs[q < nv ? q : nv - 1];
    }
#pragma unroll
    for (int i = 0; i < kPieces; ++i) {
      const int q = v0 + tid + i * kTypThreads;
      const uint32_t d[4] = {w[i].x, w[i].y, w[i].z, w[i].w};
#pragma unroll
      for (int j = 0; j < kVec; ++j) {
        uint32_t b;
        if constexpr (sizeof(In) == 4) b = d[j];
        else b = (j & 1) ? d[j >> 1] & 0xFFFF0000u : d[j >> 1] << 16;
        one(__builtin_bit_cast(float, b), head + q * kVec + j, q < nv);
      }
    }
  }
}

__device__ __forceinline__ double typ_block_sum(TypicalLds& S, double v) {
  v = wave_sum_f64_dpp(v);
  if ((threadIdx.x & 63) == 0) S.wsum[0][threadIdx.x >> 6] = v;
  __syncthreads();
  double t = 0.0;
  for (int w = 0; w < kTypWaves; ++w) t += S.wsum[0][w];
  __syncthreads();
  return t;
}
// the sum of the threads' v before this one
__device__ __forceinline__ double typ_block_before(TypicalLds& S, double v) {
  const double incl = wave_scan_f64(v);
  const int wave = threadIdx.x >> 6;
  if ((threadIdx.x & 63) == 63) S.wsum[0][wave] = incl;
  __syncthreads();
  double t = 0.0;
  for (int w = 0; w < wave; ++w) t += S.wsum[0][w];
  __syncthreads();
  return t + incl - v;
}

// (k1, k2) ascending, n entries, the rest of the power of two filled with ones
__device__ __forceinline__ void typ_sort(TypicalLds& S, int n) {
  const int tid = threadIdx.x;
  int n2 = 1;
  while (n2 < n) n2 <<= 1;
  for (int i = n + tid; i < n2; i += kTypThreads) S.k1[i] = S.k2[i] = ~0ull;
  __syncthreads();
  for (int k = 2; k <= n2; k <<= 1) {
    for (int j = k >> 1; j > 0; j >>= 1) {
      for (int h = tid; h < n2 / 2; h += kTypThreads) {
        const int i = ((h & ~(j - 1)) << 1) | (h & (j - 1)), p = i | j;
        const uint64_t a1 = S.k1[i], b1 = S.k1[p], a2 = S.k2[i], b2 = S.k2[p];
        const bool gt = a1 > b1 || (a1 == b1 && a2 > b2);
        if (gt == ((i & k) == 0)) {
          S.k1[i] = b1; S.k1[p] = a1;
          S.k2[i] = b2; S.k2[p] = a2;
        }
      }
      __syncthreads();
    }
  }
}

// Appends (k1, k2) of the wave's lanes that pass; S.n counts all of them.
__device__ __forceinline__ void typ_append(TypicalLds& S, bool pass, uint64_t k1, uint64_t k2) {
  const uint64_t m = __ballot(pass);
  if (m == 0) return;
  const int lane = threadIdx.x & 63, leader = __builtin_ctzll(m);
  uint32_t at = 0;
  if (lane == leader) at = atomicAdd(&S.n, (uint32_t)__popcll(m));
  at = (uint32_t)__shfl((int)at, leader, 64) + (uint32_t)__popcll(m & ((1ull << lane) - 1ull));
  if (pass && at < (uint32_t)kTypCap) { S.k1[at] = k1; S.k2[at] = k2; }
}

// The row's draw; false where the exact replay decides. The whole workgroup
// calls it.
template <typename In>
__device__ __forceinline__ bool typ_settle(const SampleArgs& a, TypicalLds& S, int64_t row,
                                           const gs_row_config& cfg) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const In* base = (const In*)a.logits + row * a.row_stride;
  const int V = a.vocab;
  const double T = cfg.temperature, rT = 1.0 / T, cap = cfg.softcap;
  if (tid < kExpTable) S.tab[tid] = c_exp2_256[tid * (256 / kExpTable)];
  for (int b = tid; b < kTypBins; b += kTypThreads) S.mass[b] = 0.0;
  if (tid == 0) { S.n = 0; S.flag = 0; S.first = 0xFFFFFFFFu; S.lo = -1; S.hi = kTypBins; }

  // ---- the range of the row
  uint32_t kmax = 0, kmin = 0xFFFFFFFFu;
  typ_visit<In>(base, V, cap, [&](float l, uint32_t, bool live) {
    const uint32_t k = f32_key(l);
    kmax = live && k > kmax ? k : kmax;
    kmin = live && k < kmin ? k : kmin;
  });
  kmax = wave_max_u32(kmax);
  kmin = wave_min_u32(kmin);
  if (lane == 0) { S.wkey[0][wave] = kmax; S.wkey[1][wave] = kmin; }
  __syncthreads();
  for (int w = 0; w < kTypWaves; ++w) {
    kmax = S.wkey[0][w] > kmax ? S.wkey[0][w] : kmax;
    kmin = S.wkey[1][w] < kmin ? S.wkey[1][w] : kmin;
  }
  // (a NaN's key lies outside the infinities')
  if (!(kmin > kKeyNegInf && kmax < kKeyPosInf)) return false;
  const double vmax = div_by_temperature((double)key_f32(kmax), T, rT);
  const double span = vmax - div_by_temperature((double)key_f32(kmin), T, rT);
  if (!(span > 0 && span <= kTypSpan)) return false;
  const double per = (double)kTypBins / span;
  auto below = [&](float l) __attribute__((always_inline)) -> double {
    return vmax - div_by_temperature((double)l, T, rT);
  };
  auto bin = [&](double x) __attribute__((always_inline)) -> int {
    const int b = (int)(x * per);
    return b < kTypBins ? b : kTypBins - 1;
  };

  // ---- Z, the mean of x and the bins' masses
  double z = 0.0, s1 = 0.0;
  typ_visit<In>(base, V, cap, [&](float l, uint32_t, bool live) {
    if (!live) return;
    const double x = below(l), e = exp_neg(-x, S.tab);
    z += e;
    s1 = __builtin_fma(x, e, s1);
    unsafeAtomicAdd(&S.mass[bin(x)], e);
  });
  z = typ_block_sum(S, z);
  const double c = typ_block_sum(S, s1) / z;
  {
    constexpr int kPer = kTypBins / kTypThreads;
    double m[kPer], sum = 0.0;
#pragma unroll
    for (int k = 0; k < kPer; ++k) { m[k] = S.mass[tid * kPer + k]; sum += m[k]; }
    double at = typ_block_before(S, sum);
#pragma unroll
    for (int k = 0; k < kPer; ++k) { S.mass[tid * kPer + k] = at; at += m[k]; }
    if (tid == kTypThreads - 1) S.mass[kTypBins] = at;
  }
  __syncthreads();

  // ---- half-widths in bins: at `lo` the bins the window touches hold less
  // than the threshold, at `hi` the bins inside it hold it
  const double target = cfg.typical_p * z;
  const double cb = c * per;
  auto clamp_bin = [&](double b) __attribute__((always_inline)) -> int {
    return b <= 0 ? 0 : (b >= (double)kTypBins ? kTypBins : (int)b);
  };
  {
    int lo = -1, hi = kTypBins;
    for (int k = tid; k < kTypBins; k += kTypThreads) {
      const double touched = S.mass[clamp_bin(__builtin_ceil(cb + k))] - S.mass[clamp_bin(__builtin_floor(cb - k))];
      if (touched <= target * (1.0 - 1.0e-9) && k > lo) lo = k;
      const int i0 = clamp_bin(__builtin_ceil(cb - k)), i1 = clamp_bin(__builtin_floor(cb + k));
      const double inside = i1 > i0 ? S.mass[i1] - S.mass[i0] : 0.0;
      if (inside >= target * (1.0 + 1.0e-9) && k < hi) hi = k;
    }
    if (lo >= 0) atomicMax(&S.lo, lo);
    if (hi < kTypBins) atomicMin(&S.hi, hi);
  }
  __syncthreads();
  const int w_lo = S.lo, w_hi = S.hi;
  if (w_hi >= kTypBins) return false;
  const int o0 = clamp_bin(__builtin_floor(cb - w_hi)), o1 = clamp_bin(__builtin_ceil(cb + w_hi));
  int i0 = clamp_bin(__builtin_ceil(cb - w_lo)), i1 = clamp_bin(__builtin_floor(cb + w_lo));
  if (w_lo < 0 || i1 <= i0) i0 = i1 = o0;  // no bin surely inside
  const double inner = S.mass[i1] - S.mass[i0];

  // the logits whose bin can be b0 .. b1 - 1, widened by more than rounding
  // the bounds moves them (or narrowed, by < 0)
  auto logits_of = [&](int b0, int b1, double by, float* lo, float* hi) __attribute__((always_inline)) {
    const double h = (vmax - b0 / per) * T, w = (vmax - b1 / per) * T;
    *hi = b0 <= 0 ? __builtin_inff() : (float)(h + by * (1.0 + fabs(h)));
    *lo = b1 >= kTypBins ? -__builtin_inff() : (float)(w - by * (1.0 + fabs(w)));
  };
  float l_lo, l_hi, in_lo, in_hi;
  logits_of(o0, o1, 1.0e-6, &l_lo, &l_hi);
  logits_of(i0, i1, -1.0e-6, &in_lo, &in_hi);
  if (i1 <= i0) in_hi = -__builtin_inff();  // none

  // ---- the items between the two, in order of surprise
  typ_visit<In>(base, V, cap, [&](float l, uint32_t id, bool live) {
    // most waves hold none of the few bins' items
    if (__ballot(live && l >= l_lo && l <= l_hi && !(l > in_lo && l < in_hi)) == 0) return;
    const double x = below(l);
    const int b = live ? bin(x) : -1;
    const bool pass = b >= o0 && b < o1 && !(b >= i0 && b < i1);
    // (the key joins the zeros: equal values are in order of id alone)
    typ_append(S, pass, gsm::bits_of(fabs(x - c)), ((uint64_t)f32_key(l) << 32) | id);
  });
  __syncthreads();
  int n = (int)S.n;
  if (n > kTypCap || n < 1) return false;
  typ_sort(S, n);

  constexpr int kOwn = kTypCap / kTypThreads;
  const double margin = z * fmax(kNearTie, 4.0 * V * 0x1p-53);
  auto logit_of = [&](uint64_t k2) __attribute__((always_inline)) -> float {
    return key_f32((uint32_t)(k2 >> 32));
  };
  // the first entry whose running sum from `from` reaches `want`, -1 when a
  // sum lies within the margin of it; in every thread, with the sum there
  auto reach = [&](double from, double want, bool by_value, double* sum_at) __attribute__((always_inline)) -> int {
    double e[kOwn], own = 0.0;
#pragma unroll
    for (int k = 0; k < kOwn; ++k) {
      const int i = tid * kOwn + k;
      e[k] = 0.0;
      if (i < n) e[k] = exp_neg(-below(by_value ? key_f32(~(uint32_t)S.k1[i]) : logit_of(S.k2[i])), S.tab);
      own += e[k];
    }
    if (tid == 0) { S.flag = fabs(from - want) <= margin ? 1u : 0u; S.first = 0xFFFFFFFFu; }
    double sum = from + typ_block_before(S, own);
    uint32_t first = 0xFFFFFFFFu;
    bool near = false;
    double at = 0.0;
#pragma unroll
    for (int k = 0; k < kOwn; ++k) {
      const int i = tid * kOwn + k;
      sum += e[k];
      if (i >= n) continue;
      near |= fabs(sum - want) <= margin;
      if (sum >= want && first == 0xFFFFFFFFu) { first = (uint32_t)i; at = sum; }
    }
    if (near) atomicOr(&S.flag, 1u);
    if (first != 0xFFFFFFFFu) atomicMin(&S.first, first);
    __syncthreads();
    if (first != 0xFFFFFFFFu && first == S.first) S.wsum[1][0] = at;
    __syncthreads();
    *sum_at = S.wsum[1][0];
    const int r = S.flag != 0 || S.first == 0xFFFFFFFFu ? -1 : (int)S.first;
    __syncthreads();
    return r;
  };
  double kept = 0.0;
  const int cut = reach(inner, target, false, &kept);
  if (cut < 0) return false;
  // whether v holds in some thread (S.flag is 0: the reach before found its entry)
  auto in_any = [&](bool v) __attribute__((always_inline)) -> bool {
    if (__ballot(v) != 0 && lane == 0) atomicOr(&S.flag, 1u);
    __syncthreads();
    const bool r = S.flag != 0;
    __syncthreads();
    return r;
  };
  {
    // the reference's surprises differ from these by the entropy's error: no
    // other logit of the list within it (however many equal ones lie between),
    // and none of the items before and after the list, which lie within lo or
    // past hi
    const double err = 2.0 * (4.0 * V * 0x1p-53 * (gsm::js_log(z) + c + 2.0) + 1.0e-12);
    const double s = gsm::double_of(S.k1[cut]), slack = err + 1.0e-6 / per;
    const uint32_t key = (uint32_t)(S.k2[cut] >> 32);
    bool near = false;
#pragma unroll
    for (int k = 0; k < kOwn; ++k) {
      const int i = tid * kOwn + k;
      near |= i < n && (uint32_t)(S.k2[i] >> 32) != key && fabs(gsm::double_of(S.k1[i]) - s) < err;
    }
    if (in_any(near) || (w_lo >= 0 && s - w_lo / per < slack) || w_hi / per - s < slack) return false;
  }

  // ---- the draw (sampling.ts:58-64): by falling probability the kept items
  // above the window's sure bins, these bins, the kept items below them
  uint64_t own1[kOwn], own2[kOwn];
  double above = 0.0;
#pragma unroll
  for (int k = 0; k < kOwn; ++k) {
    const int i = tid * kOwn + k;
    own1[k] = own2[k] = 0;
    if (i > cut) continue;
    const float l = logit_of(S.k2[i]);
    const double x = below(l);
    own1[k] = (uint32_t)~f32_key(l);
    own2[k] = 1ull << 63 | (uint64_t)(x < c ? 1u : 0u) << 62 | (uint32_t)S.k2[i];
    if (x < c) above += exp_neg(-x, S.tab);
  }
  above = typ_block_sum(S, above);
  const double u = cfg.rng_mode == GS_RNG_EXPLICIT ? cfg.uniform : gsm::mulberry32_draw(cfg.seed, cfg.draw_index);
  const double cursor = u * kept;
  double from = 0.0;
  int in_bin = -1;
  bool upper = true, lower = true;  // the kept items the draw may fall on
  if (i1 > i0) {
    if (cursor <= above) {
      lower = false;
    } else if (cursor > above + inner) {
      upper = false;
      from = above + inner;
    } else {
      upper = lower = false;
      int b0 = i0, b1 = i1 - 1;  // the last bin with less mass before it than the cursor
      while (b0 < b1) {
        const int mid = (b0 + b1 + 1) >> 1;
        if (above + (S.mass[mid] - S.mass[i0]) < cursor) b0 = mid;
        else b1 = mid - 1;
      }
      in_bin = b0;
      from = above + (S.mass[in_bin] - S.mass[i0]);
    }
  }
  if (tid == 0) S.n = 0;
  __syncthreads();
  if (in_bin >= 0) {
    logits_of(in_bin, in_bin + 1, 1.0e-6, &l_lo, &l_hi);
    typ_visit<In>(base, V, cap, [&](float l, uint32_t id, bool live) {
      if (__ballot(live && l >= l_lo && l <= l_hi) == 0) return;
      typ_append(S, live && bin(below(l)) == in_bin, (uint32_t)~f32_key(l), id);
    });
  } else {
#pragma unroll
    for (int k = 0; k < kOwn; ++k) {
      const bool high = (own2[k] >> 62 & 1u) != 0;
      typ_append(S, (own2[k] >> 63) != 0 && (high ? upper : lower), own1[k], (uint32_t)own2[k]);
    }
  }
  __syncthreads();
  n = (int)S.n;
  if (n > kTypCap || n < 1) return false;
  typ_sort(S, n);
  double unused;
  const int hit = reach(from, cursor, true, &unused);
  if (hit < 0) return false;
  const float l = key_f32(~(uint32_t)S.k1[hit]);
  const double x = below(l);
  {
    // no other logit whose probability could round out of order: in the list
    // (however many equal ones, in order of id, lie between), and, where the
    // run of equal ones reaches the list's end, in the window's next bin past
    // it. A bin there that moves no prefix sum is empty, or its items lie
    // below the margin's resolution, where no draw settles.
    const uint64_t key = S.k1[hit];
    bool near = false;
#pragma unroll
    for (int k = 0; k < kOwn; ++k) {
      const int i = tid * kOwn + k;
      near |= i < n && S.k1[i] != key && fabs(below(key_f32(~(uint32_t)S.k1[i])) - x) <= 1.0e-12;
    }
    if (in_any(near)) return false;
    const int b0 = in_bin >= 0 ? in_bin : (!upper ? i1 : 0);             // bins below b0 precede the list,
    const int b1 = in_bin >= 0 ? in_bin + 1 : (!lower ? i0 : kTypBins);  // bins from b1 on follow it
    const double edge = fmax(1.0e-6, 1.0e-12 * per);
    const bool before = S.k1[0] != key || b0 == 0 || x * per - b0 > edge || S.mass[b0] == S.mass[b0 - 1];
    const bool after = S.k1[n - 1] != key || b1 == kTypBins || b1 - x * per > edge || S.mass[b1 + 1] == S.mass[b1];
    if (!before || !after) return false;
  }
  if (tid == 0) {
    a.results[row].token = (int32_t)(uint32_t)S.k2[hit];
    a.results[row].flags = 0;
    a.results[row].probability = exp_neg(-x, S.tab) / z;
  }
  return true;
}

union TypicalKernelLds {
  TypicalLds typ;
  exact::Lds ex;
};

template <typename In>
__global__ __launch_bounds__(kTypThreads) void typical_kernel(SampleArgs) {
  __shared__ TypicalKernelLds U;
  const SampleArgs& a = *(const SampleArgs*)__builtin_amdgcn_kernarg_segment_ptr();
  const int64_t row = blockIdx.x;
  const gs_row_config cfg = a.configs[row];
  if (!typical_row(a, row, cfg)) return;  // the finish's
  if (typ_settle<In>(a, U.typ, row, cfg)) return;
  __syncthreads();
  if (row < a.exact_slots) {
    exact::process_row(a, U.ex, exact::scratch_at(a, row), row, 0u);
  } else if (threadIdx.x == 0) {
    const uint32_t q = atomicAdd(&a.queue->count, 1u);
    a.queue->rows[q] = (uint32_t)row;
    a.results[row].flags = 0;
  }
}

}  // namespace

void launch_typical(const SampleArgs& a, hipStream_t s, LaunchEvents ev) {
  const dim3 grid(a.rows), block(kTypThreads);
  if (a.dtype == GS_BF16) hipExtLaunchKernelGGL(typical_kernel<uint16_t>, grid, block, 0, s, ev.start, ev.stop, 0, a);
  else hipExtLaunchKernelGGL(typical_kernel<float>, grid, block, 0, s, ev.start, ev.stop, 0, a);
}

}  // namespace gs
