// Device-side token choice: sample_token of src/nn/sampling.rs:3-81 for a
// batch of rows, one 1024-thread block per row.
//
// The reference copies the logits, applies the repetition penalty to every
// distinct seen id, and then either takes the argmax (temperature <= 0) or
// sorts all ids by logit (descending), keeps the top_k, turns them into f64
// probabilities exp((l - max) / T) / sum, keeps the smallest prefix whose
// cumulative probability reaches top_p (renormalised), and walks the prefix
// with r = rand::random() until r < p.
//
// On the general path nothing is sorted.  Every cut the reference makes
// along the sorted order -- the k-th element, the top_p crossing, the
// element where the walk stops -- is found by a radix select over 32-bit
// order-preserving keys of the penalised logits: three histogram passes
// (11, 11 and 10 bits) narrow the key, counting elements (top_k) or summing
// their f64 weights (top_p, the walk), and the elements that share the
// final key are resolved in index order (the
// reference's unstable sort leaves that order unspecified; lower index first
// is this implementation's choice).  The per-element weights live in a
// scratch row; the repetition penalty is applied on the fly through a bitmap
// of the seen ids in LDS.
//
// Rows of at least kHistMin ids skip that: a first kernel spreads each row
// over several blocks, which bin their part's logits on the row's grid (2047
// bins below the part's maximum) and sum each bin's f64 weights, or count its
// elements where 0 < top_k <= 1024.  The row's block adds the parts' bins,
// finds the bins in which the cuts fall, gathers their members (a few hundred
// ids), puts them in order by counting the entries above each, and cuts
// exactly there.  With top_k that list is the top_k, which then goes through
// the reference's own sequence: f64 probabilities summed in order, the top_p
// prefix, the walk r -= p.  NaN, an infinite maximum, cuts below the bins and
// bins of too many ids (ties) are left to the other paths.
// Shorter rows, and those the bins leave, with 0 < top_k <= 1024: a cut on d = max
// - l admitting between top_k and 2048 elements is found by counting against 16
// thresholds per pass (powers of four, then 16-way refinements); where that
// fails too, the radix path.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <mutex>

#include "common.h"
#include "kernels.h"

namespace akh {

namespace {

#ifndef AKH_SAMPLE_NT
#define AKH_SAMPLE_NT 1024
#endif
#ifndef AKH_SAMPLE_BLOCKS
#define AKH_SAMPLE_BLOCKS 256
#endif
constexpr int NT = AKH_SAMPLE_NT;  // threads per row (per part of a binned row)
constexpr int NW = NT / 64;     // waves per block

// Radix digits of the order keys: 11, 11 and 10 bits (three passes).
constexpr int kBins = 2048;
constexpr int kPartsMax = 16;  // of a binned row (below)
struct PartHead {
  float max;
  float scale;   // of the row's grid; 0: NaN or an infinite maximum in the part
  double total;  // of the part's weights (or its count)
};
struct RowHist {
  double before[kBins];  // weight (or count) of the bins above
  PartHead head[kPartsMax];
  double part_f[kPartsMax];
  uint32_t first[2];     // list position of a run's first entry
  double target;
};
// A block's LDS also holds the seen-id bitmap (an eighth of a byte per id), so
// what never lives together shares its place: a binned row's totals and the
// radix path's bins here, the list before and after its sort in TopKShared.
// Together 58.7 KB: vocabularies of up to 840 thousand ids with a penalty.
struct SampleShared {
  union {
    struct {
      // One radix pass's bins: counts or f64 weight sums (a select uses one).
      union {
        uint32_t hist_n[kBins];
        double hist_w[kBins];
      };
      // The last pass's bins (kBins / 2): members of nonzero weight, lowest index.
      uint32_t last_n[kBins / 2];
      uint32_t last_i[kBins / 2];
    };
    RowHist rh;
  };
  double wave_d[NW];
  uint32_t wave_u[NW];
  float wave_f[NW];
  uint32_t bcast_u[4];
  double bcast_d[2];
};

__device__ __forceinline__ uint32_t order_key(float f) {
  const uint32_t u = __float_as_uint(f);
  return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}

// Penalised logit (sampling.rs:3-16): every distinct seen id once.
__device__ __forceinline__ float pen_logit(const float* row, int i, const uint32_t* bm,
                                           float penalty) {
  float l = row[i];
  if (bm && (bm[i >> 5] >> (i & 31) & 1u)) l = l > 0.0f ? __fdiv_rn(l, penalty) : __fmul_rn(l, penalty);
  return l;
}

__device__ __forceinline__ double block_sum_d(double v, SampleShared& sh) {
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  const int w = threadIdx.x >> 6;
  __syncthreads();
  if ((threadIdx.x & 63) == 0) sh.wave_d[w] = v;
  __syncthreads();
  double t = 0.0;
  for (int k = 0; k < NW; ++k) t += sh.wave_d[k];
  return t;
}

__device__ __forceinline__ uint32_t block_sum_u(uint32_t v, SampleShared& sh) {
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  const int w = threadIdx.x >> 6;
  __syncthreads();
  if ((threadIdx.x & 63) == 0) sh.wave_u[w] = v;
  __syncthreads();
  uint32_t t = 0;
  for (int k = 0; k < NW; ++k) t += sh.wave_u[k];
  return t;
}

__device__ __forceinline__ uint32_t block_min_u(uint32_t v, SampleShared& sh) {
  for (int o = 32; o > 0; o >>= 1) v = min(v, (uint32_t)__shfl_xor(v, o, 64));
  const int w = threadIdx.x >> 6;
  __syncthreads();
  if ((threadIdx.x & 63) == 0) sh.wave_u[w] = v;
  __syncthreads();
  uint32_t t = 0xFFFFFFFFu;
  for (int k = 0; k < NW; ++k) t = min(t, sh.wave_u[k]);
  return t;
}

// The value of the block's first thread that has one (0xFFFFFFFF: none).
__device__ __forceinline__ uint32_t block_first_u(uint32_t v, SampleShared& sh) {
  const unsigned long long has = __ballot(v != 0xFFFFFFFFu);
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int lead = has ? __ffsll((long long)has) - 1 : 0;
  __syncthreads();
  if (lane == lead) sh.wave_u[w] = v;
  __syncthreads();
  uint32_t t = 0xFFFFFFFFu;
#pragma unroll
  for (int k = NW - 1; k >= 0; --k) t = sh.wave_u[k] != 0xFFFFFFFFu ? sh.wave_u[k] : t;
  return t;
}

__device__ __forceinline__ float block_max_f(float v, SampleShared& sh) {
  v = wave_max(v);
  const int w = threadIdx.x >> 6;
  __syncthreads();
  if ((threadIdx.x & 63) == 0) sh.wave_f[w] = v;
  __syncthreads();
  float t = -INFINITY;
  for (int k = 0; k < NW; ++k) t = fmaxf(t, sh.wave_f[k]);
  return t;
}

// Exclusive prefix sum over the block in thread order (0 for thread 0).
template <typename T>
__device__ T block_scan_excl(T v, T* wave_tot) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  for (int o = 1; o < 64; o <<= 1) {
    const T u = __shfl_up(v, o, 64);
    if (lane >= o) v += u;
  }
  T ex = __shfl_up(v, 1, 64);
  if (lane == 0) ex = 0;
  __syncthreads();
  if (lane == 63) wave_tot[w] = v;
  __syncthreads();
  T off = 0;
  for (int k = 0; k < w; ++k) off += wave_tot[k];
  return ex + off;
}

// The element of the descending order at which a cumulative quantity
// crosses `target`: counts of elements (weights == nullptr, crossing when
// the count reaches target) or sums of weights[i] (crossing at >= target if
// inclusive, > target otherwise).  Returns the index, or n if the total
// never crosses.  `key_of(i)` gives element i's order key.
template <typename KeyFn>
__device__ __forceinline__ uint32_t select_desc(int n, KeyFn key_of, const double* weights,
                                                double target, bool inclusive,
                                                SampleShared& sh) {
  uint32_t prefix = 0, mask = 0;
  for (int pass = 0; pass < 3; ++pass) {
    const int shift = pass == 0 ? 21 : pass == 1 ? 10 : 0;
    const int nb = pass < 2 ? kBins : kBins / 2;
    for (int b = threadIdx.x; b < kBins; b += NT) {
      if (weights) sh.hist_w[b] = 0.0;
      else sh.hist_n[b] = 0u;
      if (pass == 2 && b < kBins / 2) {
        sh.last_n[b] = 0u;
        sh.last_i[b] = 0xFFFFFFFFu;
      }
    }
    __syncthreads();
    for (int i = threadIdx.x; i < n; i += NT) {
      const uint32_t k = key_of(i);
      if ((k & mask) == prefix) {
        const int bin = (k >> shift) & (nb - 1);
        const double w = weights ? weights[i] : 1.0;
        if (weights) {
          if (w != 0.0) atomicAdd(&sh.hist_w[bin], w);
        } else {
          atomicAdd(&sh.hist_n[bin], 1u);
        }
        if (pass == 2 && w != 0.0) {
          atomicAdd(&sh.last_n[bin], 1u);
          atomicMin(&sh.last_i[bin], (uint32_t)i);
        }
      }
    }
    __syncthreads();
    // The first bin in descending order whose cumulative total crosses
    // target: thread t holds bins nb - 1 - 2t and nb - 2 - 2t, one block scan
    // gives the total before them, and the lowest crossing thread wins.
    const int t = threadIdx.x, b1 = nb - 1 - 2 * t, b0 = b1 - 1;
    auto val = [&](int b) {
      return b < 0 ? 0.0 : weights ? sh.hist_w[b] : (double)sh.hist_n[b];
    };
    const double v1 = val(b1), v0 = val(b0);
    const double before = block_scan_excl<double>(v1 + v0, sh.wave_d);
    auto crosses = [&](double nxt) {
      return weights ? (inclusive ? nxt >= target : nxt > target) : nxt >= target;
    };
    const double n1 = before + v1;
    const int mine = b1 < 0 ? -1 : crosses(n1) ? b1 : (b0 >= 0 && crosses(n1 + v0)) ? b0 : -1;
    const uint32_t win = block_min_u(mine >= 0 ? (uint32_t)t : 0xFFFFFFFFu, sh);
    if (win == 0xFFFFFFFFu) return (uint32_t)n;
    if ((uint32_t)t == win) {
      sh.bcast_u[0] = (uint32_t)mine;
      sh.bcast_d[0] = target - (mine == b1 ? before : n1);
    }
    __syncthreads();
    const uint32_t sel = sh.bcast_u[0];
    prefix |= sel << shift;
    mask |= (uint32_t)(nb - 1) << shift;
    target = sh.bcast_d[0];
    // One member of nonzero weight with the final key (distinct logits):
    // the crossing is in its bin, so it is the answer.
    const bool only = pass == 2 && sh.last_n[sel] == 1u;
    const uint32_t at = only ? sh.last_i[sel] : 0u;
    __syncthreads();
    if (only) return at;
  }
  // Elements with the final key, in index order: each thread sums its
  // members over a contiguous run of the row, one block scan gives every run
  // the total before it, and each thread walks its run again from there
  // (two barriers, where 1024-element chunks of the row took three block
  // reductions each).
  const int run = (n + NT - 1) / NT;
  const int i0 = min(n, (int)threadIdx.x * run), i1 = min(n, i0 + run);
  double own = 0.0;
  for (int i = i0; i < i1; ++i)
    if (key_of(i) == prefix) own += weights ? weights[i] : 1.0;
  double incl = block_scan_excl<double>(own, sh.wave_d);
  uint32_t first = 0xFFFFFFFFu;
  for (int i = i0; i < i1; ++i) {
    if (key_of(i) != prefix) continue;
    const double v = weights ? weights[i] : 1.0;
    if (v == 0.0) continue;
    incl += v;
    if (weights ? (inclusive ? incl >= target : incl > target) : incl >= target) {
      first = (uint32_t)i;
      break;
    }
  }
  first = block_min_u(first, sh);
  return first == 0xFFFFFFFFu ? (uint32_t)n : first;
}

constexpr int KCAP = 1024;  // largest top_k of the candidate path
constexpr int CCAP = 2048;  // candidates gathered for the sort
constexpr int NTH = 16;     // thresholds counted per pass

struct TopKShared {
  union {
    unsigned long long comp[CCAP];  // key << 32 | ~index: descending = the order
    double pre[CCAP];               // once sorted: weight of the entries before each
  };
  union {
    struct {
      unsigned long long top[KCAP];  // the first entries of that order
      double prob[KCAP];
    };
    unsigned long long sorted[CCAP];  // all of them
  };
  double norm;
  int keep;
  uint32_t wcnt[NW][NTH];
  uint32_t cnt[NTH];
  uint32_t n_cand;
  uint32_t pick;
};

// The float whose order_key is k.
__device__ __forceinline__ float key_value(uint32_t k) {
  return __uint_as_float((k & 0x80000000u) ? (k & 0x7FFFFFFFu) : ~k);
}

// tk.top[0 .. min(nc, K)) = the first entries of tk.comp[0 .. nc) in
// descending order (nc <= CCAP, K <= KCAP).  The entries are distinct (each
// holds its element's index), so an entry's place is the number of entries
// above it: every thread counts for its own entries, reading the others as
// LDS broadcasts, with no barrier in between.
__device__ __forceinline__ int rank_top(int nc, int K, TopKShared& tk) {
  for (int e = threadIdx.x; e < nc; e += NT) {
    const unsigned long long x = tk.comp[e];
    int above = 0;
#pragma unroll 8
    for (int f = 0; f < nc; ++f) above += tk.comp[f] > x ? 1 : 0;
    if (above < K) tk.top[above] = x;
  }
  __syncthreads();
  return min(nc, K);
}

// The same for every entry, into tk.sorted.
__device__ __forceinline__ void rank_all(int nc, TopKShared& tk) {
  for (int e = threadIdx.x; e < nc; e += NT) {
    const unsigned long long x = tk.comp[e];
    int above = 0;
#pragma unroll 8
    for (int f = 0; f < nc; ++f) above += tk.comp[f] > x ? 1 : 0;
    tk.sorted[above] = x;
  }
  __syncthreads();
}

// sampling.rs:45-80 over tk.top[0 .. top_k) in the reference's order: f64
// probabilities, their sum folded in order (one thread), each divided by it,
// the top_p prefix by the in-order running sum, its sum folded in order and
// divided out, and the walk r -= p.  The divisions, independent per element,
// run in parallel; the folds and the walk, whose order fixes the bits, on one
// thread.
//
// Up to 64 entries stay in the first wave: lane t holds entry t and the folds
// read the lanes in order (the same operations in the same order, without an
// LDS round trip per step).
__device__ __forceinline__ uint32_t tail_topk_wave(int K, float temperature, float top_p, double r,
                                                   TopKShared& tk) {
  if (threadIdx.x < 64) {
    const int lane = threadIdx.x;
    const unsigned long long mine = tk.top[min(lane, K - 1)];
    auto at = [](double v, int t) {
      const unsigned long long u = __double_as_longlong(v);
      return __longlong_as_double(
          ((unsigned long long)(uint32_t)__builtin_amdgcn_readlane((int)(u >> 32), t) << 32) |
          (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)u, t));
    };
    const double mxd = (double)key_value((uint32_t)(tk.top[0] >> 32));
    double p = exp(((double)key_value((uint32_t)(mine >> 32)) - mxd) / (double)temperature);
    double sum = 0.0;
    for (int t = 0; t < K; ++t) sum += at(p, t);
    p /= sum;
    int len = K;
    if (top_p < 1.0f) {
      double cum = 0.0;
      for (int t = 0; t < K; ++t) {
        cum += at(p, t);
        if (cum >= (double)top_p) {
          len = t + 1;
          break;
        }
      }
      double s2 = 0.0;
      for (int t = 0; t < len; ++t) s2 += at(p, t);
      p /= s2;
    }
    int k = len - 1;
    double rr = r;
    for (int t = 0; t < len; ++t) {
      const double pt = at(p, t);
      if (rr < pt) {
        k = t;
        break;
      }
      rr -= pt;
    }
    if (lane == 0) tk.pick = 0xFFFFFFFFu - (uint32_t)(tk.top[k] & 0xFFFFFFFFull);
  }
  __syncthreads();
  return tk.pick;
}

__device__ __forceinline__ uint32_t tail_topk(uint32_t top_k, float temperature, float top_p,
                                              double r, TopKShared& tk) {
  const int K = (int)top_k;
  if (K <= 64) return tail_topk_wave(K, temperature, top_p, r, tk);
  const double mxd = (double)key_value((uint32_t)(tk.top[0] >> 32));
  for (int t = threadIdx.x; t < K; t += NT)
    tk.prob[t] = exp(((double)key_value((uint32_t)(tk.top[t] >> 32)) - mxd) / (double)temperature);
  __syncthreads();
  if (threadIdx.x == 0) {
    double sum = 0.0;
    for (int t = 0; t < K; ++t) sum += tk.prob[t];
    tk.norm = sum;
  }
  __syncthreads();
  const double sum = tk.norm;
  for (int t = threadIdx.x; t < K; t += NT) tk.prob[t] /= sum;
  __syncthreads();
  int len = K;
  if (top_p < 1.0f) {
    if (threadIdx.x == 0) {
      double cum = 0.0;
      int keep = K;
      for (int t = 0; t < K; ++t) {
        cum += tk.prob[t];
        if (cum >= (double)top_p) {
          keep = t + 1;
          break;
        }
      }
      double s2 = 0.0;
      for (int t = 0; t < keep; ++t) s2 += tk.prob[t];
      tk.keep = keep;
      tk.norm = s2;
    }
    __syncthreads();
    len = tk.keep;
    const double s2 = tk.norm;
    for (int t = threadIdx.x; t < len; t += NT) tk.prob[t] /= s2;
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    auto idx_of = [&](int t) { return 0xFFFFFFFFu - (uint32_t)(tk.top[t] & 0xFFFFFFFFull); };
    uint32_t pk = idx_of(len - 1);
    double rr = r;
    for (int t = 0; t < len; ++t) {
      if (rr < tk.prob[t]) {
        pk = idx_of(t);
        break;
      }
      rr -= tk.prob[t];
    }
    tk.pick = pk;
  }
  __syncthreads();
  return tk.pick;
}

// Calls f(l, i, live) for every index of the row in chunks of U elements per
// thread, the chunk's loads issued before any is used; every thread makes
// the same number of calls (live = i < n), so f may use wave-wide votes.
constexpr int U = 8;
template <typename LFn, typename F>
__device__ __forceinline__ void for_row(int n, LFn l_of, F f) {
  for (int c0 = 0; c0 < n; c0 += NT * U) {
    float v[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int i = c0 + u * NT + (int)threadIdx.x;
      v[u] = i < n ? l_of(i) : -INFINITY;
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int i = c0 + u * NT + (int)threadIdx.x;
      f(v[u], i, i < n);
    }
  }
}

// Block sums of per-thread counts c[j] (plus base) -> tk.cnt.
__device__ void reduce_counts(const uint32_t (&c)[NTH], uint32_t base, TopKShared& tk) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
#pragma unroll
  for (int j = 0; j < NTH; ++j) {
    uint32_t x = c[j];
    for (int o = 32; o > 0; o >>= 1) x += __shfl_xor(x, o, 64);
    if (lane == 0) tk.wcnt[w][j] = x;
  }
  __syncthreads();
  if (threadIdx.x < NTH) {
    uint32_t t = base;
    for (int k = 0; k < NW; ++k) t += tk.wcnt[k][threadIdx.x];
    tk.cnt[threadIdx.x] = t;
  }
  __syncthreads();
}

// The smallest float whose grid cell is at least `cell` (floor(l * scale),
// which grows with l; |cell| <= 2^30 and 2 <= scale <= 2^60, so the quotient is
// at most a few floats away and -2^-149 already lies in cell -1).
__device__ __forceinline__ float cell_low(float cell, float scale) {
  auto at_least = [&](float l) { return floorf(__fmul_rn(l, scale)) >= cell; };
  auto step = [](float l, int by) {  // the by-th float above or below l
    const uint32_t u = __float_as_uint(l);
    const int o = (u & 0x80000000u) ? -(int)(u & 0x7FFFFFFFu) : (int)u;
    const int v = o + by;
    return __uint_as_float(v < 0 ? 0x80000000u | (uint32_t)-v : (uint32_t)v);
  };
  float l = cell / scale;
  while (at_least(l)) l = step(l, -1);
  while (!at_least(l)) l = step(l, 1);
  return l;
}

// tk.comp[0 .. tk.n_cand) = the elements of src[0 .. n) in [a0, a1) or [b0, b1),
// in any order (n_cand counts those past CCAP too).  A chunk's test leaves a
// bit per id, and the few that are set are appended in a loop: a dispatch
// starts with cold instruction caches, and straight-line code for every id of
// a chunk cost more to fetch than to run (the row kernel on 32 x 50257: 25 us
// so, 21 here).  Loads past the row's end return nothing and touch no memory.  28
// ids a thread and round, us for 32 rows against 24 and 32, top_p alone: 4100 ids
// 24.6 / 24.3 / 25.0, 26000 28.2 / 29.6 / 28.5, 50257 33.5 / 34.8 / 34.2, 131072
// 70.5 / 70.8 / 69.2.
__device__ __forceinline__ void gather_ranges(const float* src, int n, float a0, float a1, float b0,
                                              float b1, TopKShared& tk) {
  constexpr int UN = 28;
  if (threadIdx.x == 0) tk.n_cand = 0;
  __syncthreads();
  const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<float*>(src), (short)0, n * 4, 0x00020000);
  for (int c0 = 0; c0 < n; c0 += NT * UN) {
    const int i0 = c0 + (int)threadIdx.x;
    float v[UN];
#pragma unroll
    for (int u = 0; u < UN; ++u)
      v[u] = __builtin_bit_cast(
          float, __builtin_amdgcn_raw_buffer_load_b32(rs, (i0 + u * NT) * 4, 0, 0));
    uint32_t hits = 0;
#pragma unroll
    for (int u = 0; u < UN; ++u)
      if ((v[u] >= a0 && v[u] < a1) || (v[u] >= b0 && v[u] < b1)) hits |= 1u << u;
    while (hits) {
      const int i = i0 + (__ffs((int)hits) - 1) * NT;
      hits &= hits - 1;
      if (i >= n) break;  // zeros past the end
      const uint32_t slot = atomicAdd(&tk.n_cand, 1u);
      if (slot < (uint32_t)CCAP)
        tk.comp[slot] = ((unsigned long long)order_key(src[i]) << 32) | (0xFFFFFFFFu - (uint32_t)i);
    }
  }
  __syncthreads();
}

// tk.comp[0 .. tk.n_cand) = the elements of the row that `take` accepts, in
// any order (n_cand counts those past CCAP too).
template <typename LFn, typename TakeFn>
__device__ __forceinline__ void gather(int n, LFn l_of, TakeFn take, TopKShared& tk) {
  if (threadIdx.x == 0) tk.n_cand = 0;
  __syncthreads();
  const int lane = threadIdx.x & 63;
  for_row(n, l_of, [&](float l, int i, bool live) {
    const bool in = live && take(l);
    const unsigned long long mask = __ballot(in);
    if (mask) {
      const int lead = __ffsll((long long)mask) - 1;
      uint32_t base = 0;
      if (lane == lead) base = atomicAdd(&tk.n_cand, (uint32_t)__popcll(mask));
      base = __shfl(base, lead, 64);
      const uint32_t slot = base + __popcll(mask & ((1ull << lane) - 1ull));
      if (in && slot < (uint32_t)CCAP)
        tk.comp[slot] = ((unsigned long long)order_key(l) << 32) | (0xFFFFFFFFu - (uint32_t)i);
    }
  });
  __syncthreads();
}

// The top_k elements of l_of(0 .. n) (0 < top_k <= KCAP) in order in tk.top,
// from at most CCAP candidates gathered to tk.comp: returns how many, or -1
// where the radix path must decide instead (NaN, an infinite maximum, fewer
// than top_k finite elements near the maximum, ties too wide to cut).  Every
// thread of the block calls it; the outcome is the same for all.  The first count bins d =
// max - l by its binary exponent (d < 2^(2j - 12) exactly when its
// exponent is below 2j - 12), four packed 8-bit counters per chunk;
// refinements compare only the elements inside the narrowed interval.
template <typename LFn>
__device__ __forceinline__ int topk_candidates(int n, LFn l_of, uint32_t top_k,
                                               SampleShared& sh, TopKShared& tk) {
  float mxv = -INFINITY;
  uint32_t nan = 0;
  for_row(n, l_of, [&](float l, int, bool) {
    if (l != l) nan = 1;
    else mxv = fmaxf(mxv, l);
  });
  const float mx = block_max_f(mxv, sh);
  if (block_sum_u(nan, sh) != 0) return -1;
  if (!isfinite(mx)) return -1;

  // Threshold t: 2^(2t - 12) in the first count, then (lo, hi] cut in NTH.
  bool linear = false;
  float lo = 0.0f, hi = 0.0f;
  auto thr = [&](int t) {
    return !linear ? ldexpf(1.0f, 2 * t - 12)
                   : (t == NTH - 1 ? hi : lo + (hi - lo) * (float)(t + 1) / NTH);
  };
  {
    uint32_t c[NTH];
#pragma unroll
    for (int j = 0; j < NTH; ++j) c[j] = 0u;
    uint32_t h[4] = {0u, 0u, 0u, 0u};  // this chunk's bins (at most U per field)
    int k = 0;
    for_row(n, l_of, [&](float l, int, bool) {
      const float d = mx - l;
      int j0 = 0;
      if (!(d < ldexpf(1.0f, -12))) j0 = ((int)((__float_as_uint(d) >> 23) & 255u) - 127 + 12) / 2 + 1;
      if (j0 < NTH) {
        const uint32_t inc = 1u << ((j0 & 3) * 8);
#pragma unroll
        for (int q = 0; q < 4; ++q) h[q] += (j0 >> 2) == q ? inc : 0u;
      }
      if (++k == U) {  // fold the chunk's bins into the cumulative counts
        uint32_t run = 0;
#pragma unroll
        for (int j = 0; j < NTH; ++j) {
          run += (h[j >> 2] >> ((j & 3) * 8)) & 255u;
          c[j] += run;
        }
        h[0] = h[1] = h[2] = h[3] = 0u;
        k = 0;
      }
    });
    reduce_counts(c, 0u, tk);
  }
  float cut = 0.0f;
  for (int round = 0; round < 4; ++round) {
    int j = 0;
    while (j < NTH && tk.cnt[j] < top_k) ++j;
    if (j == NTH) return -1;  // fewer than top_k finite elements near the max
    if (tk.cnt[j] <= (uint32_t)(round == 0 ? CCAP / 4 : CCAP)) {
      cut = thr(j);
      break;
    }
    if (round == 3) return -1;  // ties too wide to cut
    const uint32_t base = j > 0 ? tk.cnt[j - 1] : 0u;
    const float nlo = j > 0 ? thr(j - 1) : lo, nhi = thr(j);
    lo = nlo;
    hi = nhi;
    linear = true;
    float tv[NTH];
#pragma unroll
    for (int t = 0; t < NTH; ++t) tv[t] = thr(t);
    uint32_t c[NTH];
#pragma unroll
    for (int t = 0; t < NTH; ++t) c[t] = 0u;
    for_row(n, l_of, [&](float l, int, bool) {
      const float d = mx - l;
      if (!(d < lo) && d < hi) {
#pragma unroll
        for (int t = 0; t < NTH; ++t) c[t] += d < tv[t] ? 1u : 0u;
      }
    });
    __syncthreads();  // every thread has read cnt
    reduce_counts(c, base, tk);
  }

  gather(n, l_of, [&](float l) { return mx - l < cut; }, tk);
  const int nc = (int)tk.n_cand;
  if (nc > CCAP || nc < (int)top_k) return -1;
  return rank_top(nc, (int)top_k, tk);
}

// This row's seen ids (positions [lo, hi) of ids, a row of len entries).
struct SeenIds {
  const uint32_t* ids = nullptr;
  long len = 0;
  int lo = 0, hi = 0;
};

// The bitmap of a row's seen ids (null if the penalty changes nothing).  The
// ids are read from their whole row (its extent is known) while the range is
// still being loaded.
__device__ __forceinline__ const uint32_t* seen_bitmap(const SampleArgs& a, const SeenIds& s,
                                                       uint32_t* bitmap) {
  if (a.penalty == 1.0f || !s.ids) return nullptr;
  const int words = (a.n + 31) / 32;
  for (long s0 = 0; s0 < s.len; s0 += 4 * NT) {
    uint32_t v[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const long q = s0 + u * NT + threadIdx.x;
      v[u] = q < s.len ? s.ids[q] : 0u;
    }
    if (s0 == 0) {
      for (int k = threadIdx.x; k < words; k += NT) bitmap[k] = 0;
      __syncthreads();
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const long q = s0 + u * NT + threadIdx.x;
      if (q >= s.lo && q < s.hi && v[u] < (uint32_t)a.n)
        atomicOr(&bitmap[v[u] >> 5], 1u << (v[u] & 31));
    }
  }
  if (s.len <= 0) {
    for (int k = threadIdx.x; k < words; k += NT) bitmap[k] = 0;
  }
  __syncthreads();
  return bitmap;
}

// Row m's seen ids; false if the row is done (session mode).
__device__ __forceinline__ bool row_seen(const SampleArgs& a, int m, SeenIds& s) {
  if (a.tok) {
    const int dn = a.done[m], st = a.start[m], p = a.pos[m];
    if (dn) return false;
    s.ids = a.hist + (size_t)m * a.hist_stride;
    s.len = a.hist_stride;
    s.lo = st;
    s.hi = p > st ? p : st;
  } else if (a.seen) {
    s.ids = a.seen + (size_t)m * a.seen_stride;
    s.len = a.seen_stride;
    s.hi = a.seen_len ? (int)min(a.seen_len[m], (uint32_t)a.seen_stride) : 0;
  }
  return true;
}

// ---------------------------------------------------------------------------
// Binned rows.  Logit l lies in grid cell floor(l * scale); the bins of a part
// (and of the row) are the kCells cells from its maximum's down, bin d the
// cell d below.  What lies further below is only in the part's total.  The
// row's workspace holds kBins doubles per part (f64 weights relative to the
// part's maximum, or uint32 counts), then a header per part, then with a
// penalty the penalised logits, which the row's block reads instead of looking
// every id up again.
// ---------------------------------------------------------------------------
constexpr int kCells = kBins - 1;
static_assert(sizeof(PartHead) == 2 * sizeof(double), "two doubles of the row's workspace");
static_assert(sizeof(SampleShared) + sizeof(TopKShared) + 840000 / 8 <= 160 * 1024,
              "a block's LDS beside the bitmap of 840000 ids");
static_assert(kBins == 2 * NT && CCAP == 2 * NT, "two bins and two list entries per thread");
// Doubles of the workspace before the penalised logits.
__host__ __device__ constexpr long hist_doubles(int parts) { return (long)parts * (kBins + 2); }
// Shortest row: one part's bins, its header and the penalised logits (4 bytes
// an id, of the workspace's 8).
constexpr int kHistMin = 2 * (kBins + 2);

// Cells per logit.  For weights 64, or 48 per unit of l / T where that is finer
// (cells of ~150 ids at the densest of 50257 logits N(0, 2^2); 2047 cells reach 42
// T below the maximum, e^-42 of its weight, or 32), or finer still on a flat
// row, whose logits would share a few cells: 800 to the range lo .. hi of 1024 of
// the row's logits, which is about 6.5 standard deviations (32 rows x 50257 N(0,
// 0.01^2) on MI355X, us without / with: top_k 40 108 / 23, top_p alone 173 / 36).
// For counts, which no temperature enters, 800 to that range or 4 (with a mask's
// value in it, 2047 cells still reach 512): 32 rows of N(0, 20^2) with top_k 40
// 21 us, 66 on the weights' grid, whose end lies above the 40th.
// No finer than keeps hi's cell at 2^23, so that a large maximum's cells are
// exact (far below zero hi is a mask's value and says nothing of the maximum,
// beyond 2^22 a cell would be wider than a logit).  From 2 to 2^60: every float
// but 0 has a cell other than 0's, which cell_low's steps rely on.
inline float grid_base(float temperature, bool count) {
  return count ? 4.0f : fmaxf(64.0f, 48.0f / temperature);
}
__device__ __forceinline__ float grid_scale(float base, float hi, float lo) {
  float s = hi > lo ? fmaxf(base, 800.0f / (hi - lo)) : fmaxf(base, 64.0f);
  if (hi > -1e4f && hi <= 0x1p22f) s = fminf(s, 0x1p23f / fabsf(hi));
  return fminf(s, 0x1p60f);
}
__device__ __forceinline__ float grid_cell(float l, float scale) {
  return floorf(__fmul_rn(l, scale));
}

// `base_scale`: grid_base.  58 registers, so two blocks share a CU (with 86, 512 x 131072
// took 444 us with run_chat's parameters instead of 315).
__global__ __launch_bounds__(NT) void k_sample_hist(SampleArgs a, float base_scale) {
  extern __shared__ uint32_t bitmap[];
  __shared__ SampleShared sh;
  const int m = blockIdx.x, part = blockIdx.y, parts = gridDim.y;
  SeenIds seen;
  if (!row_seen(a, m, seen)) return;
  const uint32_t* bm = seen_bitmap(a, seen, bitmap);
  const bool count = a.top_k > 0 && a.top_k < a.n;
  const float* row = a.logits + (size_t)m * a.row_stride;
  const int per = (a.n + parts - 1) / parts, lo = min(a.n, part * per);
  const int len = min(a.n, lo + per) - lo;
  auto l_at = [&](int i) { return pen_logit(row, lo + i, bm, a.penalty); };
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  // The same 1024 logits of the row for each of its parts, for their grid.
  const float some = row[(long)(a.n - 64) * wave / (NW - 1) + lane];
  // A part of up to NT * U ids stays in registers between the two passes.
  float v[U];
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int i = u * NT + (int)threadIdx.x;
    v[u] = i < len ? l_at(i) : -INFINITY;
  }
  auto each = [&](auto f) {
#pragma unroll
    for (int u = 0; u < U; ++u) f(v[u]);
    for (int i = U * NT + (int)threadIdx.x; i < len; i += NT) f(l_at(i));
  };
  double* base = a.wbuf + (size_t)m * a.n;
  if (bm) {
    float* copy = reinterpret_cast<float*>(base + hist_doubles(parts)) + lo;
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int i = u * NT + (int)threadIdx.x;
      if (i < len) copy[i] = v[u];
    }
    for (int i = U * NT + (int)threadIdx.x; i < len; i += NT) copy[i] = l_at(i);
  }
  float mxv = -INFINITY;
  bool nan = false;
  each([&](float l) {
    nan = nan || l != l;
    mxv = fmaxf(mxv, l);
  });
  for (int b = threadIdx.x; b < kBins; b += NT) {
    if (count) sh.hist_n[b] = 0u;
    else sh.hist_w[b] = 0.0;
  }
  // The part's maximum, the range of `some` and whether there is a NaN.
  {
    const bool any_nan = __any(nan);
    const float x = wave_max(mxv), top = wave_max(some), neg = wave_max(-some);
    if (lane == 0) {
      sh.wave_f[wave] = x;
      reinterpret_cast<float2*>(sh.wave_d)[wave] = make_float2(top, neg);
      sh.wave_u[wave] = any_nan;
    }
  }
  __syncthreads();
  float mx = -INFINITY, hi = -INFINITY, nlo = -INFINITY;
  uint32_t nans = 0;
#pragma unroll
  for (int k = 0; k < NW; ++k) {
    const float2 r = reinterpret_cast<const float2*>(sh.wave_d)[k];
    mx = fmaxf(mx, sh.wave_f[k]);
    hi = fmaxf(hi, r.x);
    nlo = fmaxf(nlo, r.y);
    nans |= sh.wave_u[k];
  }
  const float scale = grid_scale(base_scale, hi, -nlo);
  const bool empty = mx == -INFINITY, bad = nans || mx == INFINITY;
  double own = 0.0;
  if (!bad && !empty) {
    const float cell = grid_cell(mx, scale);
    const double mxd = (double)mx, T = (double)a.temperature;
    each([&](float l) {
      const float d = cell - grid_cell(l, scale);
      const bool in = d < (float)kCells;
      if (count) {
        if (in) atomicAdd(&sh.hist_n[(int)d], 1u);
      } else if (l > -INFINITY) {
        const double w = exp(((double)l - mxd) / T);
        own += w;
        if (in) atomicAdd(&sh.hist_w[(int)d], w);
      }
    });
  }
  const double total = block_sum_d(own, sh);  // its barriers complete the bins
  if (!bad && !empty) {
    double* bins = base + (size_t)part * kBins;
    for (int b = threadIdx.x; b < kBins; b += NT) {
      if (count) reinterpret_cast<uint32_t*>(bins)[b] = sh.hist_n[b];
      else bins[b] = sh.hist_w[b];
    }
  }
  if (threadIdx.x == 0)
    reinterpret_cast<PartHead*>(base + (size_t)parts * kBins)[part] =
        PartHead{mx, bad ? 0.f : scale, total};
}

// The pick of row m from its parts' bins, or n where the radix path must
// decide.  Every thread of the block calls it.
__device__ __forceinline__ uint32_t pick_binned(const SampleArgs& a, int m, int parts,
                                                const float* src, double r, SampleShared& sh,
                                                TopKShared& tk) {
  RowHist& rh = sh.rh;
  const uint32_t none = (uint32_t)a.n;
  const int n = a.n, t = threadIdx.x;
  const bool count = a.top_k > 0 && a.top_k < n;
  const double* base = a.wbuf + (size_t)m * n;
  const PartHead* head = reinterpret_cast<const PartHead*>(base + (size_t)parts * kBins);
  if (t < parts) rh.head[t] = head[t];
  __syncthreads();
  float mx = -INFINITY, scale = INFINITY;
  for (int q = 0; q < parts; ++q) {
    mx = fmaxf(mx, rh.head[q].max);
    scale = fminf(scale, rh.head[q].scale);  // one value, or 0 of a part
  }
  if (scale == 0.f || mx == -INFINITY) return none;  // uniform
  // Cells are whole floats: every one from the row's first bin to the one past
  // its last has to be exact, or a bin's edge (cell - b below) rounds onto its
  // neighbour's and the bin's members are lost.  The one edge that a count's
  // cut takes is some logit's own cell, exact wherever cells are finite.
  const float cell = grid_cell(mx, scale);
  if (!(fabsf(cell) <= (count ? 0x1p30f : 0x1p24f - (float)(kCells + 1)))) return none;
  const double mxd = (double)mx, T = (double)a.temperature;
  if (t < parts)
    rh.part_f[t] = rh.head[t].max == -INFINITY ? 0.0 : exp(((double)rh.head[t].max - mxd) / T);
  __syncthreads();
  double total = 0.0;
  for (int q = 0; q < parts; ++q) total += rh.part_f[q] * rh.head[q].total;

  // Thread t's bins 2 t and 2 t + 1 over the parts, then every bin's total
  // above it.
  // Eight parts' loads at a time, without branches between them (a part past
  // the last, an empty one and bins outside a part read bin 0 and count 0).
  double v[2] = {0.0, 0.0};
  for (int p0 = 0; p0 < parts; p0 += 8) {
    double x[8][2];
    bool in[8][2];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int q = min(p0 + u, parts - 1);
      const float off = cell - grid_cell(rh.head[q].max, scale);  // inf: an empty part
      const int b0 = off < (float)kCells ? 2 * t - (int)off : -kBins;
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        in[u][e] = p0 + u < parts && b0 + e >= 0 && 2 * t + e < kCells;
        const int b = in[u][e] ? b0 + e : 0;
        x[u][e] = count ? (double)reinterpret_cast<const uint32_t*>(base + (size_t)q * kBins)[b]
                        : base[(size_t)q * kBins + b];
      }
    }
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const double f = count ? 1.0 : rh.part_f[min(p0 + u, parts - 1)];
#pragma unroll
      for (int e = 0; e < 2; ++e)
        if (in[u][e]) v[e] += f * x[u][e];
    }
  }
  const double above = block_scan_excl<double>(v[0] + v[1], sh.wave_d);
  rh.before[2 * t] = above;
  rh.before[2 * t + 1] = above + v[0];
  __syncthreads();
  // The first bin whose running total passes x (kCells: none); bin b's total
  // is before[b + 1] - before[b], so the last usable bin is kCells - 1.
  auto bin_of = [&](double x, bool inclusive) {
    uint32_t mine = 0xFFFFFFFFu;
#pragma unroll
    for (int e = 1; e >= 0; --e) {
      const int b = 2 * t + e;
      if (b >= kCells) continue;
      const double thru = rh.before[b + 1];
      if (inclusive ? thru >= x : thru > x) mine = (uint32_t)b;
    }
    return min(block_first_u(mine, sh), (uint32_t)kCells);
  };
  auto bin_at = [&](float l) { return cell - grid_cell(l, scale); };

  if (count) {
    const uint32_t c = bin_of((double)a.top_k, true);
    if (c == (uint32_t)kCells || rh.before[c + 1] > (double)CCAP) return none;
    const float lo = cell_low(cell - (float)c, scale);
    gather_ranges(src, n, lo, INFINITY, INFINITY, INFINITY, tk);
    rank_top((int)tk.n_cand, a.top_k, tk);
    return tail_topk((uint32_t)a.top_k, a.temperature, a.top_p, r, tk);
  }

  // The top_p cut's bin and the bins the walk can stop in: its target is r
  // times the kept weight, which lies between the cut bin's two ends.
  const bool cutting = a.top_p < 1.0f;
  uint32_t c = (uint32_t)kCells;
  double kept_lo = total, kept_hi = total;
  if (cutting) {
    c = bin_of((double)a.top_p * total, true);
    if (c == (uint32_t)kCells) return none;
    kept_lo = rh.before[c];
    kept_hi = rh.before[c + 1];
  }
  const uint32_t w0 = bin_of(r * kept_lo, false);
  uint32_t w1 = bin_of(r * kept_hi, false);
  if (cutting) w1 = min(w1, c);
  if (w0 > w1 || w1 == (uint32_t)kCells) return none;
  // Their members in order: the walk's bins are one run of the order, the cut
  // bin, where it lies below them, another.
  auto low_of = [&](uint32_t b) { return cell_low(cell - (float)b, scale); };
  const bool apart = cutting && c > w1;
  const float w_hi = w0 == 0 ? INFINITY : low_of(w0 - 1);
  gather_ranges(src, n, low_of(w1), w_hi, apart ? low_of(c) : INFINITY,
                apart ? low_of(c - 1) : INFINITY, tk);
  const int nc = (int)tk.n_cand;
  if (nc > CCAP) return none;
  rank_all(nc, tk);
  if (t < 2) rh.first[t] = 0xFFFFFFFFu;
  __syncthreads();
  // Entries 2 t and 2 t + 1: value, bin, weight, and the weight before them.
  double we[2];
  uint32_t be[2];
#pragma unroll
  for (int e = 0; e < 2; ++e) {
    const int k = 2 * t + e;
    we[e] = 0.0;
    be[e] = 0u;
    if (k < nc) {
      const float l = key_value((uint32_t)(tk.sorted[k] >> 32));
      be[e] = (uint32_t)bin_at(l);
      we[e] = exp(((double)l - mxd) / T);
      atomicMin(&rh.first[be[e] > w1 ? 1 : 0], (uint32_t)k);
    }
  }
  const double pre = block_scan_excl<double>(we[0] + we[1], sh.wave_d);
  if (2 * t < nc) tk.pre[2 * t] = pre;
  if (2 * t + 1 < nc) tk.pre[2 * t + 1] = pre + we[0];
  __syncthreads();
  // The row's running total through entry k.
  auto through = [&](int e) {
    const int k = 2 * t + e;
    const bool low = be[e] > w1;
    return rh.before[low ? c : w0] + ((tk.pre[k] - tk.pre[rh.first[low ? 1 : 0]]) + we[e]);
  };
  auto first_entry = [&](auto test) {
    uint32_t mine = 0xFFFFFFFFu;
#pragma unroll
    for (int e = 1; e >= 0; --e) {
      const int k = 2 * t + e;
      if (k < nc && we[e] != 0.0 && test(e, through(e))) mine = (uint32_t)k;
    }
    return block_first_u(mine, sh);
  };
  auto index_of = [&](uint32_t k) {
    return 0xFFFFFFFFu - (uint32_t)(tk.sorted[k] & 0xFFFFFFFFull);
  };
  uint32_t cut = 0xFFFFFFFFu;
  if (cutting) {
    const double want = (double)a.top_p * total;
    cut = first_entry([&](int e, double thru) { return be[e] == c && thru >= want; });
    if (cut == 0xFFFFFFFFu) return none;
    if ((uint32_t)(2 * t) == (cut & ~1u)) rh.target = cut & 1u ? through(1) : through(0);
    __syncthreads();
    total = rh.target;
  }
  // The walk stops in its own bins: the entries of a cut bin below them are
  // not what follows them in the order.
  const double stop = r * total;
  const uint32_t pick = first_entry([&](int e, double thru) {
    return (uint32_t)(2 * t + e) <= cut && be[e] <= w1 && thru > stop;
  });
  // No entry passes: the last kept one where r * total rounded up to total,
  // else the bins' sums and the entries' differ by a rounding at w1's end.
  if (pick == 0xFFFFFFFFu) return cutting && c == w1 ? index_of(cut) : none;
  return index_of(pick);
}

// `parts` > 0: k_sample_hist has left the row's bins in its workspace.
__global__ __launch_bounds__(NT) void k_sample_rows(SampleArgs a, int parts) {
  extern __shared__ uint32_t bitmap[];
  __shared__ SampleShared sh;
  __shared__ TopKShared tk;
  const int m = blockIdx.x, n = a.n;
  const float* row = a.logits + (size_t)m * a.row_stride;
  double* w = a.wbuf + (size_t)m * n;

  SeenIds seen;
  if (!row_seen(a, m, seen)) {
    if (threadIdx.x == 0) a.active[m] = 0;
    return;
  }
  double r = 0.0;
  if (a.uniform) r = a.uniform[a.tok ? (size_t)a.count[m] * gridDim.x + m : m];
  uint32_t pick = (uint32_t)n;
  if (parts > 0) {
    const float* src = a.penalty == 1.0f || !seen.ids
                           ? row
                           : reinterpret_cast<const float*>(w + hist_doubles(parts));
    pick = pick_binned(a, m, parts, src, r, sh, tk);
    __syncthreads();  // the other paths reuse the row's workspace and LDS
  }
  const uint32_t* bm = pick < (uint32_t)n ? nullptr : seen_bitmap(a, seen, bitmap);
  auto key_of = [&](int i) { return order_key(pen_logit(row, i, bm, a.penalty)); };
  auto l_at = [&](int i) { return pen_logit(row, i, bm, a.penalty); };
  if (pick >= (uint32_t)n && a.temperature > 0.0f && a.top_k > 0 && a.top_k < n &&
      a.top_k <= KCAP && topk_candidates(n, l_at, (uint32_t)a.top_k, sh, tk) >= 0)
    pick = tail_topk((uint32_t)a.top_k, a.temperature, a.top_p, r, tk);
  const bool picked = pick < (uint32_t)n;
  if (picked) {
  } else if (a.temperature <= 0.0f) {
    // sampling.rs:30-32, 83-91: first index of the maximum.
    float bv = -INFINITY;
    uint32_t bi = 0xFFFFFFFFu;
    for_row(n, l_at, [&](float l, int i, bool live) {
      if (live) amax_merge(bv, bi, l, (uint32_t)i);
    });
    const float mx = block_max_f(bv, sh);
    pick = block_min_u(bv == mx ? bi : 0xFFFFFFFFu, sh);
    // The reference's scan starts from index 0 and a NaN there never loses
    // a comparison: it stays the answer.
    if (pick == 0xFFFFFFFFu || __builtin_isnan(pen_logit(row, 0, bm, a.penalty))) pick = 0;
  } else {
    float mxv = -INFINITY;
    for (int i = threadIdx.x; i < n; i += NT) mxv = fmaxf(mxv, pen_logit(row, i, bm, a.penalty));
    const double mx = (double)block_max_f(mxv, sh);
    const double T = (double)a.temperature;

    // top_k (sampling.rs:41-43): the k-th element of the descending order.
    uint32_t kth = (uint32_t)n;
    if (a.top_k > 0 && a.top_k < n) kth = select_desc(n, key_of, nullptr, (double)a.top_k, true, sh);
    const uint32_t kkey = kth < (uint32_t)n ? key_of((int)kth) : 0u;
    // Members: key above the k-th element's, or equal and not after it.
    auto in_k = [&](int i) {
      if (kth >= (uint32_t)n) return true;
      const uint32_t k = key_of(i);
      return k > kkey || (k == kkey && (uint32_t)i <= kth);
    };

    // Probabilities (sampling.rs:45-53).
    double part = 0.0;
    for (int i = threadIdx.x; i < n; i += NT) {
      const double e = in_k(i) ? exp(((double)pen_logit(row, i, bm, a.penalty) - mx) / T) : 0.0;
      w[i] = e;
      part += e;
    }
    // The reference divides every weight by their sum (sampling.rs:50-52),
    // and by the kept sum after the top_p cut, before comparing cumulative
    // sums with top_p and r.  The weights stay unnormalised here and those
    // targets are scaled by the sums instead: the same comparisons up to
    // rounding, without a pass over the row for each division.
    const double sum = block_sum_d(part, sh);
    double total = sum;

    // top_p (sampling.rs:55-70): the smallest prefix reaching top_p, renormalised.
    uint32_t last = kth < (uint32_t)n ? kth : (uint32_t)n;  // last kept element, n = unknown
    if (a.top_p < 1.0f) {
      // No crossing keeps every element (and still renormalises).
      // A target of zero or less is met by the first element, not by an empty bin.
      const double want = (double)a.top_p * sum;
      const uint32_t cut = select_desc(n, key_of, w, want <= 0.0 ? 0x1p-1074 : want, true, sh);
      const uint32_t ckey = cut < (uint32_t)n ? key_of((int)cut) : 0u;
      double kept = 0.0;
      for (int i = threadIdx.x; i < n; i += NT) {
        if (cut < (uint32_t)n) {
          const uint32_t k = key_of(i);
          if (k < ckey || (k == ckey && (uint32_t)i > cut)) w[i] = 0.0;
        }
        kept += w[i];
      }
      total = block_sum_d(kept, sh);
      if (cut < (uint32_t)n) last = cut;
    }

    // The walk (sampling.rs:72-80): first element whose cumulative
    // probability exceeds r; the last kept element if none does.
    pick = select_desc(n, key_of, w, r * total, false, sh);
    if (pick >= (uint32_t)n) {
      if (last >= (uint32_t)n) {
        // Every element is kept: the last of the descending order is the
        // minimum, the highest index among equal minima.
        float mn = INFINITY;
        for (int i = threadIdx.x; i < n; i += NT) mn = fminf(mn, pen_logit(row, i, bm, a.penalty));
        const float lo = -block_max_f(-mn, sh);
        uint32_t hi = 0;
        for (int i = threadIdx.x; i < n; i += NT)
          if (pen_logit(row, i, bm, a.penalty) == lo) hi = max(hi, (uint32_t)i);
        pick = ~block_min_u(~hi, sh);
      } else {
        pick = last;
      }
    }
  }
  if (threadIdx.x == 0) {
    if (a.out) a.out[m] = pick;
    if (a.tok) {
      const int p = a.pos[m];
      const uint32_t c = a.count[m];
      a.gen[(size_t)m * a.max_new + c] = pick;
      a.count[m] = c + 1;
      a.hist[(size_t)m * a.hist_stride + p] = pick;
      a.tok[m] = pick;
      const bool stop = pick == a.eos || p >= a.max_ctx;
      a.active[m] = stop ? 0 : 1;
      a.done[m] = stop || (int)c + 1 >= a.max_new ? 1 : 0;
    }
  }
}

__global__ void k_advance(int* pos, const int* active, int rows, const uint32_t* tok,
                          uint32_t* hist, long hist_stride) {
  const int m = threadIdx.x;
  if (m >= rows || !active[m]) return;
  if (tok) hist[(size_t)m * hist_stride + pos[m]] = tok[m];
  pos[m] += 1;
}

}  // namespace

size_t sample_scratch_bytes(int rows, int n) { return (size_t)rows * n * sizeof(double); }

// Workspace of the allocation-free sampler entry point (the per-row f64
// weights, kNoAllocSampleElems doubles = 16 MiB).  Every GPU the library
// runs on holds its own copy until the process ends.  In host code the
// array's name is not a device address: kernels get the address from
// sample_noalloc_scratch().  A call's kernels write every bin, header and
// weight they read, so the array needs no clearing between calls.
namespace {
__device__ __align__(256) double scratch[kNoAllocSampleElems];
std::mutex g_scratch_mu;
double* g_scratch_ptr[kMaxDevices] = {};
}  // namespace

hipError_t sample_noalloc_scratch(int device, double** ptr) {
  if (device < 0 || device >= kMaxDevices || !ptr) return hipErrorInvalidValue;
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (!g_scratch_ptr[device]) {
    // The caller made `device` current: its copy of the array is resolved.
    void* p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess) return e;
    g_scratch_ptr[device] = static_cast<double*>(p);
  }
  *ptr = g_scratch_ptr[device];
  return hipSuccess;
}

hipError_t launch_advance(int* pos, const int* active, int rows, hipStream_t s,
                          const uint32_t* tok, uint32_t* hist, long hist_stride) {
  if (rows <= 0 || rows > 1024 || (tok && !hist)) return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_advance, dim3(1), dim3(64 * ((rows + 63) / 64)), 0, s, pos, active, rows,
                     tok, hist, hist_stride);
  return hipGetLastError();
}

hipError_t launch_sample_rows(const SampleArgs& a, int rows, hipStream_t s) {
  if (a.n <= 0 || a.n > kMaxSampleVocab || rows <= 0) return hipErrorInvalidValue;
  if (a.tok && (!a.pos || !a.hist || !a.start || !a.active || !a.done || !a.count || !a.gen ||
                a.max_new <= 0))
    return hipErrorInvalidValue;
  const size_t lds = a.penalty != 1.0f && (a.seen || a.tok) ? (size_t)(a.n + 31) / 32 * 4 : 0;
  // Sampled rows long enough for at least one part's bins in their workspace of
  // n doubles (top_k above KCAP stays on the radix path).  us on MI355X, one block
  // per row / binned: 32 x 50257 top_p alone 142 / 32.6, top_k 40 with top_p 37.9
  // / 28.6; 1 x 4100 29.6 / 23.3 and 34.5 / 21.9.
  // With temperature alone the radix path runs one select instead of two, and
  // short rows stay there: 32 x 8000 23.0 / 23.7, 32 x 8200 (two parts) 23.5 / 22.9,
  // 256 x 7000 23.9 / 25.4, 256 x 8000 28.3 / 25.7; over one row per CU 320 x 5000 37.8 / 40.6,
  // 512 x 6000 46.4 / 43.6, 1024 x 4100 78 / 78.
  const bool cut = a.top_p < 1.0f || (a.top_k > 0 && a.top_k < a.n);
  const int from = cut || rows > 768 ? kHistMin
                   : rows > 256      ? 5500
                   : rows > 128      ? 7800
                                     : 2 * kHistMin;
  int parts = 0;
  if (a.temperature > 0.0f && a.temperature < INFINITY && a.n >= from && (a.top_k <= KCAP || a.top_k >= a.n)) {
    // Parts for about 256 blocks of bins in all, at most 16 a row, and no part
    // above 32768 ids while there are at most 1024 blocks (top_k 40 with top_p and
    // a penalty, us at 1, 2, 4 and 8 parts: 256 x 131072 236, 169, 157, 144; 256 x
    // 50257 79, 62, 58, 67; 512 x 131072 337, 315, 315, 296, top_p alone 294, 289,
    // 291, 310).
    parts = std::max(AKH_SAMPLE_BLOCKS / rows, std::min((a.n + 32767) / 32768, 1024 / rows));
    parts = std::min(kPartsMax, std::max(1, parts));
    while (parts > 1 && (2 * hist_doubles(parts) > a.n || a.n / parts < NT)) --parts;
    hipLaunchKernelGGL(k_sample_hist, dim3(rows, parts), dim3(NT), lds, s, a,
                       grid_base(a.temperature, a.top_k > 0 && a.top_k < a.n));
  }
  hipLaunchKernelGGL(k_sample_rows, dim3(rows), dim3(NT), lds, s, a, parts);
  return hipGetLastError();
}

}  // namespace akh
