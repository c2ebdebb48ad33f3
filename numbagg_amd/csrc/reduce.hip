// Plain reductions over one axis for gfx950: nansum, nanmean, nancount,
// allnan, anynan, nanvar, nanstd (ndaggregate, numbagg/funcs.py:23-159,
// numbagg/decorators.py:188-272) and nanmax, nanmin, nanargmax, nanargmin
// (ndreduce, numbagg/funcs.py:160-228, numbagg/decorators.py:904-1028).
//
// The host moves the reduced axes last and flattens them, so a kernel sees
// a row-major (rows, n) view with a unit-stride core axis and reduces each
// row to one output; where the innermost axis is kept, it passes the
// (outer, n, cols) view as it lies and the column kernel reduces it in place
// (below), without a transposed copy.
//
// Design: one wavefront reduces one (row, chunk) item. Rows are split into
// chunks so that a launch holds enough wavefronts to fill the device; each
// lane streams 16-byte vectors of its chunk (strided by the wave), keeps a
// private state, and the wave merges its 64 lane states in a fixed butterfly
// order and writes one 32-byte partial. A finalize kernel merges each row's
// chunk partials in chunk order and writes the output. No atomics: results
// are the same bits on every run.
//
// States: float32 sums in float64 (exact differences of 24-bit significands
// stay far inside float64), float64 sums in double-double, integer sums
// wrapping mod 2**64 (narrowed like the reference's fixed-width adds); the
// variance keeps (count, mean, M2) per lane, updated batch by batch with the
// batch's own two-pass moments and Chan's merge (the reference makes two
// passes over the data, numbagg/funcs.py:108-127); extremes as orderable
// 64-bit keys with the index of the first (arg*: the reference replaces on a
// strict `>` / `<`) or last (min/max: it replaces on `>=` / `<=`) occurrence.
#include <cstring>
#include <type_traits>

#include "common.hpp"

namespace nbg {
namespace {

constexpr int kRedThreads = 256;
constexpr int kRedWaves = kRedThreads / kWave;

enum RKind {
  kRSum = 0,
  kRMean = 1,
  kRCount = 2,
  kRAllNan = 3,
  kRAnyNan = 4,
  kRVar = 5,
  kRStd = 6,
  kRMax = 7,
  kRMin = 8,
  kRArgMax = 9,
  kRArgMin = 10,
};

constexpr bool is_var_kind(int k) { return k == kRVar || k == kRStd; }
constexpr bool is_ext_kind(int k) { return k == kRMax || k == kRMin || k == kRArgMax || k == kRArgMin; }
constexpr bool first_wins(int k) { return k == kRArgMax || k == kRArgMin; }

// Partial state of one (row, chunk): 32 bytes.
//   sum/mean: w0 sum (float64 bits, or wrapping u64 for integers), w1 the
//             double-double low part (float64 data), w2 count, w3 the sum of
//             the infinite values (float64 data: +-inf or NaN, else 0);
//   count/allnan/anynan: w2 count of valid values, w3 count of NaNs;
//   var/std: w0 mean, w1 M2 (float64 bits), w2 count;
//   extremes: w0 key (0 = no valid value), w1 index.
struct RPart {
  unsigned long long w0, w1, w2, w3;
};

__device__ __forceinline__ double f64_of(unsigned long long b) { return __longlong_as_double((long long)b); }
__device__ __forceinline__ unsigned long long bits_of(double v) {
  return (unsigned long long)__double_as_longlong(v);
}

// Orderable key of a value compared as float64 (the reference's running
// extremes are float64, also for integer input); -0.0 and +0.0 tie. Maximum
// kinds use the key, minimum kinds its complement; every non-NaN value maps
// to a non-zero word, so 0 stands for "no valid value".
template <typename T>
__device__ __forceinline__ unsigned long long ext_key(T v, bool minimum) {
  const unsigned long long b = bits_of((double)v + 0.0);
  const unsigned long long k = (b & 0x8000000000000000ull) ? ~b : (b | 0x8000000000000000ull);
  return minimum ? ~k : k;
}

// a / b for a count b >= 1: the hardware's reciprocal (2^-24) refined by one
// Newton step (2^-48: 9e-16 for 255, 2e-15 for 4095), the quotient corrected by
// its exact remainder.
__device__ __forceinline__ double div_small(double a, double b) {
  const double e = __builtin_amdgcn_rcp(b);
  const double r = fma(e, fma(-b, e, 1.0), e);
  const double q = a * r;
  return fma(fma(-b, q, a), r, q);
}

// (count, mean, M2) and Chan's merge of another such triple.
struct Chan {
  double n, mean, m2;
  __device__ __forceinline__ void merge(double nb, double mb, double m2b) {
    if (nb == 0.0) return;
    const double tot = n + nb;
    const double d = mb - mean;
    const double f = nb / tot;
    mean += d * f;
    m2 += m2b + d * d * n * f;
    n = tot;
  }
};

// float32 extremes keep 32-bit keys, the best value and a 32-bit index
// within the chunk per lane (chunks are below 2**31 positions); the 64-bit
// key and the absolute index are formed once, when the lane's part is taken.
template <typename T, int KIND>
constexpr bool small_ext() {
  return is_ext_kind(KIND) && sizeof(T) == 4 && std::is_floating_point<T>::value;
}

// Orderable 32-bit key of a float32 value (-0 as +0): larger values give
// larger keys (complemented for minima); every non-NaN value's key is nonzero.
__device__ __forceinline__ uint32_t ext_key32(float v, bool minimum) {
  const uint32_t b = __float_as_uint(v + 0.0f);
  const uint32_t k = (b & 0x80000000u) ? ~b : (b | 0x80000000u);
  return minimum ? ~k : k;
}

template <typename T, int KIND>
struct Lane {
  double s = 0.0;                                 // float32 data: float64 sum
  Comp<double> cs{0.0, 0.0};                      // float64 data: double-double sum of finite values
  double sinf = 0.0;                              // float64 data: sum of the infinite values
  unsigned long long us = 0ull;                   // integers: wrapping sum
  unsigned long long cnt = 0ull, nans = 0ull;
  Chan ch = Chan{0.0, 0.0, 0.0};
  unsigned long long key = 0ull, idx = 0ull;
  uint32_t key32 = 0u, idx32 = 0u;  // small_ext: key (0: none yet), index within the chunk
  T best = T(0);                    // small_ext: the value of key32

  // small_ext: one element at position rel within the chunk, by selects (no
  // branch per element).
  __device__ __forceinline__ void fold32(T v, uint32_t rel) {
    const uint32_t k = ext_key32((float)v, KIND == kRMin || KIND == kRArgMin);
    const bool take = !is_nan(v) && (first_wins(KIND) ? k > key32 : k >= key32);
    key32 = take ? k : key32;
    idx32 = take ? rel : idx32;
    best = take ? v : best;
  }

  // One element at position i (non-variance kinds).
  __device__ __forceinline__ void fold(T v, int64_t i) {
    const bool valid = !is_nan(v);
    if constexpr (KIND == kRSum || KIND == kRMean) {
      if constexpr (!std::is_floating_point<T>::value) {
        us += (unsigned long long)(long long)v;
      } else if constexpr (sizeof(T) == 8) {
        // infinities stay out of the double-double pair, whose error terms
        // would turn them into NaN
        if (valid) {
          if (isfinite((double)v)) cs.add((double)v);
          else sinf += (double)v;
        }
      } else {
        s += valid ? (double)v : 0.0;
      }
      cnt += valid ? 1ull : 0ull;
    } else if constexpr (KIND == kRCount || KIND == kRAllNan || KIND == kRAnyNan) {
      cnt += valid ? 1ull : 0ull;
      nans += valid ? 0ull : 1ull;
    } else if constexpr (is_ext_kind(KIND)) {
      if (valid) {
        const unsigned long long k = ext_key(v, KIND == kRMin || KIND == kRArgMin);
        // a lane visits increasing positions: strictly larger keys replace
        // (first occurrence), or larger-or-equal keys (last occurrence)
        const bool take = first_wins(KIND) ? k > key : k >= key;
        if (take) {
          key = k;
          idx = (unsigned long long)i;
        }
      }
    }
  }

  // A batch of B elements (variance kinds): its own two-pass moments, merged.
  template <int B>
  __device__ __forceinline__ void fold_batch(const T (&v)[B]) {
    double sb = 0.0;
    int nb = 0;
#pragma unroll
    for (int j = 0; j < B; ++j) {
      const bool valid = !is_nan(v[j]);
      sb += valid ? (double)v[j] : 0.0;
      nb += valid ? 1 : 0;
    }
    if (nb == 0) return;
    const double mb = sb / (double)nb;
    double m2b = 0.0;
#pragma unroll
    for (int j = 0; j < B; ++j) {
      const double d = (double)v[j] - mb;
      m2b += !is_nan(v[j]) ? d * d : 0.0;
    }
    ch.merge((double)nb, mb, m2b);
  }

  // The same without float64 divisions: the batch mean and the merge's weight
  // by reciprocals (div_small), whose quotients are the rounded ones but for
  // rare ties; so equal values have exactly their value as mean, and no variance.
  template <int B>
  __device__ __forceinline__ void fold_batch_rcp(const T (&v)[B]) {
    double sb = 0.0;
    int nb = 0;
#pragma unroll
    for (int j = 0; j < B; ++j) {
      const bool valid = !is_nan(v[j]);
      sb += valid ? (double)v[j] : 0.0;
      nb += valid ? 1 : 0;
    }
    const double dn = (double)nb;
    const double mb = div_small(sb, nb > 0 ? dn : 1.0);
    double m2b = 0.0;
#pragma unroll
    for (int j = 0; j < B; ++j) {
      const double d = !is_nan(v[j]) ? (double)v[j] - mb : 0.0;
      m2b = fma(d, d, m2b);
    }
    if (nb == 0) return;
    if (ch.n == 0.0) {
      ch = Chan{dn, mb, m2b};
      return;
    }
    const double tot = ch.n + dn;
    const double d = mb - ch.mean;
    const double f = div_small(dn, tot);
    ch.mean += d * f;
    ch.m2 += m2b + d * d * ch.n * f;
    ch.n = tot;
  }

  // c0: the chunk's first position (small_ext indices are relative to it).
  __device__ __forceinline__ RPart to_part(int64_t c0) const {
    RPart p{0ull, 0ull, 0ull, 0ull};
    if constexpr (small_ext<T, KIND>()) {
      if (key32 != 0u) {
        p.w0 = ext_key(best, KIND == kRMin || KIND == kRArgMin);
        p.w1 = (unsigned long long)(c0 + (int64_t)idx32);
      }
      return p;
    }
    if constexpr (KIND == kRSum || KIND == kRMean) {
      if constexpr (!std::is_floating_point<T>::value) {
        p.w0 = us;
      } else if constexpr (sizeof(T) == 8) {
        p.w0 = bits_of(cs.hi);
        p.w1 = bits_of(cs.lo);
        p.w3 = bits_of(sinf);
      } else {
        p.w0 = bits_of(s);
      }
      p.w2 = cnt;
    } else if constexpr (KIND == kRCount || KIND == kRAllNan || KIND == kRAnyNan) {
      p.w2 = cnt;
      p.w3 = nans;
    } else if constexpr (is_var_kind(KIND)) {
      p.w0 = bits_of(ch.mean);
      p.w1 = bits_of(ch.m2);
      p.w2 = (unsigned long long)ch.n;
    } else {
      p.w0 = key;
      p.w1 = idx;
    }
    return p;
  }
};

// Merge partial b (a later or any other part of the row) into a.
template <typename T, int KIND>
__device__ __forceinline__ void merge_part(RPart& a, const RPart& b) {
  if constexpr (KIND == kRSum || KIND == kRMean) {
    if constexpr (!std::is_floating_point<T>::value) {
      a.w0 += b.w0;
    } else if constexpr (sizeof(T) == 8) {
      Comp<double> x{f64_of(a.w0), f64_of(a.w1)};
      x.add(Comp<double>{f64_of(b.w0), f64_of(b.w1)});
      a.w0 = bits_of(x.hi);
      a.w1 = bits_of(x.lo);
      a.w3 = bits_of(f64_of(a.w3) + f64_of(b.w3));
    } else {
      a.w0 = bits_of(f64_of(a.w0) + f64_of(b.w0));
    }
    a.w2 += b.w2;
  } else if constexpr (KIND == kRCount || KIND == kRAllNan || KIND == kRAnyNan) {
    a.w2 += b.w2;
    a.w3 += b.w3;
  } else if constexpr (is_var_kind(KIND)) {
    Chan c{(double)a.w2, f64_of(a.w0), f64_of(a.w1)};
    c.merge((double)b.w2, f64_of(b.w0), f64_of(b.w1));
    a.w0 = bits_of(c.mean);
    a.w1 = bits_of(c.m2);
    a.w2 = a.w2 + b.w2;
  } else {
    // larger key wins; equal keys: the smaller (first) or larger (last) index
    const bool take = b.w0 > a.w0 || (b.w0 == a.w0 && b.w0 != 0ull &&
                                      (first_wins(KIND) ? b.w1 < a.w1 : b.w1 > a.w1));
    if (take) {
      a.w0 = b.w0;
      a.w1 = b.w1;
    }
  }
}

__device__ __forceinline__ RPart shfl_xor_part(const RPart& p, int m) {
  RPart q;
  q.w0 = (unsigned long long)__shfl_xor((long long)p.w0, m, kWave);
  q.w1 = (unsigned long long)__shfl_xor((long long)p.w1, m, kWave);
  q.w2 = (unsigned long long)__shfl_xor((long long)p.w2, m, kWave);
  q.w3 = (unsigned long long)__shfl_xor((long long)p.w3, m, kWave);
  return q;
}

// One (row, chunk) item per wavefront: item = block * 4 + wave.
template <typename T, int KIND, int VEC, int U>
__global__ __launch_bounds__(kRedThreads) void reduce_kernel(const T* __restrict__ x, int64_t n, int64_t ld,
                                                             int64_t chunk, int64_t chunks_per_row,
                                                             int64_t items, RPart* __restrict__ parts) {
  const int64_t item = (int64_t)blockIdx.x * kRedWaves + wave_id();
  if (item >= items) return;  // whole wavefronts leave; no barriers below
  const int lane = lane_id();
  const int64_t row = item / chunks_per_row;
  const int64_t ck = item - row * chunks_per_row;
  const int64_t c0 = ck * chunk;
  const int64_t c1 = c0 + chunk < n ? c0 + chunk : n;
  const T* xr = x + row * ld;
  Lane<T, KIND> st;
  constexpr int64_t STEP = (int64_t)kWave * VEC;
  constexpr int64_t SUPER = STEP * U;
  struct V {
    T v[VEC];
  };
  int64_t e = c0;
  if (VEC > 1) {
    // full super-steps: U vectors per lane, all loads issued first
    for (; e + SUPER <= c1; e += SUPER) {
      V vv[U];
#pragma unroll
      for (int u = 0; u < U; ++u) vv[u] = load_stream(reinterpret_cast<const V*>(xr + e + u * STEP + lane * VEC));
      if constexpr (is_var_kind(KIND)) {
        T b[U * VEC];
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
          for (int j = 0; j < VEC; ++j) b[u * VEC + j] = vv[u].v[j];
        st.template fold_batch<U * VEC>(b);
      } else if constexpr (small_ext<T, KIND>()) {
        const uint32_t rel = (uint32_t)(e - c0) + (uint32_t)(lane * VEC);
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
          for (int j = 0; j < VEC; ++j) st.fold32(vv[u].v[j], rel + (uint32_t)(u * STEP + j));
      } else {
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
          for (int j = 0; j < VEC; ++j) st.fold(vv[u].v[j], e + u * STEP + lane * VEC + j);
      }
    }
  }
  // remainder (or the whole chunk for unaligned rows): one element per lane
  for (int64_t i = e + lane; i < c1; i += kWave) {
    if constexpr (is_var_kind(KIND)) {
      const T b[1] = {xr[i]};
      st.template fold_batch<1>(b);
    } else if constexpr (small_ext<T, KIND>()) {
      st.fold32(xr[i], (uint32_t)(i - c0));
    } else {
      st.fold(xr[i], i);
    }
  }
  RPart p = st.to_part(c0);
#pragma unroll
  for (int m = 1; m < kWave; m <<= 1) {
    const RPart q = shfl_xor_part(p, m);
    // merge in position order: the lower lane's state first
    if (lane & m) {
      RPart lo = q;
      merge_part<T, KIND>(lo, p);
      p = lo;
    } else {
      merge_part<T, KIND>(p, q);
    }
  }
  if (lane == 0) parts[item] = p;
}

// The output of one row from its merged partial; the row's element i is
// x[i * step].
template <typename T, typename TO, int KIND>
__device__ __forceinline__ TO part_value(const RPart& p, int64_t ddof, const T* __restrict__ x, int64_t step) {
  TO r;
  if constexpr (KIND == kRSum) {
    if constexpr (!std::is_floating_point<T>::value) {
      r = (TO)(T)(long long)p.w0;  // modular narrowing
    } else {
      const double inf = f64_of(p.w3);
      r = (TO)(inf != 0.0 || inf != inf ? inf : f64_of(p.w0) + f64_of(p.w1));
    }
  } else if constexpr (KIND == kRMean) {
    const double inf = f64_of(p.w3);
    const double s = inf != 0.0 || inf != inf ? inf : f64_of(p.w0) + f64_of(p.w1);
    r = p.w2 ? (TO)(s / (double)p.w2) : (TO)canonical_nan<double>();
  } else if constexpr (KIND == kRCount) {
    r = (TO)p.w2;
  } else if constexpr (KIND == kRAllNan) {
    r = (TO)(p.w2 == 0 ? 1 : 0);
  } else if constexpr (KIND == kRAnyNan) {
    r = (TO)(p.w3 != 0 ? 1 : 0);
  } else if constexpr (is_var_kind(KIND)) {
    const long long c = (long long)p.w2;
    if (c > ddof) {
      const double var = f64_of(p.w1) / (double)(c - ddof);
      r = (TO)(KIND == kRStd ? sqrt(var) : var);
    } else {
      r = (TO)canonical_nan<double>();
    }
  } else if constexpr (KIND == kRArgMax || KIND == kRArgMin) {
    r = p.w0 ? (TO)p.w1 : (TO)-1;  // -1: no valid value (the host raises)
  } else {
    // the value at the extreme's index, through float64 as the reference's
    // float64 running extreme returns it (64-bit integers round there)
    if (p.w0 == 0ull) r = (TO)canonical_nan<double>();
    else r = (TO)(double)x[(int64_t)p.w1 * step];
  }
  return r;
}

// Output of one row from its chunk partials (merged in chunk order), a thread
// per row.
template <typename T, typename TO, int KIND>
__global__ void reduce_finalize_kernel(const RPart* __restrict__ parts, int64_t rows, int64_t chunks_per_row,
                                       int64_t ddof, const T* __restrict__ x, int64_t ld, TO* __restrict__ out) {
  const int64_t row = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (row >= rows) return;
  RPart p = parts[row * chunks_per_row];
  for (int64_t c = 1; c < chunks_per_row; ++c) merge_part<T, KIND>(p, parts[row * chunks_per_row + c]);
  out[row] = part_value<T, TO, KIND>(p, ddof, x + row * ld, 1);
}

// The same for rows of many chunks, a workgroup per row: each thread merges a
// contiguous run of chunks, then a pairwise tree over the threads in order
// (left before right, so every merge keeps chunk order; deterministic).
constexpr int kRedFinishThreads = 256;

template <typename T, typename TO, int KIND>
__global__ __launch_bounds__(kRedFinishThreads) void reduce_finalize_wide_kernel(
    const RPart* __restrict__ parts, int64_t chunks_per_row, int64_t ddof, const T* __restrict__ x, int64_t ld,
    TO* __restrict__ out) {
  __shared__ RPart sp[kRedFinishThreads];
  __shared__ int hv[kRedFinishThreads];
  const int64_t row = blockIdx.x;
  const int t = threadIdx.x;
  const int64_t per = (chunks_per_row + kRedFinishThreads - 1) / kRedFinishThreads;
  const int64_t c0 = t * per;
  const int64_t c1 = c0 + per < chunks_per_row ? c0 + per : chunks_per_row;
  const RPart* rp = parts + row * chunks_per_row;
  RPart p{};
  int have = 0;
  for (int64_t c = c0; c < c1; ++c) {
    if (have) merge_part<T, KIND>(p, rp[c]);
    else p = rp[c];
    have = 1;
  }
  sp[t] = p;
  hv[t] = have;
  for (int stride = 1; stride < kRedFinishThreads; stride <<= 1) {
    __syncthreads();
    if ((t & (2 * stride - 1)) == 0 && hv[t + stride]) {
      if (hv[t]) {
        RPart a = sp[t];
        merge_part<T, KIND>(a, sp[t + stride]);
        sp[t] = a;
      } else {
        sp[t] = sp[t + stride];
        hv[t] = 1;
      }
    }
  }
  if (t == 0) out[row] = part_value<T, TO, KIND>(sp[0], ddof, x + row * ld, 1);
}

// ---- reductions over an axis that is not the innermost -----------------------
// x[a * ld_a + i * ld_r + c], a < outer, i < n, c < cols: every (a, c) reduces
// its n elements. A workgroup takes `cl` column lanes (V neighbouring columns
// each, one vector load per row) by 256 / cl row lanes of one (a, split): the
// row lanes of few-column arrays read consecutive rows, so a wave's loads stay
// contiguous for any column count. Each lane keeps U rows of loads in flight
// and a private state per column, the row lanes merge pairwise in LDS in a
// fixed order, and the splits' partials are merged in split order by the
// finalize kernel (deterministic, no atomics).
//
// Bound by HBM: one streaming read of x. 16-byte accesses need element
// alignment only, so any column offset and row stride takes the vector path.
template <typename T, int V>
struct alignas(alignof(T)) ColVec {
  T v[V];
};

constexpr int kColUnroll = 8;

template <typename T, int KIND, int V>
__global__ __launch_bounds__(kRedThreads) void reduce_cols_kernel(const T* __restrict__ x, int64_t n, int64_t cols,
                                                                  int64_t ld_a, int64_t ld_r, int cl,
                                                                  int64_t col_tiles, int64_t splits, int64_t chunk,
                                                                  int64_t total, RPart* __restrict__ parts) {
  constexpr int U = kColUnroll;
  __shared__ RPart sp[kRedThreads * V];
  const int tid = threadIdx.x;
  const int RL = kRedThreads / cl;
  const int lc = tid % cl, rl = tid / cl;
  const int64_t tile = blockIdx.x % col_tiles;
  const int64_t rest = blockIdx.x / col_tiles;
  const int64_t split = rest % splits, a = rest / splits;
  const int64_t c = (tile * cl + lc) * V;
  const int64_t i0 = split * chunk;
  const int64_t i1 = i0 + chunk < n ? i0 + chunk : n;
  const bool act = rl < RL && c < cols;
  const int nv = act ? (int)(cols - c < V ? cols - c : V) : 0;
  Lane<T, KIND> st[V];
  auto fold_one = [&](int k, T v, int64_t i) {
    if constexpr (is_var_kind(KIND)) {
      const T b[1] = {v};
      st[k].template fold_batch_rcp<1>(b);
    } else if constexpr (small_ext<T, KIND>()) {
      st[k].fold32(v, (uint32_t)(i - i0));
    } else {
      st[k].fold(v, i);
    }
  };
  if (nv == V) {
    using CV = ColVec<T, V>;
    const T* p = x + a * ld_a + c;
    int64_t i = i0 + rl;
    for (; i + (U - 1) * RL < i1; i += U * RL) {
      CV vv[U];
#pragma unroll
      for (int u = 0; u < U; ++u) vv[u] = load_stream(reinterpret_cast<const CV*>(p + (i + u * RL) * ld_r));
#pragma unroll
      for (int k = 0; k < V; ++k) {
        if constexpr (is_var_kind(KIND)) {
          T b[U];
#pragma unroll
          for (int u = 0; u < U; ++u) b[u] = vv[u].v[k];
          st[k].template fold_batch_rcp<U>(b);
        } else {
#pragma unroll
          for (int u = 0; u < U; ++u) fold_one(k, vv[u].v[k], i + u * RL);
        }
      }
    }
    for (; i < i1; i += RL) {
      const CV q = load_stream(reinterpret_cast<const CV*>(p + i * ld_r));
#pragma unroll
      for (int k = 0; k < V; ++k) fold_one(k, q.v[k], i);
    }
  } else if (nv > 0) {  // the last columns, short of a vector
    const T* p = x + a * ld_a + c;
    for (int64_t i = i0 + rl; i < i1; i += RL)
#pragma unroll
      for (int k = 0; k < V; ++k)
        if (k < nv) fold_one(k, p[i * ld_r + k], i);
  }
  RPart q[V];
#pragma unroll
  for (int k = 0; k < V; ++k) q[k] = st[k].to_part(i0);
  if (RL > 1) {  // uniform
#pragma unroll
    for (int k = 0; k < V; ++k) sp[k * kRedThreads + tid] = q[k];
    for (int s = 1; s < RL; s <<= 1) {
      __syncthreads();
      if (act && (rl & (2 * s - 1)) == 0 && rl + s < RL) {
#pragma unroll
        for (int k = 0; k < V; ++k) {
          merge_part<T, KIND>(q[k], sp[k * kRedThreads + tid + s * cl]);
          sp[k * kRedThreads + tid] = q[k];
        }
      }
    }
  }
  if (act && rl == 0) {
#pragma unroll
    for (int k = 0; k < V; ++k)
      if (k < nv) parts[split * total + a * cols + c + k] = q[k];
  }
}

template <typename T, typename TO, int KIND>
__global__ void reduce_cols_finalize_kernel(const RPart* __restrict__ parts, int64_t total, int64_t splits,
                                            int64_t cols, int64_t ld_a, int64_t ld_r, int64_t ddof,
                                            const T* __restrict__ x, TO* __restrict__ out) {
  const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= total) return;
  RPart p = parts[q];
  for (int64_t s = 1; s < splits; ++s) merge_part<T, KIND>(p, parts[s * total + q]);
  const int64_t a = q / cols;
  out[q] = part_value<T, TO, KIND>(p, ddof, x + a * ld_a + (q - a * cols), ld_r);
}

// The launch's shape: column lanes, tiles and row splits.
struct ColShape {
  int v, cl;
  int64_t tiles, splits, chunk;
};

// Vectors of 16 bytes where they fill at least half a wave; columns split
// evenly over the tiles. Row splits: a grid of about 2048 workgroups, 8 per CU,
// of which the registers (and the 32 KiB of LDS of 4-byte vectors) let 4 to 5 be
// resident with vectors, 7 to 8 with single columns; each split at least two
// unrolled steps of every row lane. (3653, 65160) float32 nanvar takes 255 tiles
// by 8 splits.
inline ColShape col_shape(int64_t outer, int64_t n, int64_t cols, int elem) {
  ColShape c{};
  const int vmax = 16 / elem;
  c.v = cols >= 32 * vmax ? vmax : 1;
  const int64_t units = (cols + c.v - 1) / c.v;
  c.tiles = (units + kWave - 1) / kWave;
  c.cl = (int)((units + c.tiles - 1) / c.tiles);
  const int64_t step = (int64_t)(kRedThreads / c.cl) * kColUnroll;
  const int64_t base = outer * c.tiles;
  int64_t splits = base > 0 ? (2048 + base - 1) / base : 1;
  const int64_t most = n / (2 * step);
  if (splits > most) splits = most;
  if (splits < 1) splits = 1;
  c.chunk = (n + splits - 1) / splits;
  c.chunk = (c.chunk + step - 1) / step * step;
  if (c.chunk < step) c.chunk = step;
  c.splits = n > 0 ? (n + c.chunk - 1) / c.chunk : 1;
  return c;
}

// Chunks per row: about 8 wavefronts per SIMD over the device, chunks of
// whole super-steps and at least 16 KiB of data.
template <typename T>
int64_t reduce_chunk(int64_t rows, int64_t n, int64_t super_elems) {
  int dev = 0, cus = 256;
  if (hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) !=
                                              hipSuccess || cus <= 0)
    cus = 256;
  const int64_t target = (int64_t)cus * 4 * 8;
  int64_t per_row = target / (rows > 0 ? rows : 1);
  if (per_row < 1) per_row = 1;
  int64_t chunk = (n + per_row - 1) / per_row;
  const int64_t min_chunk = 16384 / (int64_t)sizeof(T);
  if (chunk < min_chunk) chunk = min_chunk;
  chunk = (chunk + super_elems - 1) / super_elems * super_elems;
  // below 2**31 positions (float32 extremes index within the chunk in 32 bits)
  const int64_t max_chunk = ((int64_t)1 << 31) / super_elems * super_elems;
  return chunk < max_chunk ? chunk : max_chunk;
}

template <typename T>
constexpr int red_unroll() {
  return 4;
}

size_t reduce_ws_bytes(int64_t rows, int64_t n, int elem) {
  if (rows <= 0) return 0;
  const int64_t super = (int64_t)kWave * (16 / elem) * 4;
  // the same chunking as the launch, computed without the device query
  // (at most rows * ceil(n / min_chunk) items; bounded by rows * 8192)
  int64_t min_chunk = 16384 / elem;
  min_chunk = (min_chunk + super - 1) / super * super;
  int64_t per_row = n > 0 ? (n + min_chunk - 1) / min_chunk : 1;
  if (per_row < 1) per_row = 1;
  return (size_t)(rows * per_row) * sizeof(RPart);
}

template <typename T, typename TO, int KIND>
int reduce_impl(const T* x, TO* out, int64_t rows, int64_t n, int64_t ld, int64_t ddof, void* ws,
                size_t ws_bytes, hipStream_t s) {
  constexpr int VEC = 16 / (int)sizeof(T);
  constexpr int U = red_unroll<T>();
  const int64_t super = (int64_t)kWave * VEC * U;
  const int64_t chunk = n > 0 ? reduce_chunk<T>(rows, n, super) : super;
  const int64_t cpr = n > 0 ? (n + chunk - 1) / chunk : 1;
  const int64_t items = rows * cpr;
  if ((size_t)items * sizeof(RPart) > ws_bytes || ws == nullptr)
    return set_error(NBG_ERR_INVALID, "reduce: workspace too small (%zu < %zu)", ws_bytes,
                     (size_t)items * sizeof(RPart));
  const int64_t blocks = (items + kRedWaves - 1) / kRedWaves;
  if (blocks > 0x7fffffffLL) return set_error(NBG_ERR_INVALID, "reduce: too many rows");
  RPart* parts = static_cast<RPart*>(ws);
  // 16-byte loads need element alignment only: rows of any length and offset
  // take them (float32 nanvar of (9, 32628569): 427 -> 193 us)
  if (pick_vec_elem<T>(x, x, x) == VEC)
    hipLaunchKernelGGL((reduce_kernel<T, KIND, VEC, U>), dim3((unsigned)blocks), dim3(kRedThreads), 0, s, x, n, ld,
                       chunk, cpr, items, parts);
  else
    hipLaunchKernelGGL((reduce_kernel<T, KIND, 1, 1>), dim3((unsigned)blocks), dim3(kRedThreads), 0, s, x, n, ld,
                       chunk, cpr, items, parts);
  if (int rc = check_hip(hipGetLastError(), "reduce_kernel launch")) return rc;
  if (cpr >= 64 && rows <= 0x7fffffffLL) {
    hipLaunchKernelGGL((reduce_finalize_wide_kernel<T, TO, KIND>), dim3((unsigned)rows), dim3(kRedFinishThreads), 0,
                       s, parts, cpr, ddof, x, ld, out);
  } else {
    const int64_t fblocks = (rows + 255) / 256;
    hipLaunchKernelGGL((reduce_finalize_kernel<T, TO, KIND>), dim3((unsigned)fblocks), dim3(256), 0, s, parts, rows,
                       cpr, ddof, x, ld, out);
  }
  return check_hip(hipGetLastError(), "reduce_finalize_kernel launch");
}

template <typename T, typename TO, int KIND>
int reduce_cols_impl(const T* x, TO* out, int64_t outer, int64_t n, int64_t cols, int64_t ld_a, int64_t ld_r,
                     int64_t ddof, void* ws, size_t ws_bytes, hipStream_t s) {
  constexpr int VEC = 16 / (int)sizeof(T);
  const ColShape c = col_shape(outer, n, cols, (int)sizeof(T));
  const int64_t total = outer * cols;
  const size_t need = (size_t)(total * c.splits) * sizeof(RPart);
  if (ws == nullptr || ws_bytes < need)
    return set_error(NBG_ERR_INVALID, "reduce: workspace too small (%zu < %zu)", ws_bytes, need);
  const int64_t blocks = outer * c.tiles * c.splits;
  const int64_t fblocks = (total + 255) / 256;
  // positions relative to a split are kept in 32 bits (float32 extremes)
  if (blocks > 0x7fffffffLL || fblocks > 0x7fffffffLL || c.chunk > 0x7fffffffLL)
    return set_error(NBG_ERR_INVALID, "reduce: too many rows");
  RPart* parts = static_cast<RPart*>(ws);
  if (c.v == VEC)
    hipLaunchKernelGGL((reduce_cols_kernel<T, KIND, VEC>), dim3((unsigned)blocks), dim3(kRedThreads), 0, s, x, n,
                       cols, ld_a, ld_r, c.cl, c.tiles, c.splits, c.chunk, total, parts);
  else
    hipLaunchKernelGGL((reduce_cols_kernel<T, KIND, 1>), dim3((unsigned)blocks), dim3(kRedThreads), 0, s, x, n, cols,
                       ld_a, ld_r, c.cl, c.tiles, c.splits, c.chunk, total, parts);
  if (int rc = check_hip(hipGetLastError(), "reduce_cols_kernel launch")) return rc;
  hipLaunchKernelGGL((reduce_cols_finalize_kernel<T, TO, KIND>), dim3((unsigned)fblocks), dim3(256), 0, s, parts,
                     total, c.splits, cols, ld_a, ld_r, ddof, x, out);
  return check_hip(hipGetLastError(), "reduce_cols_finalize_kernel launch");
}

// The (rows, n) view of a reduction (cols == 0: element i of row r is
// x[r * ld + i]), or its (outer, n, cols) view (element i of (a, c) is
// x[a * ld_a + i * ld + c]).
struct RView {
  int64_t rows, n, ld, cols, ld_a;
};

// Output dtype per kind: sum -> input; mean/var/std -> input (floats only);
// count, argmax, argmin -> int64; allnan/anynan -> uint8 (bool); max/min ->
// input for floats, int64 for integers.
template <int KIND>
int reduce_view(const char* name, int dtype, const void* x, void* out, const RView& w, int64_t ddof, void* ws,
                size_t ws_bytes, void* stream) {
  const int64_t rows = w.rows, n = w.n, ld = w.ld;
  if (int rc = injected_error(name)) return rc;
  if (rows < 0 || n < 0) return set_error(NBG_ERR_INVALID, "%s: negative shape", name);
  if (rows == 0) return NBG_OK;
  if ((x == nullptr && n > 0) || out == nullptr) return set_error(NBG_ERR_INVALID, "%s: null pointer", name);
  if (w.cols == 0 && rows > 1 && ld < n) return set_error(NBG_ERR_INVALID, "%s: row stride < n", name);
  if (w.cols > 0 && ((n > 1 && ld < w.cols) || (rows > 1 && w.ld_a < 0)))
    return set_error(NBG_ERR_INVALID, "%s: row stride < cols", name);
  if (n == 0 && (KIND == kRArgMax || KIND == kRArgMin || KIND == kRMax || KIND == kRMin))
    return set_error(NBG_ERR_INVALID, "%s: zero-size reduction", name);
  constexpr bool FLOAT_ONLY = KIND == kRMean || is_var_kind(KIND);
  hipStream_t s = static_cast<hipStream_t>(stream);
  const bool flt = dtype == NBG_F32 || dtype == NBG_F64;
  if (FLOAT_ONLY && !flt) return set_error(NBG_ERR_INVALID, "%s: float32 or float64 input required", name);
#define NBG_R(T, TO)                                                                                          \
  do {                                                                                                        \
    if (w.cols > 0)                                                                                           \
      return reduce_cols_impl<T, TO, KIND>((const T*)x, (TO*)out, rows, n, w.cols, w.ld_a, ld, ddof, ws,      \
                                           ws_bytes, s);                                                      \
    return reduce_impl<T, TO, KIND>((const T*)x, (TO*)out, rows, n, ld, ddof, ws, ws_bytes, s);               \
  } while (0)
  if constexpr (KIND == kRCount || KIND == kRArgMax || KIND == kRArgMin) {
    switch (dtype) {
      case NBG_F32: NBG_R(float, int64_t);
      case NBG_F64: NBG_R(double, int64_t);
      case NBG_I32: NBG_R(int32_t, int64_t);
      case NBG_I64: NBG_R(int64_t, int64_t);
    }
  } else if constexpr (KIND == kRAllNan || KIND == kRAnyNan) {
    switch (dtype) {
      case NBG_F32: NBG_R(float, uint8_t);
      case NBG_F64: NBG_R(double, uint8_t);
      case NBG_I32: NBG_R(int32_t, uint8_t);
      case NBG_I64: NBG_R(int64_t, uint8_t);
    }
  } else if constexpr (FLOAT_ONLY) {
    switch (dtype) {
      case NBG_F32: NBG_R(float, float);
      case NBG_F64: NBG_R(double, double);
    }
  } else if constexpr (KIND == kRSum) {
    switch (dtype) {
      case NBG_F32: NBG_R(float, float);
      case NBG_F64: NBG_R(double, double);
      case NBG_I32: NBG_R(int32_t, int32_t);
      case NBG_I64: NBG_R(int64_t, int64_t);
    }
  } else {  // max / min
    switch (dtype) {
      case NBG_F32: NBG_R(float, float);
      case NBG_F64: NBG_R(double, double);
      case NBG_I32: NBG_R(int32_t, int64_t);
      case NBG_I64: NBG_R(int64_t, int64_t);
    }
  }
#undef NBG_R
  return set_error(NBG_ERR_INVALID, "%s: unsupported dtype code %d", name, dtype);
}

template <int KIND>
int reduce_entry(const char* name, int dtype, const void* x, void* out, int64_t rows, int64_t n, int64_t ld,
                 int64_t ddof, void* ws, size_t ws_bytes, void* stream) {
  return reduce_view<KIND>(name, dtype, x, out, RView{rows, n, ld, 0, 0}, ddof, ws, ws_bytes, stream);
}

}  // namespace
}  // namespace nbg

extern "C" {

size_t nbg_reduce_cols_workspace_bytes(int64_t outer, int64_t n, int64_t cols, int dtype) {
  if (outer <= 0 || cols <= 0 || n < 0) return 0;
  const int elem = (dtype == NBG_F64 || dtype == NBG_I64) ? 8 : 4;
  return (size_t)(outer * cols * nbg::col_shape(outer, n, cols, elem).splits) * sizeof(nbg::RPart);
}

int nbg_reduce_cols(const char* name, int dtype, const void* x, void* out, int64_t outer, int64_t n, int64_t cols,
                    int64_t ld_outer, int64_t ld_row, int64_t ddof, void* ws, size_t ws_bytes, void* stream) {
  using namespace nbg;
  if (name == nullptr) return set_error(NBG_ERR_INVALID, "nbg_reduce_cols: null name");
  if (cols < 0) return set_error(NBG_ERR_INVALID, "%s: negative shape", name);
  if (cols == 0) return NBG_OK;
  const RView w{outer, n, ld_row, cols, ld_outer};
#define NBG_COLS(NAME, KIND) \
  if (strcmp(name, NAME) == 0) return reduce_view<KIND>(NAME, dtype, x, out, w, ddof, ws, ws_bytes, stream)
  NBG_COLS("nbg_nansum", kRSum);
  NBG_COLS("nbg_nanmean", kRMean);
  NBG_COLS("nbg_nancount", kRCount);
  NBG_COLS("nbg_allnan", kRAllNan);
  NBG_COLS("nbg_anynan", kRAnyNan);
  NBG_COLS("nbg_nanvar", kRVar);
  NBG_COLS("nbg_nanstd", kRStd);
  NBG_COLS("nbg_nanmax", kRMax);
  NBG_COLS("nbg_nanmin", kRMin);
  NBG_COLS("nbg_nanargmax", kRArgMax);
  NBG_COLS("nbg_nanargmin", kRArgMin);
#undef NBG_COLS
  return set_error(NBG_ERR_INVALID, "nbg_reduce_cols: unknown reduction %s", name);
}

size_t nbg_reduce_workspace_bytes(int64_t rows, int64_t n, int dtype) {
  const int elem = (dtype == NBG_F64 || dtype == NBG_I64) ? 8 : 4;
  return nbg::reduce_ws_bytes(rows, n, elem);
}

#define NBG_REDUCE(NAME, KIND)                                                                          \
  int NAME(int dtype, const void* x, void* out, int64_t rows, int64_t n, int64_t ld, void* ws,          \
           size_t ws_bytes, void* stream) {                                                             \
    return nbg::reduce_entry<KIND>(#NAME, dtype, x, out, rows, n, ld, 0, ws, ws_bytes, stream);       \
  }
#define NBG_REDUCE_DDOF(NAME, KIND)                                                                     \
  int NAME(int dtype, const void* x, void* out, int64_t rows, int64_t n, int64_t ld, int64_t ddof,      \
           void* ws, size_t ws_bytes, void* stream) {                                                   \
    return nbg::reduce_entry<KIND>(#NAME, dtype, x, out, rows, n, ld, ddof, ws, ws_bytes, stream);    \
  }

NBG_REDUCE(nbg_nansum, nbg::kRSum)
NBG_REDUCE(nbg_nanmean, nbg::kRMean)
NBG_REDUCE(nbg_nancount, nbg::kRCount)
NBG_REDUCE(nbg_allnan, nbg::kRAllNan)
NBG_REDUCE(nbg_anynan, nbg::kRAnyNan)
NBG_REDUCE_DDOF(nbg_nanvar, nbg::kRVar)
NBG_REDUCE_DDOF(nbg_nanstd, nbg::kRStd)
NBG_REDUCE(nbg_nanmax, nbg::kRMax)
NBG_REDUCE(nbg_nanmin, nbg::kRMin)
NBG_REDUCE(nbg_nanargmax, nbg::kRArgMax)
NBG_REDUCE(nbg_nanargmin, nbg::kRArgMin)

}  // extern "C"
