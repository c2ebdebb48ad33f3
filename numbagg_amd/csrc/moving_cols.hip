// Moving-window statistics over an axis that is not the innermost (gfx950).
//
// Reference semantics: numbagg/moving.py:12-275 with the gufunc's axis
// argument; the arithmetic is that of moving.hip (float64 running sums of
// exact differences for float32 sum and mean, float64 moments about a shift
// for var / std / cov / corr, double-double for float64 data).
//
// x[a * ld_o + i * ld_r + c], a < outer, i < n, c < cols (cols contiguous);
// out is (outer * cols, n): each (a, c) series becomes one contiguous row, the
// layout the general path (series moved last, then moving.hip) also returns.
//
// Design: a wave owns 64 neighbouring columns and a range of `tc` positions.
// Each lane walks its own column: the window ending before the range is summed
// first, then every position adds its head and removes its tail (`window`
// positions back, read again: those lines were fetched `window` steps ago and
// come from the L2 or the MALL). An infinity that leaves makes the lane sum its
// window anew. All loads are whole 256-byte lines of a wave,
// and the next 16 positions are in flight while 8 are evaluated.
// Outputs turn through LDS, one 128-byte line of each of the 64 series at a
// time, and leave as whole lines past the caches: each series is written up to
// its own last line boundary, the rest waits in LDS for the next tile (pieces
// at the tile's boundaries left every line in two halves: 787 instead of
// 594 us below; streaming the whole lines, so that they leave the L2 to the
// tails, 552 us). One wave per workgroup: the barriers around the LDS tile are
// then waits of the wave on itself.
//
// Bound by the memory traffic of the tails that the L2 no longer holds (2.7 GB
// read for 0.95): (3653, 65160) float32 move_mean, window 30, takes 552 us
// against 294 for one read and one write. A transposed copy (1.43 ms) and
// moving.hip on the rows (0.63 ms) took its place before.
#include <cstring>

#include "rolling.hpp"

namespace nbg {
namespace {

constexpr int kColsStep = 8;  // positions in flight per lane
// Positions per tile: one 128-byte line of outputs per series.
template <typename T>
constexpr int cols_tile() {
  return 128 / (int)sizeof(T);
}

struct MoveColsArgs {
  const void* xa;
  const void* xb;
  void* out;
  int64_t n, cols, lda_o, lda_r, ldb_o, ldb_r, window, min_count;
  int64_t groups, chunks, tc;
};

template <typename S>
struct IsMoments : std::false_type {};
template <typename T, int NM>
struct IsMoments<MomStats<T, NM>> : std::true_type {};

// c * s12 - s1 * s2 (c times the co-moment about the mean) of double-double
// sums, rounded once: the products keep their low parts, so data far from the
// lane's shift loses nothing here.
__device__ __forceinline__ double scaled_comoment(double c, const Comp<double>& s12, const Comp<double>& s1,
                                                  const Comp<double>& s2) {
  const double p = c * s12.hi, q = s1.hi * s2.hi;
  const double pe = fma(c, s12.hi, -p) + c * s12.lo;
  const double qe = fma(s1.hi, s2.hi, -q) + (s1.hi * s2.lo + s1.lo * s2.hi);
  double d, e;
  two_sum(p, -q, d, e);
  return d + (e + (pe - qe));
}

// The same for a variance, which is zero where all that is left is the rounding
// of the sums: for one repeated value after others that is up to 2^-92 of
// c * s11 where both are alike in size, 2^-77 where that value lies nearest to
// the shift (2000 positions of random values or walks, emulated).
// Taken for a variance it made correlations of noise.
__device__ __forceinline__ double scaled_m2(double c, const Comp<double>& s11, const Comp<double>& s1) {
  const double d = scaled_comoment(c, s11, s1, s1);
  return fabs(d) <= 0x1p-76 * (c * s11.hi) ? 0.0 : d;
}

template <typename T, int KIND>
__device__ __forceinline__ T cols_out(const typename Traits<T, KIND>::S& s, int64_t mc) {
  if constexpr (sizeof(T) == 8 && Traits<T, KIND>::SHIFT) {
    if (s.c < (KIND == kCorr ? (mc > 1 ? mc : 1) : (mc > 2 ? mc : 2))) return canonical_nan<T>();
    const double c = (double)s.c;
    // The scaled forms leave the range of float64 sooner than the row kernel's,
    // which the fallback below is; infinite inputs (NaN here) take it too.
    if constexpr (KIND == kCorr) {
      const double vv = scaled_m2(c, s.s11, s.s1) * scaled_m2(c, s.s22, s.s2);
      if (__builtin_expect(vv < __builtin_inf(), 1))
        return vv > 0 ? scaled_comoment(c, s.s12, s.s1, s.s2) / sqrt(vv) : canonical_nan<T>();
    } else if constexpr (KIND == kCov) {
      const double cov = scaled_comoment(c, s.s12, s.s1, s.s2);
      if (__builtin_expect(fabs(cov) < __builtin_inf(), 1)) return cov / (c * (c - 1.0));
    } else {
      const double m2 = scaled_m2(c, s.s11, s.s1);
      if (__builtin_expect(fabs(m2) < __builtin_inf(), 1)) {
        const double var = m2 / (c * (c - 1.0));
        return KIND == kStd ? sqrt(var) : var;
      }
    }
    return Traits<T, KIND>::out(s, mc, nullptr);
  } else {
    return Traits<T, KIND>::out(s, mc, nullptr);
  }
}

// LINES: outputs leave line by line past the caches, as described above; else
// (outputs that the caches hold) tile by tile, with half the LDS.
template <typename T, int KIND, bool LINES>
__global__ __launch_bounds__(kWave) void move_cols_kernel(MoveColsArgs A) {
  using Tr = Traits<T, KIND>;
  using S = typename Tr::S;
  constexpr bool TWO = Tr::NARGS == 2;
  constexpr int U = kColsStep, TB = cols_tile<T>(), LD = kWave + 1;
  constexpr int ROWS = LINES ? 2 * TB : TB;
  __shared__ T tr[ROWS * LD];  // outputs: position t in row (t - t0) mod ROWS
  const int lane = threadIdx.x;
  const int64_t group = blockIdx.x % A.groups;
  const int64_t rest = blockIdx.x / A.groups;
  const int64_t ck = rest % A.chunks, a = rest / A.chunks;
  const int64_t cg = group * kWave;
  const int ncol = (int)(A.cols - cg < kWave ? A.cols - cg : kWave);
  const int lc = lane < ncol ? lane : ncol - 1;  // spare lanes repeat the last column, their outputs are dropped
  const T* pa = static_cast<const T*>(A.xa) + a * A.lda_o + cg;
  const T* pb = TWO ? static_cast<const T*>(A.xb) + a * A.ldb_o + cg : nullptr;
  T* po = static_cast<T*>(A.out) + (a * A.cols + cg) * A.n;
  const int64_t n = A.n, w = A.window;
  const int64_t t0 = ck * A.tc;
  const int64_t t1 = t0 + A.tc < n ? t0 + A.tc : n;

  // positions [p, p + U) of both inputs; outside [lo, hi): NaN (uniform tests)
  auto load = [&](T (&va)[U], T (&vb)[U], int64_t p, int64_t lo, int64_t hi) {
    if (p >= lo && p + U <= hi) {
#pragma unroll
      for (int u = 0; u < U; ++u) {
        va[u] = (pa + (p + u) * A.lda_r)[lc];
        vb[u] = TWO ? (pb + (p + u) * A.ldb_r)[lc] : T(0);
      }
      return;
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const bool in = p + u >= lo && p + u < hi;
      va[u] = in ? (pa + (p + u) * A.lda_r)[lc] : canonical_nan<T>();
      vb[u] = TWO ? (in ? (pb + (p + u) * A.ldb_r)[lc] : canonical_nan<T>()) : T(0);
    }
  };

  S st = S::zero();
  // Shift of the moment kinds: the lane's first finite value (pair) of the
  // window before the range or of the range itself. The state is zero until
  // then, or holds an infinity, after which the window is summed anew, with a
  // shift of its own.
  T ka = T(0), kb = T(0);
  bool shifted = false;
  // Compensated sums would turn an infinity into NaN: those keep the sum of
  // the window's infinities (0: none) beside the finite values.
  constexpr bool COMP = !IsMoments<S>::value && !std::is_same<S, SumStats<T, D>>::value;
  double inf_part = 0.0;
  auto step = [&](T ha, T hb, T ta, T tb) {
    const bool hv = TWO ? !(is_nan(ha) || is_nan(hb)) : !is_nan(ha);
    const bool tv = TWO ? !(is_nan(ta) || is_nan(tb)) : !is_nan(ta);
    if constexpr (IsMoments<S>::value) {
      if (!shifted && fabs((double)ha) < __builtin_inf() && (!TWO || fabs((double)hb) < __builtin_inf())) {
        ka = ha;
        kb = hb;
        shifted = true;
      }
      acc_moments<false>(st, hv, ha, hb, ka, kb);
      acc_moments<true>(st, tv, ta, tb, ka, kb);
    } else {
      T h0 = hv ? ha : T(0), l0 = tv ? ta : T(0);
      if constexpr (COMP) {
        if (fabs((double)h0) == __builtin_inf()) {
          inf_part += (double)h0;
          h0 = T(0);
        }
        l0 = fabs((double)l0) == __builtin_inf() ? T(0) : l0;
      }
      st.s.add(exact_diff<typename S::Acc, T>(h0, l0));
      st.c += (int)hv - (int)tv;
    }
  };

  // The window ending at t0 - 1.
  T ha[U], hb[U], ta[U], tb[U], na[U], nb[U];
  load(ha, hb, t0, 0, t1);
  load(na, nb, t0 + U, 0, t1);
  {
    const int64_t h0 = t0 - w > 0 ? t0 - w : 0;
    T va[U], vb[U];
    for (int64_t p = h0; p < t0; p += U) {
      load(va, vb, p, 0, t0);
#pragma unroll
      for (int u = 0; u < U; ++u) step(va[u], vb[u], canonical_nan<T>(), T(0));
    }
  }
  load(ta, tb, t0 - w, 0, t1);
  // Offset of position t0 of this lane's series within its line, per store
  // below: series `col` is written by lanes (col % CPS) * LPL .. + LPL.
  constexpr int VO = 16 / (int)sizeof(T);
  constexpr int LPL = TB / VO;         // lanes per line
  constexpr int CPS = kWave / LPL;     // lines per store
  const int j = (lane % LPL) * VO;
  const uint32_t e0 = (uint32_t)((uintptr_t)(po + t0) / sizeof(T));
  const uint32_t n32 = (uint32_t)n;
  // One tile more than the positions fill, to write what waits in LDS.
  for (int64_t q0 = t0; q0 < t1 + (LINES ? TB : 0); q0 += TB) {
    const int row0 = (int)(q0 - t0) & (ROWS - TB);  // LDS rows of this tile: 0.. or TB..
#pragma unroll 1
    for (int g = 0; q0 < t1 && g < TB / U; ++g) {
      const int64_t p = q0 + g * U;
      T fa[U], fb[U], nta[U], ntb[U];  // two steps ahead; tails one step ahead
      load(fa, fb, p + 2 * U, 0, t1);
      load(nta, ntb, p + U - w, 0, t1);
#pragma unroll
      for (int u = 0; u < U; ++u) {
        step(ha[u], hb[u], ta[u], tb[u]);
        // An infinity that leaves the window leaves inf - inf behind: sum the
        // window anew (no other value can).
        if (__builtin_expect(fabs((double)ta[u]) == __builtin_inf() ||
                                 (TWO && fabs((double)tb[u]) == __builtin_inf()),
                             0)) {
          st = S::zero();
          inf_part = 0.0;
          ka = kb = T(0);
          shifted = false;
          const int64_t e = p + u;
          for (int64_t r = e - w + 1 > 0 ? e - w + 1 : 0; r <= e && r < n; ++r)
            step((pa + r * A.lda_r)[lc], TWO ? (pb + r * A.ldb_r)[lc] : T(0), canonical_nan<T>(), T(0));
        }
        T r = cols_out<T, KIND>(st, A.min_count);
        if constexpr (COMP) r = inf_part == 0.0 || is_nan(r) ? r : (T)inf_part;
        tr[(row0 + g * U + u) * LD + lane] = r;
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        ha[u] = na[u];
        hb[u] = nb[u];
        na[u] = fa[u];
        nb[u] = fb[u];
        ta[u] = nta[u];
        tb[u] = ntb[u];
      }
    }
    __syncthreads();
    // Line boundary to line boundary: [q0 - off, q0 - off + TB) of each series.
#pragma unroll
    for (int s = 0; s < LPL; ++s) {
      const int col = s * CPS + lane / LPL;
      const int off = LINES ? (int)((e0 + (uint32_t)col * n32) % TB) : 0;
      const int64_t t = q0 - off + j;
      if (col < ncol && t < t1) {
        T* dst = po + (int64_t)col * n + t;
        const int r = (int)(t - t0);  // from -TB on
        T v[VO];
#pragma unroll
        for (int k = 0; k < VO; ++k) v[k] = tr[((r + k) & (ROWS - 1)) * LD + col];
        if (r >= 0 && t + VO <= t1) {
          if (LINES && t - j >= t0 && t - j + TB <= t1) {  // a whole line
            store_stream16(dst, v);
          } else {
            Vec16<T> q;
#pragma unroll
            for (int k = 0; k < VO; ++k) q.v[k] = v[k];
            *reinterpret_cast<Vec16<T>*>(dst) = q;
          }
        } else {
#pragma unroll
          for (int k = 0; k < VO; ++k)
            if (r + k >= 0 && t + k < t1) dst[k] = v[k];
        }
      }
    }
    __syncthreads();
  }
}

// Positions per wave, or 0 where the general path is the better one: fewer
// than half a wave of columns, or a window that would be summed anew (and its
// tails read) for too few positions. A grid of about 8192 waves where the array
// holds that many of at least 64 positions (a CU holds 9 of them at a time where
// whole lines are written, by LDS, else 8 to 19, by registers and LDS: the rest
// of the grid evens out the end); at most 4096 positions (2048 for float64), after
// which the running sums start afresh, as the tiles of moving.hip do.
int64_t move_cols_chunk(int elem, int64_t outer, int64_t n, int64_t cols, int64_t window) {
  if (outer <= 0 || n <= 0 || cols < 32 || window <= 0) return 0;
  const int64_t groups = (cols + kWave - 1) / kWave;
  if (outer > 0x7fffffffLL / groups) return 0;
  const int64_t most = elem == 4 ? 4096 : 2048;
  int64_t tc = (int64_t)((double)n * (double)(outer * groups) / 8192.0);
  tc = tc < 64 ? 64 : (tc > most ? most : tc);
  tc = (tc + 31) / 32 * 32;  // whole tiles
  if (window > 2 * tc) return 0;
  const int64_t chunks = (n + tc - 1) / tc;
  return chunks > 0x7fffffffLL / (outer * groups) ? 0 : tc;
}

template <typename T, int KIND>
int move_cols_launch(MoveColsArgs a, int64_t outer, hipStream_t s) {
  // Outputs that fit the 256 MB MALL twice stay in the caches, where half lines
  // meet their other halves: (301, 29736) float32 move_std takes 44 us in tiles,
  // 60 in lines; (3653, 65160) move_mean 787 against 552 us.
  const dim3 grid((unsigned)(outer * a.groups * a.chunks)), block(kWave);
  if ((double)outer * a.cols * a.n * sizeof(T) > 128e6)
    hipLaunchKernelGGL((move_cols_kernel<T, KIND, true>), grid, block, 0, s, a);
  else
    hipLaunchKernelGGL((move_cols_kernel<T, KIND, false>), grid, block, 0, s, a);
  return check_hip(hipGetLastError(), "move_cols_kernel launch");
}

template <int KIND>
int move_cols_entry(const char* name, int dtype, MoveColsArgs a, int64_t outer, void* stream) {
  constexpr bool TWO = KIND == kCov || KIND == kCorr;
  if (int rc = injected_error(name)) return rc;
  if (outer < 0 || a.n < 0 || a.cols < 0) return set_error(NBG_ERR_INVALID, "%s: negative shape", name);
  if (a.min_count < 0)
    return set_error(NBG_ERR_INVALID, "%s: min_count must be positive: %lld", name, (long long)a.min_count);
  if (!(a.window > 0 && a.window <= a.n))
    return set_error(NBG_ERR_INVALID, "%s: window not in valid range: %lld", name, (long long)a.window);
  if (dtype != NBG_F32 && dtype != NBG_F64)
    return set_error(NBG_ERR_INVALID, "%s: unsupported dtype code %d", name, dtype);
  if (outer == 0 || a.cols == 0) return NBG_OK;
  if (a.xa == nullptr || a.out == nullptr || (TWO && a.xb == nullptr))
    return set_error(NBG_ERR_INVALID, "%s: null pointer", name);
  if (a.lda_r < a.cols || (TWO && a.ldb_r < a.cols)) return set_error(NBG_ERR_INVALID, "%s: row stride < cols", name);
  a.tc = move_cols_chunk(dtype == NBG_F32 ? 4 : 8, outer, a.n, a.cols, a.window);
  if (a.tc == 0) return set_error(NBG_ERR_INVALID, "%s: shape outside the column kernel's range", name);
  a.groups = (a.cols + kWave - 1) / kWave;
  a.chunks = (a.n + a.tc - 1) / a.tc;
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (dtype == NBG_F64) return move_cols_launch<double, KIND>(a, outer, s);
  if constexpr (KIND == kSum || KIND == kMean) {
    if (f32_twosum_requested()) return move_cols_launch<float, KIND + 16>(a, outer, s);
  }
  return move_cols_launch<float, KIND>(a, outer, s);
}

}  // namespace
}  // namespace nbg

extern "C" {

int64_t nbg_move_cols_chunk(int dtype, int64_t outer, int64_t n, int64_t cols, int64_t window) {
  return nbg::move_cols_chunk(dtype == NBG_F64 ? 8 : 4, outer, n, cols, window);
}

int nbg_move_cols(const char* name, int dtype, const void* a, const void* b, void* out, int64_t outer, int64_t n,
                  int64_t cols, int64_t lda_outer, int64_t lda_row, int64_t ldb_outer, int64_t ldb_row,
                  int64_t window, int64_t min_count, void* stream) {
  using namespace nbg;
  if (name == nullptr) return set_error(NBG_ERR_INVALID, "nbg_move_cols: null name");
  MoveColsArgs m{};
  m.xa = a;
  m.xb = b;
  m.out = out;
  m.n = n;
  m.cols = cols;
  m.lda_o = lda_outer;
  m.lda_r = lda_row;
  m.ldb_o = ldb_outer;
  m.ldb_r = ldb_row;
  m.window = window;
  m.min_count = min_count;
#define NBG_COLS(NAME, KIND) \
  if (strcmp(name, NAME) == 0) return move_cols_entry<KIND>(NAME, dtype, m, outer, stream)
  NBG_COLS("nbg_move_sum", kSum);
  NBG_COLS("nbg_move_mean", kMean);
  NBG_COLS("nbg_move_var", kVar);
  NBG_COLS("nbg_move_std", kStd);
  NBG_COLS("nbg_move_cov", kCov);
  NBG_COLS("nbg_move_corr", kCorr);
#undef NBG_COLS
  return set_error(NBG_ERR_INVALID, "nbg_move_cols: unknown function %s", name);
}

}  // extern "C"
