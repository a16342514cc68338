// Device code of the exact-order small-matrix factor and solve, shared by the
// single-matrix kernels (k_small.hip) and the batched kernels (k_batch.hip).
// Files that include it are compiled with -ffp-contract=off and
// `#pragma clang fp contract(off)`: every `s += x*y` must stay a separately
// rounded multiply and add.
#pragma once

#include "llh_common.h"
#include "llh_kernels.h"

namespace llh {

// Packed column-major lower triangle: entry (j, k), j >= k.
__device__ __forceinline__ int pk(int n, int j, int k) { return k * n - ((k * (k - 1)) >> 1) + (j - k); }

// Stages the lower triangle of the n x n matrix at `a` (row-major, lda) in Ap (packed
// column-major): groups of LG loads are issued before any of them is stored, so
// their latencies overlap.
template <typename TS, typename T, int NT>
__device__ __forceinline__ void stage_lower(const TS* __restrict__ a, int64_t lda, int n, T* Ap) {
  constexpr int LG = 16;
  const int tid = threadIdx.x, sq = n * n;
  for (int e0 = 0; e0 < sq; e0 += NT * LG) {
    TS v[LG];
#pragma unroll
    for (int g = 0; g < LG; ++g) {
      const int e = e0 + g * NT + tid, j = e / n, k = e - j * n;
      v[g] = (e < sq && k <= j) ? a[(int64_t)j * lda + k] : TS(0);
    }
#pragma unroll
    for (int g = 0; g < LG; ++g) {
      const int e = e0 + g * NT + tid, j = e / n, k = e - j * n;
      if (e < sq && k <= j) Ap[pk(n, j, k)] = T(v[g]);
    }
  }
}

// The value of lane `from` (wave-uniform), in every lane.
template <typename T>
__device__ __forceinline__ T lane_value(T v, int from) {
  if constexpr (sizeof(T) == 8) {
    const uint64_t u = __builtin_bit_cast(uint64_t, v);
    const uint32_t lo = __builtin_amdgcn_readlane((uint32_t)u, from);
    const uint32_t hi = __builtin_amdgcn_readlane((uint32_t)(u >> 32), from);
    return __builtin_bit_cast(T, (uint64_t)hi << 32 | lo);
  } else {
    return __builtin_bit_cast(T, __builtin_amdgcn_readlane(__builtin_bit_cast(uint32_t, v), from));
  }
}

// Factors the n x n matrix at `a` (row-major, lda): Ap receives the lower triangle of
// A, W the columns of L below the diagonal (both packed column-major) and Dg its
// diagonal.  Returns -1 on success or the first row j whose pivot fails `d <= 0`; W and
// Dg then hold the columns before it.
//
// A lane holds rows lane + 64 r and a wave the columns wave + NW i: the pending sums
// S[j, k'] (see k_small.hip) stay in registers (on 16 waves in f64, with 128 registers
// each, 36 are spilled; with 8 waves and none the factor takes longer, k_small.hip).  Once column k is in LDS, its successor's
// wave brings that column up to date before any other, takes its pivot and publishes
// it, while the rest of the sums is updated.  The sums move down by one place every NW
// columns, so that the next column is always at place 0 (or 1).
//
// What bounds it: the chain of n pivots (LDS exchange, square root, division: 0.5 us each up
// to n = 64, 1 us with two rows a lane).  With the sums in LDS and every wave waiting for each pivot and then
// each update, one matrix (whole call, us): f64 n = 24 75 -> 38, 64 148 -> 61, 128 411 ->
// 144, f32 n = 176 903 -> 204.
template <typename TS, typename T, int NT, int NMAX>
__device__ int factor_exact(const TS* __restrict__ a, int64_t lda, int n, T* W, T* Ap, T* Dg) {
  constexpr int NW = NT / 64, R = (NMAX + 63) / 64, G = 4;  // places in groups of G
  constexpr int SLOTS = ((NMAX + NW - 1) / NW + G - 1) / G * G;
  __shared__ int s_fail[2];  // by the column's parity: one is read while the other is written
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  if (tid < 2) s_fail[tid] = -1;
  stage_lower<TS, T, NT>(a, lda, n, Ap);
  int jr[R];  // this lane's rows
#pragma unroll
  for (int r = 0; r < R; ++r) jr[r] = min(lane + 64 * r, n - 1);
  T S[R][SLOTS];
#pragma unroll
  for (int r = 0; r < R; ++r)
#pragma unroll
    for (int i = 0; i < SLOTS; ++i) S[r][i] = T(0);
  __syncthreads();
  // column k from its sums s, on one wave
  auto publish = [&](int k, const T (&ak)[R], const T (&s)[R]) __attribute__((always_inline)) {
    T v[R];
#pragma unroll
    for (int r = 0; r < R; ++r) v[r] = ak[r] - s[r];
    T d = lane_value(v[0], k & 63);
#pragma unroll
    for (int r = 1; r < R; ++r)
      if ((k >> 6) == r) d = lane_value(v[r], k & 63);
    if (d <= T(0)) {  // cholesky.rs:69; NaN passes
      if (lane == 0) s_fail[k & 1] = k;
      return;
    }
    const T piv = sqrt_rn(d);
    if (lane == 0) Dg[k] = piv;
    const int colk = pk(n, k, k) - k;
#pragma unroll
    for (int r = 0; r < R; ++r)
      if (64 * r + 63 > k) {
        const T l = v[r] / piv;  // cholesky.rs:62
        const int j = lane + 64 * r;
        if (j > k && j < n) W[colk + j] = l;
      }
  };
  auto column_a = [&](int k, T (&ak)[R]) __attribute__((always_inline)) {
    const int colk = pk(n, k, k) - k;
#pragma unroll
    for (int r = 0; r < R; ++r) ak[r] = Ap[colk + max(jr[r], k)];
  };
  if (wave == 0) {
    T ak[R], z[R];
    column_a(0, ak);
#pragma unroll
    for (int r = 0; r < R; ++r) z[r] = T(0);
    publish(0, ak, z);
  }
  __syncthreads();
  for (int kb = 0; kb < n; kb += NW) {
    for (int c = 0; c < NW && kb + c < n; ++c) {
      const int k = kb + c, colk = pk(n, k, k) - k;
      const int fail = s_fail[k & 1];
      T lj[R];
#pragma unroll
      for (int r = 0; r < R; ++r) lj[r] = W[colk + max(jr[r], k)];  // (rows up to k: not used)
      const int first = kb + wave;  // the column at place 0
      // S[., place] += L[k', k] L[., k], k' the column there
      const bool next0 = c + 1 < NW && wave == c + 1, next1 = c + 1 == NW && wave == 0;
      T ak[R];
      if ((next0 || next1) && k + 1 < n) column_a(k + 1, ak);
      if (__builtin_amdgcn_readfirstlane(fail) >= 0) return fail;
      if ((next0 || next1) && k + 1 < n) {
        const T lk = W[colk + k + 1];
        T s[R];
#pragma unroll
        for (int r = 0; r < R; ++r) {
          s[r] = (next1 ? S[r][1 % SLOTS] : S[r][0]) + lk * lj[r];
        }
        publish(k + 1, ak, s);
      }
#pragma unroll
      for (int i0 = 0; i0 < SLOTS; i0 += G) {
        if (first + NW * i0 < n) {
          T lk[G];
#pragma unroll
          for (int g = 0; g < G; ++g) lk[g] = W[colk + max(min(first + NW * (i0 + g), n - 1), k)];
#pragma unroll
          for (int g = 0; g < G; ++g)
#pragma unroll
            for (int r = 0; r < R; ++r) S[r][i0 + g] = S[r][i0 + g] + lk[g] * lj[r];
        }
      }
      __syncthreads();
    }
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
      for (int i = 0; i + 1 < SLOTS; ++i) S[r][i] = S[r][i + 1];
  }
  return -1;
}

// The same on one wave, with the sums in LDS (W): the wave has no other to wait for,
// and its lanes share the rows of one column.
template <typename TS, typename T, int NMAX>
__device__ int factor_exact_wave(const TS* __restrict__ a, int64_t lda, int n, T* W, T* Ap, T* Dg) {
  constexpr int KG = 8;  // columns whose loads are issued together
  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = tid >> 6;
  constexpr int NT = 64, NW = 1;
  const int tot = (n * (n + 1)) >> 1;
  for (int e = tid; e < tot; e += NT) W[e] = T(0);
  stage_lower<TS, T, NT>(a, lda, n, Ap);
  __syncthreads();
  for (int k = 0; k < n; ++k) {
    // Every thread evaluates the pivot identically, so no broadcast is needed.
    const T d = Ap[pk(n, k, k)] - W[pk(n, k, k)];
    if (d <= T(0)) return k;  // cholesky.rs:69; NaN passes
    const T piv = sqrt_rn(d);
    if (tid == 0) Dg[k] = piv;
    for (int j = k + 1 + tid; j < n; j += NT) {
      const int o = pk(n, j, k);
      W[o] = (Ap[o] - W[o]) / piv;  // cholesky.rs:62
    }
    __syncthreads();
    // Pending sums: S[j,k'] += L[k',k] * L[j,k] for k < k' <= j (k' == j is d_j).
    // Thread (lane, wave) owns rows j = lane + 64 r and columns k' = k+1+wave+NW i;
    // the loads of a group of KG columns are issued together (they never alias
    // the column-k values read), then the group is updated.
    const int colk = pk(n, k, k) - k;  // W[colk + i] == L[i, k]
#pragma unroll
    for (int r = 0; r < (NMAX + 63) / 64; ++r) {
      const int j = lane + 64 * r;
      if (j > k && j < n) {
        const T ljk = W[colk + j];
        for (int kp0 = k + 1 + wave; kp0 <= j; kp0 += KG * NW) {
          T lk[KG], sv[KG];
#pragma unroll
          for (int g = 0; g < KG; ++g) {
            const int kp = kp0 + g * NW;
            const bool on = kp <= j;
            lk[g] = on ? W[colk + kp] : T(0);
            sv[g] = on ? W[pk(n, j, kp)] : T(0);
          }
#pragma unroll
          for (int g = 0; g < KG; ++g) {
            const int kp = kp0 + g * NW;
            if (kp <= j) W[pk(n, j, kp)] = sv[g] + lk[g] * ljk;
          }
        }
      }
    }
    __syncthreads();
  }
  return -1;
}

// Writes the factor back into `a` (lower triangle only; the strict upper
// triangle is never touched, which is the dirty form).  On failure at row f it
// writes rows < f and L[f, 0..f-1], exactly what the reference has written when
// it returns NotPositiveDefinite.
template <typename TS, typename T, int NT>
__device__ void write_back(TS* __restrict__ a, int64_t lda, int n, int fail, const T* W, const T* Dg) {
  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = tid >> 6;
  constexpr int NW = NT / 64;
  const int rows = fail < 0 ? n : fail + 1;
  for (int j = wave; j < rows; j += NW) {
    const int kend = (j == fail) ? j : j + 1;
    for (int k = lane; k < kend; k += 64) a[(int64_t)j * lda + k] = TS((k == j) ? Dg[j] : W[pk(n, j, k)]);
  }
}

// LDS of one small factor + solve on NT threads: only a single wave solves in LDS.
template <typename T, int NMAX, int NT, int MCH>
struct SmallLds {
  T W[(NMAX * (NMAX + 1)) / 2];
  T Ap[(NMAX * (NMAX + 1)) / 2];
  T Dg[NMAX];
  T Bs[NT == 64 ? NMAX * MCH : 1];
  T Xs[NT == 64 ? NMAX * MCH : 1];
};
static_assert(4 * sizeof(SmallLds<double, 64, 128, 8>) <= 160 * 1024, "four matrices of order 64 on a CU");

// Both substitutions with the factor in W and Dg, for all columns of ds.b: a wave
// takes MCH / NW columns at a time, a lane rows lane + 64 r of them in registers, so
// that no wave waits for another (one barrier and two LDS passes per pivot before:
// 8000 systems of order 100 to 128, f64, 12.9 -> 5.0 ms with the factor above).
template <typename T, int NT, int NMAX, int MCH>
__device__ void solve_exact(const SmallDesc<T>& ds, const T* W, const T* Dg) {
  constexpr int NW = NT / 64, R = (NMAX + 63) / 64, CW = MCH / NW;
  const int n = ds.n, lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  int jr[R], row[R];  // this lane's rows, and W[row + i] == L[i, j]
#pragma unroll
  for (int r = 0; r < R; ++r) {
    jr[r] = min(lane + 64 * r, n - 1);
    row[r] = pk(n, jr[r], jr[r]) - jr[r];
  }
  for (int c0 = CW * wave; c0 < ds.m; c0 += MCH) {
    T x[R][CW];
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
      for (int c = 0; c < CW; ++c) x[r][c] = ds.b[(int64_t)jr[r] * ds.ldb + min(c0 + c, ds.m - 1)];
    // L y = b (Lower: rows 0..n, a[r, i] = L[r, i] for r > i), triangular.rs:142.
#pragma unroll
    for (int q = 0; q < R; ++q)
      for (int i = 64 * q; i < min(n, 64 * q + 64); ++i) {
        const int coli = pk(n, i, i) - i;
        const T dg = Dg[i];
        T l[R];
#pragma unroll
        for (int r = q; r < R; ++r) l[r] = W[coli + max(jr[r], i)];
#pragma unroll
        for (int c = 0; c < CW; ++c) {
          const T coeff = lane_value(x[q][c], i & 63) / dg;
#pragma unroll
          for (int r = q; r < R; ++r) {
            const int j = lane + 64 * r;
            const T u = x[r][c] + ((-coeff) * l[r]);
            x[r][c] = j > i ? u : (j == i ? coeff : x[r][c]);
          }
        }
      }
    // L^T x = y (Upper on L.t(): rows n-1..0, a[r, i] = L[i, r] for r < i),
    // cholesky.rs:142 with triangular.rs:140.
#pragma unroll
    for (int q = R - 1; q >= 0; --q)
      for (int i = min(n, 64 * q + 64) - 1; i >= 64 * q; --i) {
        const T dg = Dg[i];
        T l[R];
#pragma unroll
        for (int r = 0; r <= q; ++r) l[r] = W[row[r] + max(i, jr[r])];
#pragma unroll
        for (int c = 0; c < CW; ++c) {
          const T coeff = lane_value(x[q][c], i & 63) / dg;
#pragma unroll
          for (int r = 0; r <= q; ++r) {
            const int j = lane + 64 * r;
            const T u = x[r][c] + ((-coeff) * l[r]);
            x[r][c] = j < i ? u : (j == i ? coeff : x[r][c]);
          }
        }
      }
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
      for (int c = 0; c < CW; ++c)
        if (lane + 64 * r < n && c0 + c < ds.m) ds.b[(int64_t)jr[r] * ds.ldb + c0 + c] = x[r][c];
  }
}

// Factors ds.a (dirty, in place) and, when do_solve, solves ds.b in place in the
// reference's operation order; ds.info receives kNoFail or the failing row.
// do_solve == 2: ds.a already holds the factor (a solve against it, as the
// refinement steps of a batched mixed-precision solve need); ds.info is read:
// a matrix whose factor failed is skipped.
template <typename T, int NMAX, int NT, int MCH>
__device__ void small_solve_one(const SmallDesc<T>& ds, int do_solve, SmallLds<T, NMAX, NT, MCH>& lds) {
  const int n = ds.n;
  if (n > NMAX) return;  // the host never routes a larger matrix here
  T* W = lds.W;
  T* Ap = lds.Ap;
  T* Dg = lds.Dg;
  T* Bs = lds.Bs;
  T* Xs = lds.Xs;
  const int tid = threadIdx.x;
  if (do_solve == 2) {
    if (ds.info[0] != kNoFail) return;
    for (int e = tid; e < n * n; e += NT) {
      const int j = e / n, k = e - j * n;
      if (k < j) W[pk(n, j, k)] = ds.a[(int64_t)j * ds.lda + k];
      else if (k == j) Dg[j] = ds.a[(int64_t)j * ds.lda + j];
    }
  } else {
    int fail;
    if constexpr (NT == 64)
      fail = factor_exact_wave<T, T, NMAX>(ds.a, ds.lda, n, W, Ap, Dg);
    else
      fail = factor_exact<T, T, NT, NMAX>(ds.a, ds.lda, n, W, Ap, Dg);
    __syncthreads();
    write_back<T, T, NT>(ds.a, ds.lda, n, fail, W, Dg);
    if (threadIdx.x == 0) ds.info[0] = fail < 0 ? kNoFail : fail;
    if (fail >= 0 || !do_solve) return;
  }
  if constexpr (NT > 64) {
    __syncthreads();
    solve_exact<T, NT, NMAX, MCH>(ds, W, Dg);
    __syncthreads();
    return;
  }
  // Solve in chunks of MCH right-hand-side columns; b is row-major n x m.
  for (int c0 = 0; c0 < ds.m; c0 += MCH) {
    const int mc = min(MCH, ds.m - c0);
    const int tot = n * mc;
    __syncthreads();
    for (int e = tid; e < tot; e += NT) {
      const int r = e / mc, c = e - r * mc;
      Bs[r * MCH + c] = ds.b[(int64_t)r * ds.ldb + c0 + c];
    }
    __syncthreads();
    // L y = b (Lower: rows 0..n, a[r, i] = L[r, i] for r > i), triangular.rs:142.
    for (int i = 0; i < n; ++i) {
      for (int e = tid; e < (n - i) * mc; e += NT) {
        const int rr = e / mc, c = e - rr * mc, r = i + rr;
        const T coeff = Bs[i * MCH + c] / Dg[i];
        if (r == i) Xs[i * MCH + c] = coeff;
        else Bs[r * MCH + c] = Bs[r * MCH + c] + ((-coeff) * W[pk(n, r, i)]);
      }
      __syncthreads();
    }
    // L^T x = y (Upper on L.t(): rows n-1..0, a[r, i] = L[i, r] for r < i),
    // cholesky.rs:142 with triangular.rs:140.
    for (int i = n - 1; i >= 0; --i) {
      for (int e = tid; e < (i + 1) * mc; e += NT) {
        const int r = e / mc, c = e - r * mc;
        const T coeff = Xs[i * MCH + c] / Dg[i];
        if (r == i) Bs[i * MCH + c] = coeff;
        else Xs[r * MCH + c] = Xs[r * MCH + c] + ((-coeff) * W[pk(n, i, r)]);
      }
      __syncthreads();
    }
    for (int e = tid; e < tot; e += NT) {
      const int r = e / mc, c = e - r * mc;
      ds.b[(int64_t)r * ds.ldb + c0 + c] = Bs[r * MCH + c];
    }
  }
}

}  // namespace llh
