// Products of the dedicated inverse A^-1 = L^-T L^-1 (potri_enqueue): W = L^-1 one
// level of halves at a time, then the lower triangle of W^T W and its mirror.
// Every product has a triangular operand, whose zero blocks bound the sum of a
// tile; each launch holds all independent tiles of a level.
//
// What bounds it: MFMA and, for small orders, the longest sum of one 64 x 64 tile
// (n products of 16 x 16 x 4 on four SIMDs); 64 x 64 tiles keep that short and the
// chip full.  Against the recursion with one product per launch and full
// operands, n = 3000 f64: 7.1 -> 1.8 ms with the factor (n = 8192 36.0 -> 15.7); with
// the tiles' order and addresses below 1.58.
#include "k_gemm_impl.h"
#include "llh_common.h"
#include "llh_kernels.h"

namespace llh {
namespace {

constexpr int kInvT = 512;  // 8 waves, 32 x 16 of the tile each
constexpr int kInvK = 32;   // k per slab
constexpr int kInvRun = 128;

// acc = sum over k in [klo, khi) of op(A)[m0 + i, k] B[k, n0 + j] for this wave's
// part of a 64 x 64 tile; A is M x K row-major (TA: K x M), B is K x N row-major.
// Slabs of kInvK go through LDS in k-major order, the next one loaded into
// registers while the current one is multiplied.  k beyond khi reads as zero.  The sum is taken in runs of kInvRun k, each
// added to the total as a whole: summed straight through, the rounding grows with
// the order (f32 inverse, n = 3000: 1.2e-6 against 4.3e-7 relative).
template <typename T, bool TA>
__device__ __forceinline__ void inv_tile(int M, int N, int klo, int khi, const T* __restrict__ A, int64_t lda,
                                         const T* __restrict__ B, int64_t ldb, int m0, int n0,
                                         typename Mfma<T>::acc_t (&acc)[2]) {
  using MF = Mfma<T>;
  constexpr int PER = 64 * kInvK / kInvT, S = 64 + 16 / (int)sizeof(T);
  __shared__ T As[2][kInvK * S], Bs[2][kInvK * S];
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6, fr = lane & 15, fk = lane >> 4;
  const int wm = (wave >> 2) * 32, wn = (wave & 3) * 16;
  T va[PER], vb[PER];
  // This thread's pieces: addresses of slab klo, advanced slab by slab (computed
  // anew for each they cost the last level's first product 131 us instead of 116, W^T W
  // 242 instead of 223).  Rows and columns
  // beyond M, N repeat the last one; what they give is not stored.
  const T *pa[PER], *pb[PER];
  int ka[PER], kb[PER];
#pragma unroll
  for (int p = 0; p < PER; ++p) {
    const int e = t + p * kInvT;
    ka[p] = TA ? e / 64 : e % kInvK;
    kb[p] = e / 64;
    const int64_t gr = min(m0 + (TA ? e % 64 : e / kInvK), M - 1), gk = klo + ka[p];
    pa[p] = TA ? A + gk * lda + gr : A + gr * lda + gk;
    pb[p] = B + (int64_t)(klo + kb[p]) * ldb + min(n0 + e % 64, N - 1);
  }
  const int64_t da = TA ? kInvK * lda : kInvK, db = kInvK * ldb;
  auto load = [&](int k0) __attribute__((always_inline)) {
    const bool whole = k0 + kInvK <= khi;
#pragma unroll
    for (int p = 0; p < PER; ++p) {
      if (whole) {
        va[p] = *pa[p];
        vb[p] = *pb[p];
      } else {
        va[p] = k0 + ka[p] < khi ? *pa[p] : T(0);
        vb[p] = k0 + kb[p] < khi ? *pb[p] : T(0);
      }
      pa[p] += da;
      pb[p] += db;
    }
  };
  auto store = [&](int buf) __attribute__((always_inline)) {
#pragma unroll
    for (int p = 0; p < PER; ++p) {
      const int e = t + p * kInvT;
      As[buf][(TA ? e / 64 : e % kInvK) * S + (TA ? e % 64 : e / kInvK)] = va[p];
      Bs[buf][(e / 64) * S + e % 64] = vb[p];
    }
  };
  typename MF::acc_t run[2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int r = 0; r < 4; ++r) acc[i][r] = run[i][r] = T(0);
  load(klo);
  store(0);
  __syncthreads();
  int buf = 0;
  for (int k0 = klo; k0 < khi; k0 += kInvK, buf ^= 1) {
    const bool more = k0 + kInvK < khi;
    if (more) load(k0 + kInvK);
#pragma unroll
    for (int s = 0; s < kInvK / 4; ++s) {
      const T* as = &As[buf][(4 * s + fk) * S + wm + fr];
      const T b = Bs[buf][(4 * s + fk) * S + wn + fr];
      run[0] = MF::mma(as[0], b, run[0]);
      run[1] = MF::mma(as[16], b, run[1]);
    }
    if (!more || (k0 - klo) % kInvRun == kInvRun - kInvK) {
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          acc[i][r] += run[i][r];
          run[i][r] = T(0);
        }
    }
    if (more) store(buf ^ 1);
    __syncthreads();
  }
}

// Level h of W = L^-1: for each pair of diagonal blocks (n1 = h rows at o = 2 h y,
// then n2 <= h) FIRST: T_y = L21 W11 (T at tmp + y h^2, ld h); otherwise W21 =
// -W22 T_y.  Column block n0 of W11 starts at its row n0; row block m0 of W22 ends
// with its column m0 + 63.
template <typename T, bool FIRST>
__global__ __launch_bounds__(kInvT) void inv_level_kernel(int n, int h, const T* __restrict__ L, int64_t lda, T* W,
                                                          int64_t ldw, T* tmp) {
  const int o = 2 * h * blockIdx.y, n2 = min(h, n - o - h), nt = h / 64;
  const int mt = (n2 + 63) / 64, tiles = mt * nt, half = (tiles + 1) / 2;
  int t0 = blockIdx.x;
  if (t0 >= tiles) return;
  // Tiles by the length of their sums, the longer half first and the rest from the
  // shortest up: workgroups that share a CU come half a launch apart (n = 3000, f64:
  // the last level's first product 197 -> 131 us, its second 76 -> 64, against row
  // order, in which the longest shared one).
  if (t0 >= half) t0 = tiles - 1 - (t0 - half);
  const int m0 = (FIRST ? t0 % mt : mt - 1 - t0 / nt) * 64, n0 = (FIRST ? t0 / mt : t0 % nt) * 64;
  T* t = tmp + (int64_t)blockIdx.y * h * h;
  const T* w = W + (int64_t)o * ldw + o;
  typename Mfma<T>::acc_t acc[2];
  if constexpr (FIRST)
    inv_tile<T, false>(n2, h, n0, h, L + (int64_t)(o + h) * lda + o, lda, w, ldw, m0, n0, acc);
  else
    inv_tile<T, false>(n2, h, 0, min(m0 + 64, n2), w + (int64_t)h * ldw + h, ldw, t, h, m0, n0, acc);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int col = n0 + (wave & 3) * 16 + (lane & 15);
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int row = m0 + (wave >> 2) * 32 + 16 * i + Mfma<T>::row(lane, r);
      if (row >= n2) continue;
      if constexpr (FIRST)
        t[(int64_t)row * h + col] = acc[i][r];
      else
        W[(int64_t)(o + h + row) * ldw + o + col] = -acc[i][r];
    }
}

// X = W^T W, both triangles: tile (tm, tn), tm >= tn, sums k from its first row on
// and is stored at (tm, tn) and, transposed, at (tn, tm).  Tiles with the longest
// sums come first.
template <typename T>
__global__ __launch_bounds__(kInvT) void inv_wtw_kernel(int n, const T* __restrict__ W, int64_t ldw,
                                                        T* __restrict__ X, int64_t ldx) {
  const int64_t t = blockIdx.x;
  int64_t tm = (int64_t)((sqrt(8.0 * (double)t + 1.0) - 1.0) * 0.5);
  while (tm * (tm + 1) / 2 > t) --tm;
  while ((tm + 1) * (tm + 2) / 2 <= t) ++tm;
  const int m0 = (int)tm * 64, n0 = (int)(t - tm * (tm + 1) / 2) * 64;
  typename Mfma<T>::acc_t acc[2];
  inv_tile<T, true>(n, n, m0, n, W, ldw, W, ldw, m0, n0, acc);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int col = n0 + (wave & 3) * 16 + (lane & 15);
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int row = m0 + (wave >> 2) * 32 + 16 * i + Mfma<T>::row(lane, r);
      if (row >= n || col > row) continue;  // (the strict upper part of a diagonal tile is the lower's mirror)
      X[(int64_t)row * ldx + col] = acc[i][r];
      X[(int64_t)col * ldx + row] = acc[i][r];
    }
}

// The diagonal blocks of W: the inverses the factor has left.
template <typename T>
__global__ __launch_bounds__(256) void inv_diag_kernel(int n, const T* __restrict__ dinv, T* __restrict__ W,
                                                       int64_t ldw) {
  const int k0 = blockIdx.x * kNB;
  const T* d = dinv + (int64_t)blockIdx.x * kNB * kNB;
  for (int e = threadIdx.x; e < kNB * kNB; e += 256) {
    const int r = e / kNB, c = e % kNB;
    if (k0 + r < n && k0 + c < n) W[(int64_t)(k0 + r) * ldw + k0 + c] = d[e];
  }
}

}  // namespace

template <typename T>
hipError_t launch_inv_diag(int n, const T* dinv, T* w, int64_t ldw, hipStream_t s) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL((inv_diag_kernel<T>), dim3((n + kNB - 1) / kNB), dim3(256), 0, s, n, dinv, w, ldw);
  return hipGetLastError();
}

template <typename T>
hipError_t launch_inv_level(int n, int h, const T* l, int64_t lda, T* w, int64_t ldw, T* tmp, hipStream_t s) {
  if (h <= 0 || h % kNB != 0) return hipErrorInvalidValue;
  const int pairs = n > h ? (n - h + 2 * h - 1) / (2 * h) : 0;  // those with a second block
  if (pairs <= 0) return hipSuccess;
  const int first_rows = pairs == 1 ? (n - h < h ? n - h : h) : h;  // rows of the largest second block
  const dim3 grid(((first_rows + 63) / 64) * (h / 64), pairs);
  hipLaunchKernelGGL((inv_level_kernel<T, true>), grid, dim3(kInvT), 0, s, n, h, l, lda, w, ldw, tmp);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL((inv_level_kernel<T, false>), grid, dim3(kInvT), 0, s, n, h, l, lda, w, ldw, tmp);
  return hipGetLastError();
}

template <typename T>
hipError_t launch_inv_wtw(int n, const T* w, int64_t ldw, T* x, int64_t ldx, hipStream_t s) {
  if (n <= 0) return hipSuccess;
  const int64_t nt = (n + 63) / 64;
  hipLaunchKernelGGL((inv_wtw_kernel<T>), dim3((unsigned)(nt * (nt + 1) / 2)), dim3(kInvT), 0, s, n, w, ldw, x, ldx);
  return hipGetLastError();
}

#define LLH_INV_INST(T)                                                                                          \
  template hipError_t launch_inv_diag<T>(int, const T*, T*, int64_t, hipStream_t);                               \
  template hipError_t launch_inv_level<T>(int, int, const T*, int64_t, T*, int64_t, T*, hipStream_t);            \
  template hipError_t launch_inv_wtw<T>(int, const T*, int64_t, T*, int64_t, hipStream_t);
LLH_INV_INST(double)
LLH_INV_INST(float)
#undef LLH_INV_INST

}  // namespace llh
