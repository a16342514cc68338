// One 64-column step of a panel of the blocked factor in one launch
// (launch_panel_step).
#include "k_diag_impl.h"
#include "k_gemm_impl.h"
#include "llh_kernels.h"

namespace llh {
namespace {

// Eight waves: four factor the diagonal block, four carry the workgroup's rows.
constexpr int kStepT = 512;

template <typename TS>
constexpr int step_ls() { return kNB + 16 / (int)sizeof(TS); }

template <typename TS, typename T>
union StepLds {
  struct {
    union {
      T l[14 * diag_blk<T>()];
      TS ai[kNB * step_ls<TS>()];  // the workgroup's rows of column k (before the sweeps)
    };
    TS lk[kNB * step_ls<TS>()];  // L(k, k-1)
    TS li[kNB * step_ls<TS>()];  // the workgroup's rows of column k - 1
    T conv[sizeof(TS) == sizeof(T) ? 1 : 4][diag_blk<T>()];  // a block's change of layout, one per wave
    int fail[kNB / kDiagW];
    int skip;
  } c;
  struct {
    NtSlab<TS, 64> as[2];
    NtSlab<TS, 64> bs[2];
  } t;
};

// Launch k of a panel [p0, kend): block column k0, every column before k0 - 64
// having been applied to columns k0 .. kend.
//
// Chain workgroups (the first max(R, 1), R row blocks below the diagonal block):
// each applies column k - 1 to the diagonal block and factors it itself, so that
// no workgroup waits for another one and the step is one launch instead of
// three; beside it the other four waves apply column k - 1 to the workgroup's own
// 64 rows (held transposed, in registers) and multiply them by each column block
// of the inverse as soon as the sweep has it.  Workgroup 0 also stores the
// inverse (dinv slot k) and L_kk.  The other workgroups still read the block
// that L_kk replaces, so L_kk waits in the next inverse's slot until launch k + 1
// copies it (the launch without rows below stores it directly).
// Update workgroups (the rest): apply column k - 1 to the panel's later columns,
// one 64 x 64 tile each.
//
// What bounds it: latency -- the four sweeps (about 4k cycles each with their
// exchanges), 5k cycles from launch to the last operand, 3k for column k - 1's
// products on the first blocks: 17.5 us (f64), 13.4 us (f32) a step for small n,
// where the diagonal kernel, the panel solve and the update took about 36 us.
// potrf with the new diagonal block, three launches -> one (us): n = 1024 f64 493 ->
// 294, f32 423 -> 222; n = 4096 f64 2518 -> 1592, f32 1995 -> 1146.
template <typename TS, typename T, bool VEC>
__global__ __launch_bounds__(kStepT, 2) void panel_step_kernel(TS* a, int64_t lda, int n, int k0, int p0, int kend,
                                                               TS* dinv, int32_t* info, int nchain, int ncol,
                                                               bool copy) {
  __shared__ __attribute__((aligned(16))) StepLds<TS, T> sm;
  constexpr int W = kDiagW, NS = kNB / W, LK = step_ls<TS>();
  const bool prev = k0 > p0;
  const int r0 = k0 + kNB;  // first row below the diagonal block
  if ((int)blockIdx.x >= nchain) {
    if (*info != kNoFail) return;
    const int u = blockIdx.x - nchain, ri = u / ncol, jj = u % ncol;
    if (jj > ri) return;
    const TS* p = a + (int64_t)r0 * lda + (k0 - kNB);
    nt_tile_in<TS, 64, 64, 2, 4, true, VEC, sizeof(TS) == 8>(n - r0, kend - r0, kNB, TS(-1), p, lda, p, lda, TS(1),
                                                             a + (int64_t)r0 * lda + r0, lda, 64 * ri, 64 * jj,
                                                             sm.t.as, sm.t.bs);
    return;
  }
  using MS = Mfma<TS>;
  using MT = Mfma<T>;
  const int tid = threadIdx.x, lane = tid & 63, fr = lane & 15, fq = lane >> 4;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6), g = wv & 3;
  const int b = min(kNB, n - k0);
  const bool rows = r0 < n, first = blockIdx.x == 0;
  if (tid == 0) sm.c.skip = *info != kNoFail;
  TS* const slot = dinv + (int64_t)(k0 / kNB) * kNB * kNB;
  TS* const akk = a + (int64_t)k0 * lda + k0;

  // the diagonal block's strips (factor waves; negated); the other operands are
  // staged through LDS by whole rows
  typename MS::acc_t acc[NS];
  const int row0 = r0 + kNB * (int)blockIdx.x;      // the workgroup's rows
  const int myrow = row0 + W * g + fr;              // this lane's (helper waves)
  if (wv < NS) diag_load<TS, TS>(akk, lda, b, g, acc);
  auto stage = [&](int src_row, int col, TS* dst) __attribute__((always_inline)) {
    constexpr int V = VEC ? 16 / (int)sizeof(TS) : 1, PER = kNB * kNB / V / kStepT;
    typedef TS vs __attribute__((ext_vector_type(V)));
#pragma unroll
    for (int e = 0; e < PER; ++e) {
      const int idx = tid + kStepT * e, row = idx / (kNB / V), c = (idx % (kNB / V)) * V;
      vs v = *reinterpret_cast<const vs*>(a + (int64_t)min(src_row + row, n - 1) * lda + col + c);
      if (src_row + row >= n) v = vs{};  // (a block row beyond n stays the identity's)
      *reinterpret_cast<vs*>(&dst[row * LK + c]) = v;
    }
  };
  if (prev) stage(k0, k0 - kNB, sm.c.lk);
  if (rows) {
    stage(row0, k0, sm.c.ai);
    if (prev) stage(row0, k0 - kNB, sm.c.li);
  }
  TS lprev[kNB * kNB / kStepT];
  if (copy && first) {
#pragma unroll
    for (int e = 0; e < kNB * kNB / kStepT; ++e) lprev[e] = slot[tid + kStepT * e];
  }
  __syncthreads();
  if (sm.c.skip) return;
  if (copy && first) {
    // L_(k-1)(k-1) from this block's slot, read above, to its place
    TS* dst = a + (int64_t)(k0 - kNB) * lda + (k0 - kNB);
#pragma unroll
    for (int e = 0; e < kNB * kNB / kStepT; ++e) {
      const int idx = tid + kStepT * e, row = idx / kNB, col = idx % kNB;
      if (col <= row) dst[(int64_t)row * lda + col] = lprev[e];
    }
  }

  // The product of L(k, k-1)'s strip c with operand m (16 k values of this lane:
  // 16 fq + s), added to x.  In f32 it is summed by itself first: added term by
  // term, every partial sum would be rounded at the size of x.
  auto apply = [&](typename MS::acc_t& x, int c, const TS (&m)[W], bool left) __attribute__((always_inline)) {
    typename MS::acc_t t;
#pragma unroll
    for (int r = 0; r < 4; ++r) t[r] = sizeof(TS) == 8 ? x[r] : TS(0);
#pragma unroll
    for (int s = 0; s < W; ++s) {
      const TS v = sm.c.lk[(W * c + fr) * LK + W * fq + s];
      t = left ? MS::mma(v, m[s], t) : MS::mma(m[s], v, t);
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) x[r] = sizeof(TS) == 8 ? t[r] : x[r] + t[r];
  };
  // a factor wave's block in T's result layout (through LDS when the layouts differ)
  auto to_t = [&](typename MT::acc_t& y, const typename MS::acc_t& x) __attribute__((always_inline)) {
    if constexpr (sizeof(TS) == sizeof(T)) {
#pragma unroll
      for (int r = 0; r < 4; ++r) y[r] = x[r];
    } else {
      T* t = sm.c.conv[g];
      __builtin_amdgcn_wave_barrier();
#pragma unroll
      for (int r = 0; r < 4; ++r) t[MS::row(lane, r) * diag_ls<T>() + fr] = T(x[r]);
      __builtin_amdgcn_wave_barrier();
#pragma unroll
      for (int r = 0; r < 4; ++r) y[r] = t[MT::row(lane, r) * diag_ls<T>() + fr];
    }
  };
  typename MT::acc_t tacc[NS];
  TS m[W];  // factor waves: this lane's row of L(k, k-1); the others: of the workgroup's rows' column k - 1
#pragma unroll
  for (int s = 0; s < W; ++s) m[s] = TS(0);
  if (wv < NS) {
    if (prev) {
#pragma unroll
      for (int s = 0; s < W; ++s) m[s] = sm.c.lk[(W * g + fr) * LK + W * fq + s];
      apply(acc[0], 0, m, false);
    }
#pragma unroll
    for (int c = 0; c < NS; ++c) to_t(tacc[c], acc[c]);
  } else if (rows) {
    // the rows, transposed and negated
#pragma unroll
    for (int c = 0; c < NS; ++c)
#pragma unroll
      for (int r = 0; r < 4; ++r) acc[c][r] = -sm.c.ai[(W * g + fr) * LK + W * c + MS::row(lane, r)];
    if (prev) {
#pragma unroll
      for (int s = 0; s < W; ++s) m[s] = sm.c.li[(W * g + fr) * LK + W * fq + s];
    }
  }
  diag_barrier();  // ai is read: its memory is the sweeps' now
  // column block c of the rows: X^T_c = sum_{j <= c} inv(L_kk)_cj A^T_j
  auto solve = [&](int c) __attribute__((always_inline)) {
    if (!rows) return;
    typename MS::acc_t x;
#pragma unroll
    for (int r = 0; r < 4; ++r) x[r] = TS(0);
    const T* p = diag_rows(sm.c.l, c);
#pragma unroll
    for (int j = 0; j < NS; ++j)
      if (j <= c) {
#pragma unroll
        for (int s = 0; s < 4; ++s)
          x = MS::mma(TS(p[j * diag_blk<T>() + MS::row(lane, s) * diag_ls<T>() + fr]), acc[j][s], x);
      }
    if (myrow < n) {
      TS* dst = a + (int64_t)myrow * lda + k0 + W * c;
#pragma unroll
      for (int r = 0; r < 4; ++r) dst[MS::row(lane, r)] = -x[r];
    }
  };
  const int fail = diag_core<T>(
      tacc, wv, sm.c.l, sm.c.fail,
      [&](int w, int it, int f) __attribute__((always_inline)) {
        if (!first) return;
        // L_kk beside the block while others may read it; a failing block's rows
        // go to their place (nothing after this launch reads the block)
        if (f >= 0) {
          diag_put<TS, T>(sm.c.l, w, it, f, b, akk, lda, slot);
        } else {
          diag_put<TS, T>(sm.c.l, w, it, f, b, rows ? slot + kNB * kNB : akk, rows ? kNB : lda, slot);
        }
      },
      // Beside sweep w: the rows' column block w - 1 solved, and column k - 1 applied
      // to the later ones, but not beside the sweep of the wave on the same SIMD
      // (f64 products and the sweep's f64 FMAs share its pipe).
      [&](int w) __attribute__((always_inline)) {
        if (rows && prev && w != g) {
          const int from = w == 0 ? 0 : w + (w == g + 1 && g == 0 ? -1 : 0), to = w + 1 + (w + 1 == g);
#pragma unroll
          for (int c = 0; c < NS; ++c)
            if (c >= from && c < to) {
              asm volatile("; rows' column %0" ::"n"(c));
              apply(acc[c], c, m, true);
            }
        }
        if (w > 0) solve(w - 1);
      },
      // Column k - 1 applied to the diagonal block's column block w + 1.
      [&](int w, typename MT::acc_t& x) __attribute__((always_inline)) {
        if (!prev) return;
        if constexpr (sizeof(TS) == sizeof(T)) {
          apply(x, w + 1, m, false);
        } else {
          typename MS::acc_t t;
          typename MT::acc_t y;
#pragma unroll
          for (int r = 0; r < 4; ++r) t[r] = TS(0);
          apply(t, w + 1, m, false);
          to_t(y, t);
#pragma unroll
          for (int r = 0; r < 4; ++r) x[r] += y[r];
        }
      });
  if (fail >= 0) {
    if (first) {
      if (rows) {
        // the columns of the steps before the failing one, stored beside the block
        const int w = fail / W;
        __syncthreads();
        for (int e = tid; e < kNB * W * w; e += kStepT) {
          const int row = e / (W * w), col = e % (W * w);
          if (col <= row && row <= fail) akk[(int64_t)row * lda + col] = slot[kNB * kNB + row * kNB + col];
        }
      }
      if (tid == 0) atomicMin(info, (int32_t)(k0 + fail));
    }
    return;
  }
  if (wv >= NS) solve(NS - 1);
}

}  // namespace

template <typename TS, typename T>
hipError_t launch_panel_step(TS* a, int64_t lda, int n, int k0, int p0, int kend, TS* dinv, int32_t* info,
                             bool copy_prev, hipStream_t s) {
  if (k0 < p0 || k0 >= n || kend > n || k0 % kNB != 0 || p0 % kNB != 0) return hipErrorInvalidValue;
  const int below = n - k0 - kNB;
  const int rb = below > 0 ? (below + kNB - 1) / kNB : 0;
  const int nchain = rb > 0 ? rb : 1;
  const int ncol = k0 > p0 && kend > k0 + kNB ? (kend - k0 - kNB + kNB - 1) / kNB : 0;
  const dim3 grid(nchain + rb * ncol), block(kStepT);
  const bool vec = reinterpret_cast<uintptr_t>(a) % 16 == 0 && (lda * sizeof(TS)) % 16 == 0;
  if (vec)
    hipLaunchKernelGGL((panel_step_kernel<TS, T, true>), grid, block, 0, s, a, lda, n, k0, p0, kend, dinv, info,
                       nchain, ncol, copy_prev);
  else
    hipLaunchKernelGGL((panel_step_kernel<TS, T, false>), grid, block, 0, s, a, lda, n, k0, p0, kend, dinv, info,
                       nchain, ncol, copy_prev);
  return hipGetLastError();
}

template hipError_t launch_panel_step<double, double>(double*, int64_t, int, int, int, int, double*, int32_t*, bool,
                                                      hipStream_t);
template hipError_t launch_panel_step<float, float>(float*, int64_t, int, int, int, int, float*, int32_t*, bool,
                                                    hipStream_t);
template hipError_t launch_panel_step<float, double>(float*, int64_t, int, int, int, int, float*, int32_t*, bool,
                                                     hipStream_t);

}  // namespace llh
