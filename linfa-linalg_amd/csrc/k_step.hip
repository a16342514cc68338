// The panel of the blocked factor: one 64-column step in one launch
// (launch_panel_step), and the rows below a factored top block (launch_panel_rows).
#include "k_diag_impl.h"
#include "k_gemm_impl.h"
#include "llh_kernels.h"

#include <algorithm>

namespace llh {
namespace {

// Up to so many rows below, panel_rows_kernel takes 32 of them a workgroup; beyond it
// 64, whose 256 workgroups fill the chip and read L11 half as often.
constexpr int kRowsNarrow = 16384;

template <typename TS>
constexpr int step_ls() { return kNB + 16 / (int)sizeof(TS); }

template <typename TS, typename T>
union StepLds {
  struct {
    T l[14 * diag_blk<T>()];
    TS lk[kNB * step_ls<TS>()];  // L(k, k-1)
    T conv[4][sizeof(TS) == sizeof(T) ? 1 : diag_blk<T>()];  // a block's change of layout, one per wave
    int fail[kNB / kDiagW];
    int status;
  } c;
  struct {
    NtSlab<TS, 64> as[2];
    NtSlab<TS, 64> bs[2];
  } t;
};

// Launch k of the panel of columns [p0, kend), rows p0 .. n: block column k0, every
// column before k0 - 64 having been applied to columns k0 .. kend.
//
// Chain workgroups (the first max(R, 1), R row blocks below the diagonal block):
// each applies column k - 1 to the diagonal block and factors it itself, so that
// no workgroup waits for another one and the step is one launch instead of
// three; beside the sweeps it applies column k - 1 to its own 64 rows (held
// transposed, in registers) and multiplies them by each column block of the inverse
// once the sweep has it.  Workgroup 0 also stores the inverse (dinv slot k) and L_kk, and
// the status of a failing pivot.  The other workgroups, some of which may start late, still
// read the block that L_kk replaces: L_kk, or what a failing block has of it, waits in
// the next inverse's slot until launch k + 1 copies it (the launch without rows below
// stores it directly).  For the same reason a launch looks at failures before its own
// block only: every workgroup of the launch that fails finds the block and the status as
// they were and does the same, whenever it runs.
// Update workgroups (the rest): apply the columns before k to the panel's later columns,
// one 64 x 64 tile each.  f64: column k - 1.  f32: columns k - 2 and k - 1 at every second
// launch, and at those between column k - 1 to block column k + 1 only, which the next
// launch needs: C is rounded half as often (potrf n = 5003: error 8.8e-8 against 9.9e-8,
// 1767 against 1744 us; in f64 the error is the same, invc n = 3000 1619 against 1587 us).
// An f32 factor with f64 diagonal blocks is refined afterwards and goes the f64 way.
//
// WIDE: eight waves, the rows on four of their own; otherwise four waves, the rows on
// those that do not sweep.  The narrow form fits where a workgroup of the trailing update
// (nt_dma_kernel) has ended, beside the other one of the CU (188 registers of 256, 66.1
// and 65.5 KB of LDS): the wide form, or one of 70 KB, finds no room on a CU until the whole update has
// drained (n = 16384 f64: one step's launch waited 600 to 1800 us).  Beside the update a
// step takes 60 us (its FMAs wait for the other workgroup's f64 MFMAs), alone 19; the
// wide form 17.  solvec n = 1500 765 us with the narrow form alone, 725 with the wide.
//
// What bounds it: latency -- the four sweeps (about 4k cycles each with their
// exchanges), 5k cycles from launch to the last operand, 3k for column k - 1's
// products on the first blocks: 17 us (f64), 13 us (f32) a step for small n,
// where the diagonal kernel, the panel solve and the update took about 36 us.
// potrf with the new diagonal block, three launches -> one (us): n = 1024 f64 493 ->
// 294, f32 423 -> 222; n = 4096 f64 2518 -> 1592, f32 1995 -> 1146.
template <typename TS, typename T, bool VEC, bool WIDE>
__global__ __launch_bounds__(WIDE ? 512 : 256, 2) void panel_step_kernel(TS* a, int64_t lda, int n, int k0, int p0, int kend,
                                                               TS* dinv, int32_t* info, int nchain, int ncol,
                                                               bool copy) {
  __shared__ __attribute__((aligned(16))) StepLds<TS, T> sm;
  constexpr int W = kDiagW, NS = kNB / W, LK = step_ls<TS>();
  const bool prev = k0 > p0;
  const int r0 = k0 + kNB;  // first row below the diagonal block
  if ((int)blockIdx.x >= nchain) {
    if (*info < k0) return;
    const int u = blockIdx.x - nchain, ri = u / ncol, jj = u % ncol;
    if (jj > ri) return;
    const int kw = step_rank<T>(k0, p0);
    const TS* p = a + (int64_t)r0 * lda + (k0 - kw);
    nt_tile_in<TS, 64, 64, 2, WIDE ? 4 : 2, true, VEC, false, TS, false, true>(
        n - r0, kend - r0, kw, TS(-1), p, lda, p, lda, TS(1), a + (int64_t)r0 * lda + r0, lda, 64 * ri, 64 * jj,
        sm.t.as, sm.t.bs);
    return;
  }
  __builtin_amdgcn_s_setprio(3);
  using MS = Mfma<TS>;
  using MT = Mfma<T>;
  const int tid = threadIdx.x, lane = tid & 63, fr = lane & 15, fq = lane >> 4;
  constexpr int NT = WIDE ? 512 : 256;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6), g = wv & 3;
  const bool factor = !WIDE || wv < NS, solver = !WIDE || wv >= NS;
  const int b = min(kNB, n - k0);
  const bool rows = r0 < n, first = blockIdx.x == 0;
  if (tid == 0) sm.c.status = *info;
  TS* const slot = dinv + (int64_t)(k0 / kNB) * kNB * kNB;
  TS* const akk = a + (int64_t)k0 * lda + k0;

  // the diagonal block's strip (negated) and L(k, k-1), which the sweeps wait for
  typename MS::acc_t acc[NS];
  const int myrow = r0 + kNB * (int)blockIdx.x + W * g + fr;  // this lane's row below
  if (factor) diag_load<TS, TS>(akk, lda, b, g, acc);
  constexpr int V = VEC ? 16 / (int)sizeof(TS) : 1;
  typedef TS vs __attribute__((ext_vector_type(V)));
  if (prev) {
    constexpr int PER = kNB * kNB / V / NT;
#pragma unroll
    for (int e = 0; e < PER; ++e) {
      const int idx = tid + NT * e, row = idx / (kNB / V), c = (idx % (kNB / V)) * V;
      vs v = *reinterpret_cast<const vs*>(a + (int64_t)min(k0 + row, n - 1) * lda + (k0 - kNB) + c);
      if (k0 + row >= n) v = vs{};  // (a block row beyond n stays the identity's)
      *reinterpret_cast<vs*>(&sm.c.lk[row * LK + c]) = v;
    }
  }
  // the rows below, transposed, and their column k - 1 (16 k values of this lane):
  // scattered loads, behind those that the first sweep waits for
  asm volatile("" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
  typename MS::acc_t xt[NS];
  TS m[W];
  if (rows && solver) {
    const TS* src = a + (int64_t)min(myrow, n - 1) * lda + k0;
#pragma unroll
    for (int c = 0; c < NS; ++c)
#pragma unroll
      for (int r = 0; r < 4; ++r) xt[c][r] = -src[W * c + MS::row(lane, r)];
    if (prev) {
#pragma unroll
      for (int s = 0; s < W; s += V) {
        const vs v = *reinterpret_cast<const vs*>(src + W * fq + s - kNB);
#pragma unroll
        for (int e = 0; e < V; ++e) m[s + e] = v[e];
      }
    }
  }
  TS lprev[kNB * kNB / NT];
  if (copy && first) {
#pragma unroll
    for (int e = 0; e < kNB * kNB / NT; ++e) lprev[e] = slot[tid + NT * e];
  }
  diag_barrier();
  const int status = sm.c.status;
  if (copy && first) {
    // L_(k-1)(k-1) from this block's slot, read above, to its place; of a block that failed
    // at row `last` the rows before it and L[last, ..last] (an earlier failure: nothing)
    const int last = status < k0 ? status - (k0 - kNB) : kNB;
    TS* dst = a + (int64_t)(k0 - kNB) * lda + (k0 - kNB);
#pragma unroll
    for (int e = 0; e < kNB * kNB / NT; ++e) {
      const int idx = tid + NT * e, row = idx / kNB, col = idx % kNB;
      if (row < last ? col <= row : row == last && col < row) dst[(int64_t)row * lda + col] = lprev[e];
    }
  }
  if (status < k0) return;

  // L(k, k-1)'s strip c times this wave's strip (!left) or the transposed rows (left),
  // added to x, summed by itself first: added term by term, every partial sum would
  // be rounded at the size of x (n = 512, f64: error of L 2.6e-16 against 1.8e-16).
  auto apply = [&](typename MS::acc_t& x, int c, auto left) __attribute__((always_inline)) {
    typename MS::acc_t t;
#pragma unroll
    for (int r = 0; r < 4; ++r) t[r] = TS(0);
#pragma unroll
    for (int s = 0; s < W; ++s) {
      const TS v = sm.c.lk[(W * c + fr) * LK + W * fq + s];
      if constexpr (decltype(left)::value)
        t = MS::mma(v, m[s], t);
      else
        t = MS::mma(sm.c.lk[(W * g + fr) * LK + W * fq + s], v, t);
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) x[r] += t[r];
  };
  using Left = std::true_type;
  using Diag = std::false_type;
  // a block in T's result layout, through LDS
  auto to_t = [&](typename MT::acc_t& y, const typename MS::acc_t& x) __attribute__((always_inline)) {
    T* t = sm.c.conv[g];
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int r = 0; r < 4; ++r) t[MS::row(lane, r) * diag_ls<T>() + fr] = T(x[r]);
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int r = 0; r < 4; ++r) y[r] = t[MT::row(lane, r) * diag_ls<T>() + fr];
  };
  constexpr bool kSame = sizeof(TS) == sizeof(T);
  typename MT::acc_t conv[kSame ? 1 : NS];
  auto& tacc = [&]() -> auto& {
    if constexpr (kSame)
      return acc;
    else
      return conv;
  }();
  if (factor) {
    if (prev) apply(acc[0], 0, Diag{});
    if constexpr (!kSame) {
#pragma unroll
      for (int c = 0; c < NS; ++c) to_t(tacc[c], acc[c]);
    }
  }
  // column block c of the rows: X^T_c = sum_{j <= c} inv(L_kk)_cj A^T_j
  auto solve = [&](int c) __attribute__((always_inline)) {
    typename MS::acc_t x;
#pragma unroll
    for (int r = 0; r < 4; ++r) x[r] = TS(0);
    const T* p = diag_rows(sm.c.l, c);
#pragma unroll
    for (int j = 0; j < NS; ++j)
      if (j <= c) {
#pragma unroll
        for (int s = 0; s < 4; ++s)
          x = MS::mma(TS(p[j * diag_blk<T>() + MS::row(lane, s) * diag_ls<T>() + fr]), xt[j][s], x);
      }
    if (myrow < n) {
      TS* dst = a + (int64_t)myrow * lda + k0 + W * c;
#pragma unroll
      for (int r = 0; r < 4; ++r) dst[MS::row(lane, r)] = -x[r];
    }
  };
  const int fail = diag_core<T, WIDE>(
      tacc, wv, sm.c.l, sm.c.fail,
      [&](int w, int it, int f) __attribute__((always_inline)) {
        // L_kk beside the block while others may read it
        if (first) diag_put<TS, T>(sm.c.l, w, it, f, b, rows ? slot + kNB * kNB : akk, rows ? kNB : lda, slot);
      },
      // The rows, on the waves that have time: strips that column k - 1 is applied to
      // and column blocks solved beside sweep w, as masks (4 bits per sweep, 16 per
      // wave).  A column block is solved within two sweeps of its own.
      [&](int w) __attribute__((always_inline)) {
        if (!rows) return;
        constexpr uint64_t kApply = WIDE ? 0x0c21ull << 48 | 0x8061ull << 32 | 0x8403ull << 16 | 0x8430ull
                                         : 0x0843ull << 48 | 0xc021ull << 32 | 0xc201ull << 16 | 0x8430ull;
        constexpr uint64_t kSolve = WIDE ? 0x4210ull * 0x0001000100010001ull
                                         : 0x0210ull << 48 | 0x6010ull << 32 | 0x4300ull << 16 | 0x4210ull;
        const int sh = 16 * g + 4 * w;
        if (prev) {
          const uint32_t todo = (uint32_t)(kApply >> sh);
#pragma unroll
          for (int c = 0; c < NS; ++c)
            if (todo & (1u << c)) {
              asm volatile("; rows' strip %0" ::"n"(c));
              apply(xt[c], c, Left{});
            }
        }
        const uint32_t todo = (uint32_t)(kSolve >> sh);
#pragma unroll
        for (int c = 0; c < NS - 1; ++c)
          if (todo & (1u << c)) {
            asm volatile("; rows' column %0" ::"n"(c));
            solve(c);
          }
      },
      // Column k - 1 applied to the diagonal block's column block w + 1.
      [&](int w, typename MT::acc_t& x) __attribute__((always_inline)) {
        if (!prev) return;
        if constexpr (kSame) {
          apply(x, w + 1, Diag{});
        } else {
          typename MS::acc_t t;
          typename MT::acc_t y;
#pragma unroll
          for (int r = 0; r < 4; ++r) t[r] = TS(0);
          apply(t, w + 1, Diag{});
          to_t(y, t);
#pragma unroll
          for (int r = 0; r < 4; ++r) x[r] += y[r];
        }
      });
  if (fail >= 0) {
    if (first && tid == 0) atomicMin(info, (int32_t)(k0 + fail));
    return;
  }
  if (rows && solver) {
    if (!WIDE && g == NS - 1) solve(NS - 2);
    solve(NS - 1);
  }
}

// L21 = A21 L11^-T for the rows below a panel whose kb x kb top block [k0, k0 + kb)
// is factored (dinv: the inverses of all diagonal blocks): one workgroup per 64
// rows walks the panel's 64-column blocks,
//   X_k = (A_k - sum_{j < k} X_j L_kj^T) inv(L_kk)^T,
// the sum as one product of rank 64 k over its own rows of the columns left of k,
// which it has just stored.  Workgroups depend on the top block only, so the
// chain of a panel is its top block's, whatever the rows below, and this launch.
//
// What bounds it: the latency of a slab's loads (kb^2 / 128 of 64 columns each, one
// after the other); hence 256 bytes a row and slab, and 32 rows a workgroup (MT = 2), so
// that every CU has one up to kRowsNarrow rows; the inverse's rows and A_k are loaded
// before the sum.  Its registers and LDS, like a narrow step's, fit where a workgroup
// of the trailing update has ended.  8448 x 512 f64: 119 us with 64 rows, 16 columns a
// slab and eight waves; this form 71 us alone, 110 to 190 beside the update.  Under the
// register bound that lets it fit, the f64 form of 64 rows spills 22 to 24 of them
// (n = 32768: 1681 us a launch beside the update).  potrf
// against the recursion of 64-wide panels (ms): f64 n = 16384 29.5 -> 29.0, f32 n = 12000
// 8.65 -> 8.40, 16384 18.1 -> 17.4.
template <typename T, bool VEC, int MT>
__global__ __launch_bounds__(256, 2) __attribute__((amdgpu_num_vgpr(108))) void panel_rows_kernel(T* a, int64_t lda, int n, int k0, int kb,
                                                            const T* __restrict__ dinv,
                                                            const int32_t* __restrict__ gate) {
  using MF = Mfma<T>;
  using acc_t = typename MF::acc_t;
  constexpr int KPL = 16 / sizeof(T), SUB = 4 * KPL, SK = (MT == 2 ? 4 : 2) * SUB, LDK = SK + KPL, TS = kNB + KPL;
  constexpr int RS = 16 * MT, PR = SK / KPL, NA = RS * PR / 256, NBP = kNB * PR / 256;
  typedef T vec_t __attribute__((ext_vector_type(KPL)));
  __shared__ __attribute__((aligned(16))) union {
    struct {
      T as[2][RS * LDK], bs[2][kNB * LDK];
    } s;
    T ts[RS * TS];
  } sm;
  if (*gate != kNoFail) return;
  __builtin_amdgcn_s_setprio(3);
  const int tid = threadIdx.x, lane = tid & 63, fr = lane & 15, fq = lane >> 4;
  const int wn = (tid >> 6) * 16;
  const int r0 = k0 + kb + RS * (int)blockIdx.x;
  // this thread's pieces of a slab: rows srow, srow + 256 / PR, .., k sk .. sk + KPL
  const int srow = tid / PR, sk = (tid % PR) * KPL;
  // (byte offsets from wave-uniform bases; VEC: below 2^32, see launch_panel_rows)
  using off_t = std::conditional_t<VEC, uint32_t, int64_t>;
  const off_t pitch = (off_t)lda * (off_t)sizeof(T);
  off_t oa[NA], ob[NBP];
#pragma unroll
  for (int e = 0; e < NA; ++e)
    oa[e] = (off_t)min(srow + 256 / PR * e, n - 1 - r0) * pitch + (off_t)(sk * (int)sizeof(T));
#pragma unroll
  for (int e = 0; e < NBP; ++e) ob[e] = (off_t)(srow + 256 / PR * e) * pitch + (off_t)(sk * (int)sizeof(T));
  auto fetch = [&](const T* base, off_t off) __attribute__((always_inline)) -> vec_t {
    const T* p = reinterpret_cast<const T*>(reinterpret_cast<const char*>(base) + off);
    vec_t v;
    if constexpr (VEC) {
      v = *reinterpret_cast<const vec_t*>(p);
    } else {
#pragma unroll
      for (int e = 0; e < KPL; ++e) v[e] = p[e];
    }
    return v;
  };
  for (int kc = 0; kc < kb; kc += kNB) {
    vec_t ra[NA], rb[NBP];
    auto load = [&](int k) __attribute__((always_inline)) {
      const T *pa = a + (int64_t)r0 * lda + k0 + k, *pb = a + (int64_t)(k0 + kc) * lda + k0 + k;
#pragma unroll
      for (int e = 0; e < NA; ++e) ra[e] = fetch(pa, oa[e]);
#pragma unroll
      for (int e = 0; e < NBP; ++e) rb[e] = fetch(pb, ob[e]);
    };
    auto put = [&](int buf) __attribute__((always_inline)) {
#pragma unroll
      for (int e = 0; e < NA; ++e) *reinterpret_cast<vec_t*>(&sm.s.as[buf][(srow + 256 / PR * e) * LDK + sk]) = ra[e];
#pragma unroll
      for (int e = 0; e < NBP; ++e) *reinterpret_cast<vec_t*>(&sm.s.bs[buf][(srow + 256 / PR * e) * LDK + sk]) = rb[e];
    };
    if (kc > 0) load(0);
    // this lane's entries of A_k and row of the inverse, used after the sum
    T cv[MT][4];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        cv[i][r] = *reinterpret_cast<const T*>(
            reinterpret_cast<const char*>(a + (int64_t)r0 * lda + k0 + kc) +
            (off_t)min(16 * i + MF::row(lane, r), n - 1 - r0) * pitch + (off_t)((wn + fr) * (int)sizeof(T)));
    vec_t iv[kNB / SUB];
    const T* inv = dinv + (int64_t)((k0 + kc) / kNB) * kNB * kNB + (wn + fr) * kNB + KPL * fq;
#pragma unroll
    for (int c = 0; c < kNB / SUB; ++c) iv[c] = *reinterpret_cast<const vec_t*>(inv + c * SUB);
    acc_t acc[MT];
#pragma unroll
    for (int i = 0; i < MT; ++i) acc[i] = acc_t{0, 0, 0, 0};
    if (kc > 0) {
      put(0);
      __syncthreads();
      for (int k = 0, buf = 0; k < kc; k += SK, buf ^= 1) {
        const bool more = k + SK < kc;
        if (more) load(k + SK);
#pragma unroll
        for (int c = 0; c < SK; c += SUB) {
          const vec_t bf = *reinterpret_cast<const vec_t*>(&sm.s.bs[buf][(wn + fr) * LDK + c + KPL * fq]);
          vec_t af[MT];
#pragma unroll
          for (int i = 0; i < MT; ++i)
            af[i] = *reinterpret_cast<const vec_t*>(&sm.s.as[buf][(16 * i + fr) * LDK + c + KPL * fq]);
#pragma unroll
          for (int e = 0; e < KPL; ++e)
#pragma unroll
            for (int i = 0; i < MT; ++i) acc[i] = MF::mma(af[i][e], bf[e], acc[i]);
        }
        if (more) put(buf ^ 1);
        __syncthreads();
      }
    }
    // the tile through LDS (the slabs' memory, free after the loop's last barrier)
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) sm.ts[(16 * i + MF::row(lane, r)) * TS + wn + fr] = cv[i][r] - acc[i][r];
    __syncthreads();
    acc_t x[MT];
#pragma unroll
    for (int i = 0; i < MT; ++i) x[i] = acc_t{0, 0, 0, 0};
#pragma unroll
    for (int c = 0; c < kNB / SUB; ++c) {
      vec_t af[MT];
#pragma unroll
      for (int i = 0; i < MT; ++i)
        af[i] = *reinterpret_cast<const vec_t*>(&sm.ts[(16 * i + fr) * TS + c * SUB + KPL * fq]);
#pragma unroll
      for (int e = 0; e < KPL; ++e)
#pragma unroll
        for (int i = 0; i < MT; ++i) x[i] = MF::mma(af[i][e], iv[c][e], x[i]);
    }
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = r0 + 16 * i + MF::row(lane, r);
        if (row < n)
          *reinterpret_cast<T*>(reinterpret_cast<char*>(a + (int64_t)r0 * lda + k0 + kc) +
                                (off_t)(16 * i + MF::row(lane, r)) * pitch +
                                (off_t)((wn + fr) * (int)sizeof(T))) = x[i][r];
      }
    __syncthreads();  // X_k is stored (the next block's sum reads it), ts is read
  }
}

}  // namespace

template <typename TS, typename T>
hipError_t launch_panel_step(TS* a, int64_t lda, int n, int k0, int p0, int kend, TS* dinv, int32_t* info,
                             bool copy_prev, bool beside, hipStream_t s) {
  if (k0 < p0 || k0 >= kend || kend > n || k0 % kNB != 0 || p0 % kNB != 0) return hipErrorInvalidValue;
  const int below = n - k0 - kNB;
  const int rb = below > 0 ? (below + kNB - 1) / kNB : 0;
  const int nchain = rb > 0 ? rb : 1;
  const int later = k0 > p0 && kend > k0 + kNB ? (kend - k0 - 1) / kNB : 0;
  const int ncol = step_ahead<T>(k0, p0) ? std::min(later, 1) : later;
  const dim3 grid(nchain + rb * ncol);
  const bool vec = reinterpret_cast<uintptr_t>(a) % 16 == 0 && (lda * sizeof(TS)) % 16 == 0;
#define LLH_STEP_GO(VEC, WIDE)                                                                                    \
  hipLaunchKernelGGL((panel_step_kernel<TS, T, VEC, WIDE>), grid, dim3(WIDE ? 512 : 256), 0, s, a, lda, n, k0, p0, \
                     kend, dinv, info, nchain, ncol, copy_prev)
  if (beside) {
    if (vec) LLH_STEP_GO(true, false);
    else LLH_STEP_GO(false, false);
  } else {
    if (vec) LLH_STEP_GO(true, true);
    else LLH_STEP_GO(false, true);
  }
#undef LLH_STEP_GO
  return hipGetLastError();
}

template <typename T>
hipError_t launch_panel_rows(T* a, int64_t lda, int n, int k0, int kb, const T* dinv, const int32_t* gate,
                             hipStream_t s) {
  const int below = n - k0 - kb;
  if (below <= 0) return hipSuccess;
  if (k0 % kNB != 0 || kb % kNB != 0 || gate == nullptr) return hipErrorInvalidValue;
  const bool vec = reinterpret_cast<uintptr_t>(a) % 16 == 0 && (lda * sizeof(T)) % 16 == 0 &&
                   lda * (int64_t)sizeof(T) < ((int64_t)1 << 26);
#define LLH_ROWS_GO(VEC, MT)                                                                                        \
  hipLaunchKernelGGL((panel_rows_kernel<T, VEC, MT>), dim3((below + 16 * MT - 1) / (16 * MT)), dim3(256), 0, s, a, \
                     lda, n, k0, kb, dinv, gate)
  if (below <= kRowsNarrow) {
    if (vec) LLH_ROWS_GO(true, 2);
    else LLH_ROWS_GO(false, 2);
  } else {
    if (vec) LLH_ROWS_GO(true, 4);
    else LLH_ROWS_GO(false, 4);
  }
#undef LLH_ROWS_GO
  return hipGetLastError();
}

template hipError_t launch_panel_rows<double>(double*, int64_t, int, int, int, const double*, const int32_t*,
                                              hipStream_t);
template hipError_t launch_panel_rows<float>(float*, int64_t, int, int, int, const float*, const int32_t*,
                                             hipStream_t);
template hipError_t launch_panel_step<double, double>(double*, int64_t, int, int, int, int, double*, int32_t*, bool, bool, hipStream_t);
template hipError_t launch_panel_step<float, float>(float*, int64_t, int, int, int, int, float*, int32_t*, bool, bool, hipStream_t);
template hipError_t launch_panel_step<float, double>(float*, int64_t, int, int, int, int, float*, int32_t*, bool, bool, hipStream_t);

}  // namespace llh
