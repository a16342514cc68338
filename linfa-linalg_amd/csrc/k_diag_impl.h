// Device code of the fast factor + inverse of one 64 x 64 diagonal block,
// shared by the blocked paths' kernels (k_diag.hip) and the fused batched
// kernel (k_batch.hip).  The trailing updates of the blocked paths round
// differently from the reference anyway, so the block may too; small whole
// matrices keep the exact-order kernel.
//
// Four waves; wave g holds the 16-row strip g of [A; I] in MFMA result layout:
// the blocks (g, c), c <= g, of A and, for c > g, those of the identity rows g
// (the rows of L^-T, which are zero up to block g).  The block is factored in four
// steps of 16 columns.  In step w every strip publishes its column block w to
// LDS and wave w sweeps the 16 columns once for all of them: each of its four
// 16-lane groups holds a copy of the diagonal block (lane = row) and the rows of
// one strip, and takes the pivot and each L[q, j] from its own group by DPP row
// broadcasts, so a column costs one reciprocal square root and two FMAs per
// later column, whichever strip the rows belong to.  Strip w's rows are the
// identity there, so the same sweep yields inv(L_ww) and, with the strips left
// of w, block row w of the inverse.  Then every wave subtracts its strip's
// 16 x 16 product from its next column block (MFMA), publishes it, and does the
// products for the later blocks and the step's global stores while the next
// sweep runs.  A strip has four blocks in every step, so the inverse costs no
// sweep of its own.
//
// What bounds it: the chain of 64 pivots on one wave (latency), about 2.5k cycles
// per 16 columns (about 400 instructions at ~7 cycles each).  One block alone in
// f64: 19.0 -> 10.4 us against a column chain through v_readlane with the trailing
// work on the VALU and the inverse after the factor; potrf n = 512 290 -> 214 us
// f64, 255 -> 190 us f32; the 20000-system batch 8.80 -> 8.51 ms.
//
// Rows beyond b are identity rows, so the block factors to diag(L, I) and its
// inverse likewise.  Pivot test and failure row follow cholesky.rs:54-74: on a
// failure at row f the block holds rows < f and L[f, ..f] (rows beyond f hold the
// columns of the steps before the failing one).
#pragma once

#include <type_traits>
#include <utility>

#include "k_gemm_impl.h"
#include "llh_common.h"

namespace llh {

// The instructions of a sweep's column, as blocks of volatile asm that issue in
// the order given.  row_newbcast:Q is the DPP broadcast of lane Q of each group of
// 16 lanes; the compiler would split a broadcast FMA into a move and a dependent
// FMA (17 cycles a pair on one wave, against 7.4 for the single instruction) and
// pad between shorter blocks.  Kept here by hand: two instructions between the
// write of a VGPR and its use as a DPP source, one between v_rsq and its use.
//
// 1 / sqrt(d) of a pivot d > 0 goes in kSteps steps that are issued between the
// updates of later columns: the hardware reciprocal square root and, in f64, one
// third-order step y (1 + e/2 + 3 e^2 / 8), e = 1 - d y^2 (the hardware value is good
// to ~3e-8, so the next term is below 1e-22), in f32 one Newton step
// y (3/2 - d y^2 / 2).  Within an ulp or two, which the blocked factor's tolerance
// admits (the exact-order kernel keeps the reference's square root and division).
template <typename T>
struct SweepCol;

#define LLH_DPP(Q) " row_newbcast:" Q " row_mask:0xf bank_mask:0xf"
// %0 y / t / u of the step, %1 d[q], %2 p[q], then the step's inputs
#define LLH_SWEEP_TYPE(T, SFX, MOV)                                                                               \
  template <>                                                                                                    \
  struct SweepCol<T> {                                                                                           \
    T d, y, t, u; /* the pivot, its reciprocal root, intermediate values */                                        \
    /* the first pivot: broadcast, and its sign test */                                                           \
    __device__ __forceinline__ uint64_t first(T d0) {                                                            \
      uint64_t m;                                                                                                \
      asm volatile("s_nop 1\n\tv_cmp_ge_" SFX " %0, 0, %2\n\tv_mov_" MOV "_dpp %1, %2" LLH_DPP("0")             \
                   : "=&s"(m), "=&v"(d)                                                                          \
                   : "v"(d0));                                                                                   \
      return m;                                                                                                  \
    }                                                                                                            \
    /* column j scaled by 1 / sqrt(pivot) */                                                                      \
    __device__ __forceinline__ void scale(T& dj, T& pj) {                                                        \
      asm volatile("v_mul_" SFX " %0, %0, %2\n\tv_mul_" SFX " %1, %1, %2" : "+v"(dj), "+v"(pj) : "v"(y));        \
    }                                                                                                            \
    /* the same, then column q = j + 1 updated, and its pivot */                                                  \
    template <int Q>                                                                                             \
    __device__ __forceinline__ uint64_t next(T& dj, T& pj, T& dq, T& pq) {                                       \
      uint64_t m;                                                                                                \
      asm volatile(                                                                                              \
          "v_mul_" SFX " %0, %0, %6\n\tv_mul_" SFX " %1, %1, %6\n\ts_nop 0\n\t"                                 \
          "v_fmac_" SFX "_dpp %2, %0, -%0" LLH_DPP("%7") "\n\t"                                                  \
          "v_fmac_" SFX "_dpp %3, %0, -%1" LLH_DPP("%7") "\n\t"                                                  \
          "v_cmp_ge_" SFX " %4, 0, %2\n\tv_mov_" MOV "_dpp %5, %2" LLH_DPP("%7")                                 \
          : "+v"(dj), "+v"(pj), "+v"(dq), "+v"(pq), "=&s"(m), "=&v"(d)                                           \
          : "v"(y), "n"(Q));                                                                                     \
      return m;                                                                                                  \
    }                                                                                                            \
    /* column q updated with column j */                                                                          \
    template <int Q>                                                                                             \
    __device__ __forceinline__ void update(T dj, T pj, T& dq, T& pq) {                                           \
      asm volatile("v_fmac_" SFX "_dpp %0, %2, -%2" LLH_DPP("%4") "\n\t"                                         \
                   "v_fmac_" SFX "_dpp %1, %2, -%3" LLH_DPP("%4")                                                 \
                   : "+v"(dq), "+v"(pq)                                                                          \
                   : "v"(dj), "v"(pj), "n"(Q));                                                                  \
    }                                                                                                            \
    /* step S of the reciprocal root, then column q updated with column j */                                      \
    template <int S, int Q>                                                                                      \
    __device__ __forceinline__ void step(T dj, T pj, T& dq, T& pq);                                              \
    /* the steps from S on, without updates */                                                                    \
    template <int S>                                                                                             \
    __device__ __forceinline__ void rest();                                                                      \
    static constexpr int kSteps = sizeof(T) == 8 ? 6 : 5;                                                        \
  };
LLH_SWEEP_TYPE(double, "f64", "b64")
LLH_SWEEP_TYPE(float, "f32", "b32")
#undef LLH_SWEEP_TYPE

#define LLH_UPD(SFX, D, P, DJ, PJ, Q) \
  "\n\tv_fmac_" SFX "_dpp " D ", " DJ ", -" DJ LLH_DPP(Q) "\n\tv_fmac_" SFX "_dpp " P ", " DJ ", -" PJ LLH_DPP(Q)
template <int S, int Q>
__device__ __forceinline__ void SweepCol<double>::step(double dj, double pj, double& dq, double& pq) {
#define LLH_U LLH_UPD("f64", "%1", "%2", "%3", "%4", "%5")
  if constexpr (S == 0)
    asm volatile("v_rsq_f64 %0, %6" LLH_U : "=&v"(y), "+v"(dq), "+v"(pq) : "v"(dj), "v"(pj), "n"(Q), "v"(d));
  if constexpr (S == 1)
    asm volatile("v_mul_f64 %0, -%6, %7" LLH_U : "=&v"(t), "+v"(dq), "+v"(pq) : "v"(dj), "v"(pj), "n"(Q), "v"(d), "v"(y));
  if constexpr (S == 2)
    asm volatile("v_fma_f64 %0, %0, %6, 1.0" LLH_U : "+v"(t), "+v"(dq), "+v"(pq) : "v"(dj), "v"(pj), "n"(Q), "v"(y));
  if constexpr (S == 3)
    asm volatile("v_mul_f64 %0, %6, %7" LLH_U : "=&v"(u), "+v"(dq), "+v"(pq) : "v"(dj), "v"(pj), "n"(Q), "v"(y), "v"(t));
  if constexpr (S == 4)
    asm volatile("v_fma_f64 %0, %0, %6, 0.5" LLH_U : "+v"(t), "+v"(dq), "+v"(pq) : "v"(dj), "v"(pj), "n"(Q), "s"(0.375));
  if constexpr (S == 5)
    asm volatile("v_fma_f64 %0, %6, %7, %0" LLH_U : "+v"(y), "+v"(dq), "+v"(pq) : "v"(dj), "v"(pj), "n"(Q), "v"(u), "v"(t));
}
template <int S>
__device__ __forceinline__ void SweepCol<double>::rest() {
#define LLH_S1 "v_mul_f64 %1, -%3, %0\n\t"
#define LLH_S2 "v_fma_f64 %1, %1, %0, 1.0\n\t"
#define LLH_S3 "v_mul_f64 %2, %0, %1\n\t"
#define LLH_S4 "v_fma_f64 %1, %1, %4, 0.5\n\t"
#define LLH_S5 "v_fma_f64 %0, %2, %1, %0"
  if constexpr (S == 0)
    asm volatile("v_rsq_f64 %0, %3\n\ts_nop 0\n\t" LLH_S1 LLH_S2 LLH_S3 LLH_S4 LLH_S5
                 : "=&v"(y), "=&v"(t), "=&v"(u) : "v"(d), "s"(0.375));
  if constexpr (S == 1)
    asm volatile(LLH_S1 LLH_S2 LLH_S3 LLH_S4 LLH_S5 : "+v"(y), "=&v"(t), "=&v"(u) : "v"(d), "s"(0.375));
  if constexpr (S == 2)
    asm volatile(LLH_S2 LLH_S3 LLH_S4 LLH_S5 : "+v"(y), "+v"(t), "=&v"(u) : "v"(d), "s"(0.375));
  if constexpr (S == 3)
    asm volatile(LLH_S3 LLH_S4 LLH_S5 : "+v"(y), "+v"(t), "=&v"(u) : "v"(d), "s"(0.375));
  if constexpr (S == 4) asm volatile(LLH_S4 LLH_S5 : "+v"(y), "+v"(t) : "v"(u), "v"(d), "s"(0.375));
  if constexpr (S == 5) asm volatile(LLH_S5 : "+v"(y) : "v"(t), "v"(u));
#undef LLH_S1
#undef LLH_S2
#undef LLH_S3
#undef LLH_S4
#undef LLH_S5
#undef LLH_U
}
template <int S, int Q>
__device__ __forceinline__ void SweepCol<float>::step(float dj, float pj, float& dq, float& pq) {
#define LLH_U LLH_UPD("f32", "%1", "%2", "%3", "%4", "%5")
  if constexpr (S == 0)
    asm volatile("v_rsq_f32 %0, %6" LLH_U : "=&v"(y), "+v"(dq), "+v"(pq) : "v"(dj), "v"(pj), "n"(Q), "v"(d));
  if constexpr (S == 1)
    asm volatile("v_mul_f32 %0, -0.5, %6" LLH_U : "=&v"(t), "+v"(dq), "+v"(pq) : "v"(dj), "v"(pj), "n"(Q), "v"(d));
  if constexpr (S == 2)
    asm volatile("v_mul_f32 %0, %6, %6" LLH_U : "=&v"(u), "+v"(dq), "+v"(pq) : "v"(dj), "v"(pj), "n"(Q), "v"(y));
  if constexpr (S == 3)
    asm volatile("v_fma_f32 %0, %0, %6, %7" LLH_U
                 : "+v"(t), "+v"(dq), "+v"(pq) : "v"(dj), "v"(pj), "n"(Q), "v"(u), "s"(1.5f));
  if constexpr (S == 4)
    asm volatile("v_mul_f32 %0, %0, %6" LLH_U : "+v"(y), "+v"(dq), "+v"(pq) : "v"(dj), "v"(pj), "n"(Q), "v"(t));
}
template <int S>
__device__ __forceinline__ void SweepCol<float>::rest() {
#define LLH_S1 "v_mul_f32 %1, -0.5, %3\n\t"
#define LLH_S2 "v_mul_f32 %2, %0, %0\n\t"
#define LLH_S3 "v_fma_f32 %1, %1, %2, %4\n\t"
#define LLH_S4 "v_mul_f32 %0, %0, %1"
  if constexpr (S == 0)
    asm volatile("v_rsq_f32 %0, %3\n\t" LLH_S1 LLH_S2 LLH_S3 LLH_S4
                 : "=&v"(y), "=&v"(t), "=&v"(u) : "v"(d), "s"(1.5f));
  if constexpr (S == 1)
    asm volatile(LLH_S1 LLH_S2 LLH_S3 LLH_S4 : "+v"(y), "=&v"(t), "=&v"(u) : "v"(d), "s"(1.5f));
  if constexpr (S == 2) asm volatile(LLH_S2 LLH_S3 LLH_S4 : "+v"(y), "+v"(t), "=&v"(u) : "v"(d), "s"(1.5f));
  if constexpr (S == 3) asm volatile(LLH_S3 LLH_S4 : "+v"(y), "+v"(t) : "v"(u), "v"(d), "s"(1.5f));
  if constexpr (S == 4) asm volatile(LLH_S4 : "+v"(y) : "v"(t));
#undef LLH_S1
#undef LLH_S2
#undef LLH_S3
#undef LLH_S4
#undef LLH_U
}
#undef LLH_UPD
#undef LLH_DPP

// A workgroup barrier that orders LDS accesses only: __syncthreads() also waits
// for the global loads and stores in flight.
__device__ __forceinline__ void diag_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

constexpr int kDiagW = 16;   // columns per step, rows per strip
constexpr int kDiagT = 256;  // threads of a diagonal-block workgroup

// LDS row stride of a 16 x 16 block: whole 16-byte vectors, and the 16 rows of a
// vector read start in different bank groups.
template <typename T>
constexpr int diag_ls() { return kDiagW + 16 / (int)sizeof(T); }
template <typename T>
constexpr int diag_blk() { return kDiagW * diag_ls<T>(); }

// 38.1 KB in f64 (four workgroups per CU).  Inside diag_quad_block l holds 14
// blocks: the steps' strips, published and then swept (3 x 4), and L_ww (2); a
// caller may use l and x as scratch afterwards.
template <typename T>
struct DiagLds {
  static constexpr int kL = 14 * diag_blk<T>() > kNB * (kNB + 1) ? 14 * diag_blk<T>() : kNB * (kNB + 1);
  T l[(kL + 1) / 2 * 2];
  T x[kNB * 8];
  int fail[kNB / kDiagW];  // per step: failing column or -1
  int skip;                // the system has already failed: nothing to do
};

// The four steps on a 64 x 64 block whose strips are in acc (negated, see above; one
// strip per wave g).  A step's column block is published in the buffer that its
// rows go to afterwards, and there are three such buffers: the rows of step w stay
// until step w + 3.  put(w, it, f) stores piece it of step w: the rows of strip it
// (0..3) or L_ww (4), up to a failure at row f (f < 0: none).  pend(w, x) runs beside
// sweep w on the waves g > w and may still change their block (g, w + 1), which is x;
// help(w) follows on every wave g != w, which wave w + 1 should leave early; with WIDE
// it runs on four further waves instead, beside every sweep.  Returns
// the failing row or -1, the same in every thread.  l: 14 * diag_blk<T>() elements
// of LDS, fails: one word per step.
template <typename T>
__device__ __forceinline__ T* diag_rows(T* l, int w) {
  return l + (w == 3 ? 0 : w) * 4 * diag_blk<T>();
}
template <typename T>
__device__ __forceinline__ T* diag_lww(T* l, int w) {
  return l + (12 + (w & 1)) * diag_blk<T>();
}

template <typename T, bool WIDE = false, typename Put, typename Help, typename Pend>
__device__ __forceinline__ int diag_core(typename Mfma<T>::acc_t (&acc)[kNB / kDiagW], int g, T* l, int* fails,
                                         Put&& put, Help&& help, Pend&& pend) {
  constexpr int W = kDiagW, NS = kNB / W, LS = diag_ls<T>(), BLK = diag_blk<T>(), VL = 16 / sizeof(T);
  using MF = Mfma<T>;
  using acc_t = typename MF::acc_t;
  typedef T vec_t __attribute__((ext_vector_type(VL)));
  const bool factor = !WIDE || g < NS;  // wave-uniform (g comes from readfirstlane)
  int fail = -1;
  // One copy of the step's code for all four steps (a quarter of the
  // instruction fetches).
#pragma unroll 1
  for (int w = 0; w < NS && fail < 0; ++w) {
    // the LDS addresses are formed in each step: kept across the steps they take
    // a hundred registers
    int lane = threadIdx.x & 63;
    asm volatile("" : "+v"(lane));
    const int fr = lane & 15, fq = lane >> 4;
    // acc[c] += P_g L_c^T with the rows of a sweep in buffer p
    auto update = [&](acc_t& x, const T* p, int c) __attribute__((always_inline)) {
#pragma unroll
      for (int s = 0; s < 4; ++s)
        x = MF::mma(p[g * BLK + fr * LS + 4 * s + fq], p[c * BLK + fr * LS + 4 * s + fq], x);
    };
    // acc[0] is column block w: the blocks move down by one each step, so that the
    // registers are addressed by constants
    T* const stg = diag_rows(l, w);
    if (factor) {
#pragma unroll
      for (int r = 0; r < 4; ++r) stg[g * BLK + MF::row(lane, r) * LS + fr] = -acc[0][r];
    }
    diag_barrier();
    if (!factor) {
      help(w);
    } else if (g == w) {
      // the sweep: d = row fr of the diagonal block, p = row fr of strip fq
      T d[W], p[W];
#pragma unroll
      for (int q = 0; q < W; q += VL) {
        const vec_t vd = *reinterpret_cast<const vec_t*>(&stg[w * BLK + fr * LS + q]);
        const vec_t vp = *reinterpret_cast<const vec_t*>(&stg[fq * BLK + fr * LS + q]);
#pragma unroll
        for (int e = 0; e < VL; ++e) {
          d[q + e] = vd[e];
          p[q + e] = fq == w ? T(q + e == fr ? 1 : 0) : vp[e];
        }
      }
      // No branch depends on the data: a failing pivot (cholesky.rs:69; NaN passes)
      // only sets its bit and the sweep runs on.  Entries of d above the diagonal
      // hold values that no kept result reads.
      using SC = SweepCol<T>;
      SC sc;
      uint32_t fm = (uint32_t)sc.first(d[0]) & 1u;
      sc.template rest<0>();
      static_for(std::make_integer_sequence<int, W - 1>{}, [&](auto ji) {
        constexpr int j = decltype(ji)::value, later = W - 2 - j;  // columns after the next
        fm |= (uint32_t)sc.template next<j + 1>(d[j], p[j], d[j + 1], p[j + 1]) & (2u << j);
        static_for(std::make_integer_sequence<int, later>{}, [&](auto ki) {
          constexpr int k = decltype(ki)::value, q = j + 2 + k;
          if constexpr (k < SC::kSteps)
            sc.template step<k, q>(d[j], p[j], d[q], p[q]);
          else
            sc.template update<q>(d[j], p[j], d[q], p[q]);
        });
        if constexpr (later < SC::kSteps) sc.template rest<(later < SC::kSteps ? later : 0)>();
      });
      sc.scale(d[W - 1], p[W - 1]);
      T* pr = diag_rows(l, w) + fq * BLK + fr * LS;
#pragma unroll
      for (int q = 0; q < W; q += VL) {
        vec_t vp;
#pragma unroll
        for (int e = 0; e < VL; ++e) vp[e] = p[q + e];
        *reinterpret_cast<vec_t*>(pr + q) = vp;
      }
      if (fq == 0) {
        T* dr = diag_lww(l, w) + fr * LS;
#pragma unroll
        for (int q = 0; q < W; q += VL) {
          vec_t vd;
#pragma unroll
          for (int e = 0; e < VL; ++e) vd[e] = d[q + e];
          *reinterpret_cast<vec_t*>(dr + q) = vd;
        }
      }
      if (lane == 0) fails[w] = fm != 0 ? W * w + __builtin_ctz(fm) : -1;
    } else {
      // meanwhile the other waves: the previous step's products for the
      // later column blocks, and its stores
      if (g > w) pend(w, acc[1]);
      if (w > 0) {
#pragma unroll
        for (int e = 1; e < NS - 1; ++e) {
          const int c = w + e;
          if (c < NS && (g < w || c <= g)) update(acc[e], diag_rows(l, w - 1), c);
        }
        const int k = g < w ? g : g - 1;
        put(w - 1, k, -1);
        if (k + 3 <= NS) put(w - 1, k + 3, -1);
      }
      if constexpr (!WIDE) help(w);
    }
    diag_barrier();
    fail = fails[w];
    if (!factor) continue;
    if (fail < 0) {
#pragma unroll
      for (int e = 0; e < NS - 1; ++e) acc[e] = acc[e + 1];
      if (w + 1 < NS) update(acc[0], diag_rows(l, w), w + 1);
    } else if (g == 0) {
      put(w, NS, fail);
    }
  }
  if (fail < 0 && factor) {
    put(NS - 1, g, -1);
    if (g == 0) put(NS - 1, NS, -1);
  }
  return fail;
}

// The strip of wave g < 4 of a b x b block (b <= 64), negated, in T's MFMA result
// layout; rows and columns beyond b are the identity's.  Only the lower triangle
// is read: masked entries load the block's first element, so that the loads
// carry no branches.
template <typename TS, typename T>
__device__ __forceinline__ void diag_load(const TS* __restrict__ a, int64_t lda, int b, int g,
                                          typename Mfma<T>::acc_t (&acc)[kNB / kDiagW]) {
  const int lane = threadIdx.x & 63;
  T v[kNB / kDiagW][4];  // every load is in flight before one is used
#pragma unroll
  for (int c = 0; c < kNB / kDiagW; ++c)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int row = kDiagW * g + Mfma<T>::row(lane, r), col = kDiagW * c + (lane & 15);
      v[c][r] = T(a[row < b && col <= row ? (int64_t)row * lda + col : 0]);
    }
#pragma unroll
  for (int c = 0; c < kNB / kDiagW; ++c)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int row = kDiagW * g + Mfma<T>::row(lane, r), col = kDiagW * c + (lane & 15);
      acc[c][r] = row < b && col <= row ? -v[c][r] : (row >= b && row == col ? T(-1) : T(0));
    }
}

// Stores piece it of step w (see diag_core) of a b x b block: L to lo (ld ldl), the
// inverse to inv (64 x 64, row-major).
template <typename TS, typename T>
__device__ __forceinline__ void diag_put(T* l, int w, int it, int f, int b, TS* lo, int64_t ldl, TS* inv) {
  constexpr int W = kDiagW, NS = kNB / W, LS = diag_ls<T>(), BLK = diag_blk<T>();
  int lane = threadIdx.x & 63;
  asm volatile("" : "+v"(lane));  // the addresses are formed here, not kept across the sweeps
  const int rr = lane >> 2, cc = (lane & 3) * 4;
  if (it > w) {  // L, or its diagonal block
    const bool dia = it == NS;
    const T* src = (dia ? diag_lww(l, w) : diag_rows(l, w) + it * BLK) + rr * LS + cc;
    const int row = W * (dia ? w : it) + rr;
    if (row >= b) return;
    const int last = f < 0 ? row : (row < f ? row : (row == f ? f - 1 : -1));
    TS* dst = lo + (int64_t)row * ldl + W * w + cc;
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (W * w + cc + e <= last) dst[e] = TS(src[e]);
  } else if (f < 0) {  // block (w, it) of the inverse, and the zero block (it, w)
    const T* src = diag_rows(l, w) + it * BLK + cc * LS + rr;
    TS* dst = inv + (W * w + rr) * kNB + W * it + cc;
#pragma unroll
    for (int e = 0; e < 4; ++e) dst[e] = TS(src[e * LS]);
    if (it < w) {
      TS* z = inv + (W * it + rr) * kNB + W * w + cc;
#pragma unroll
      for (int e = 0; e < 4; ++e) z[e] = TS(0);
    }
  }
}

// TS: storage type of the block and of the inverse; T: arithmetic type.
// Called by all kDiagT threads of a workgroup; returns true (in every thread)
// when the block failed, after recording the failing row in *info.  inv is 64 x
// 64, row-major.
template <typename TS, typename T>
__device__ __forceinline__ bool diag_quad_block(TS* __restrict__ a, int64_t lda, int b, TS* __restrict__ inv,
                                                int32_t* __restrict__ info, int64_t info_base, DiagLds<T>& sm) {
  const int g = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  typename Mfma<T>::acc_t acc[kNB / kDiagW];
  diag_load<TS, T>(a, lda, b, g, acc);
  const int fail = diag_core<T>(
      acc, g, sm.l, sm.fail,
      [&](int w, int it, int f) { diag_put<TS, T>(sm.l, w, it, f, b, a, lda, inv); }, [](int) {},
      [](int, auto&) {});
  if (fail >= 0 && threadIdx.x == 0) atomicMin(info, (int32_t)(info_base + fail));
  return fail >= 0;
}

}  // namespace llh
