// Host drivers: the blocked right-looking POTRF and the blocked triangular
// solves, as sequences of kernel launches on one stream.
#include <algorithm>
#include <climits>

#include "llh_driver.h"
#include "llh_kernels.h"

namespace llh {

#define LLH_TRY(expr)                  \
  do {                                 \
    hipError_t e_ = (expr);            \
    if (e_ != hipSuccess) return e_;   \
  } while (0)

// Brackets one launch on stream st with the profiler's events (no-op when
// profiling is off).
#define LLH_PROF_ON(st, cls, flops, bytes, expr)                                \
  do {                                                                          \
    const int pi_ = prof ? prof->begin((cls), (flops), (bytes), (st)) : -1;     \
    LLH_TRY(expr);                                                              \
    if (prof) prof->end(pi_, (st));                                             \
  } while (0)
#define LLH_PROF(cls, flops, bytes, expr) LLH_PROF_ON(s, cls, flops, bytes, expr)

namespace {

// The rows of the panel [k0, k0 + kb) that its steps factor end here.
int top_end(int n, int k0, int kb) { return n - k0 <= kStepRows ? n : k0 + kb; }

// Factors the columns [k0, k0 + kb) of the rows k0 .. n on stream st, everything left
// of k0 having been applied to them: one launch per 64 columns.  *stepped: whether
// the block before k0 still waits beside its place (launch_panel_step).
template <typename T>
hipError_t factor_steps(T* a, int64_t lda, int n, int k0, int kb, int32_t* info, T* dinv, bool beside, bool* stepped,
                        hipStream_t st, Profiler* prof, bool diag_f64) {
  const double es = (double)sizeof(T);
  const int end = k0 + kb;
  for (int k = k0; k < end; k += kNB) {
    const double db = std::min(kNB, n - k), below = std::max(0, n - k - kNB), pb = k > k0 ? db : 0.0;
    const bool ahead = !diag_f64 && step_ahead<T>(k, k0);
    const double cols = std::max(0, ahead ? std::min(kNB, end - k - kNB) : end - k - kNB);
    const double outs = below * cols - cols * (cols - 1.0) / 2.0;
    const double rank = pb > 0.0 ? (diag_f64 ? kNB : step_rank<T>(k, k0)) : 0.0;
    LLH_PROF_ON(st, kDiagFactor, 2.0 * db * db * db / 3.0 + 2.0 * below * db * (db + pb) + 2.0 * outs * rank,
                es * (2.0 * db * db + below * (2.0 * db + rank) + (pb > 0.0 ? 2.0 * outs : 0.0)),
                (diag_f64 && sizeof(T) == 4
                     ? launch_panel_step<T, double>(a, lda, n, k, k0, end, dinv, info, *stepped, beside, st)
                     : launch_panel_step<T>(a, lda, n, k, k0, end, dinv, info, *stepped, beside, st)));
    *stepped = k + kNB < n;
  }
  return hipSuccess;
}

// The rows below the factored top block of a panel: L21 = A21 L11^-T.
template <typename T>
hipError_t factor_rows(T* a, int64_t lda, int n, int k0, int kb, int32_t* info, const T* dinv, hipStream_t st,
                       Profiler* prof) {
  const double below = n - top_end(n, k0, kb), dkb = kb;
  if (below <= 0.0) return hipSuccess;
  LLH_PROF_ON(st, kPanelTrsm, below * dkb * dkb, sizeof(T) * (2.0 * below * dkb + dkb * dkb / 2.0),
              (launch_panel_rows<T>(a, lda, n, k0, kb, dinv, info, st)));
  return hipSuccess;
}

// The trailing update C -= P P^T (lower triangle of the m x m C, P m x kb).
// With half (f32 storage only), P is first rounded to f16 into half (ld kb) and
// the SYRK multiplies in f16 with f32 accumulation.
template <typename T>
hipError_t trailing_syrk(int m, int kb, const T* p, int64_t lda, T* c, int32_t* info, _Float16* half,
                         hipStream_t s) {
  if constexpr (sizeof(T) == 4) {
    if (half != nullptr) {
      LLH_TRY(launch_convert_s2h(m, kb, p, lda, half, kb, s));
      return launch_syrk_lower_h(m, kb, -1.0f, half, kb, 1.0f, c, lda, info, s);
    }
  }
  return launch_syrk_lower<T>(m, kb, T(-1), p, lda, T(1), c, lda, info, s);
}

}  // namespace

// Right-looking blocked Cholesky of the lower triangle (the blocked equivalent
// of cholesky.rs:54-74).  Each outer panel (panel_width() columns) is factored in
// steps of 64 columns (factor_steps, and factor_rows for the rows that these leave);
// then one SYRK of that rank on MFMA updates the trailing matrix.  With lookahead, the
// trailing update of panel k is split: the rows of the next panel's steps are updated
// and the steps taken on the side stream while s updates the panel's other rows and
// then the remaining trailing matrix.  Matrices no larger than the LDS
// kernel's limit are factored by that kernel alone, in the reference's exact
// operation order.
template <typename T>
hipError_t potrf_enqueue(T* a, int64_t lda, int n, int32_t* info, bool zero_upper, T* dinv, hipStream_t s,
                         Profiler* prof, bool diag_f64, const Lookahead* la, _Float16* half, const FwdFuse<T>* ff) {
  const double es = (double)sizeof(T);
  if (half != nullptr && sizeof(T) != 4) return hipErrorInvalidValue;
  if (ff != nullptr && (la == nullptr || la->fwd == nullptr || dinv == nullptr || n <= small_max<T>() ||
                        ff->m <= 0 || ff->m > 64 || ff->sync == nullptr))
    return hipErrorInvalidValue;
  // The fused forward step of the outer panel [k0, k0 + kb), on la->fwd once
  // the panel is factored: Y_k := L11^-1 Y_k (one-launch triangle), then
  // Y[k0 + kb:] -= L21 Y_k.
  auto fwd_panel = [&](int k0, int kb) -> hipError_t {
    const int m = ff->m;
    T* yk = ff->y + (int64_t)k0 * ff->ldy;
    LLH_TRY(trsm_enqueue<T>(false, false, kb, a + (int64_t)k0 * lda + k0, lda, m, yk, ff->ldy,
                            dinv + (int64_t)(k0 / kNB) * kNB * kNB, false, nullptr, ff->sync, la->fwd, prof, info));
    const int rest = n - k0 - kb;
    if (rest <= 0) return hipSuccess;
    LLH_PROF_ON(la->fwd, kSolveGemm, 2.0 * rest * m * kb, es * ((double)rest * kb + 2.0 * rest * m + (double)kb * m),
                (launch_gemm<T>(false, false, false, rest, m, kb, T(-1), a + (int64_t)(k0 + kb) * lda + k0, lda, yk,
                                ff->ldy, T(1), yk + (int64_t)kb * ff->ldy, ff->ldy, info, la->fwd)));
    return hipSuccess;
  };
  // bytes per panel element of the trailing update (the f16 copy is written
  // and read once more)
  const double pes = half != nullptr ? es + 4.0 : es;
  if (n > small_max<T>() && dinv == nullptr) return hipErrorInvalidValue;  // the blocked path needs the inverses
  if (n <= 0 || n > small_max<T>()) LLH_TRY(launch_fill_i32(info, kNoFail, 1, s));
  if (n <= 0) return hipSuccess;
  if (n <= small_max<T>()) {
    LLH_TRY(launch_potrf_exact_single<T>(a, lda, n, info, zero_upper, s));
    if (dinv != nullptr) LLH_TRY(launch_trtri_blocks<T>(n, a, lda, false, false, dinv, info, s));
  } else {
    const int kb0 = std::min(panel_width(n, n, half != nullptr), n);
    bool stepped = false;
    LLH_TRY(factor_steps<T>(a, lda, top_end(n, 0, kb0), 0, kb0, info, dinv, false, &stepped, s, prof, diag_f64));
    LLH_TRY(factor_rows<T>(a, lda, n, 0, kb0, info, dinv, s, prof));
    if (ff != nullptr) {
      LLH_TRY(hipEventRecord(la->fwd_ev, s));
      LLH_TRY(hipStreamWaitEvent(la->fwd, la->fwd_ev, 0));
      if (ff->b != nullptr)
        LLH_TRY(hipMemcpy2DAsync(ff->y, ff->ldy * sizeof(T), ff->b, ff->ldb * sizeof(T), ff->m * sizeof(T), n,
                                 hipMemcpyDeviceToDevice, la->fwd));
      LLH_TRY(fwd_panel(0, kb0));
    }
    for (int k0 = 0, kb = kb0, kb2 = 0; k0 + kb < n; k0 += kb, kb = kb2) {
      const int m2 = n - k0 - kb;
      kb2 = std::min(panel_width(m2, n, half != nullptr), m2);  // width of the next panel
      T* p = a + (int64_t)(k0 + kb) * lda + k0;  // L21: rows k0+kb.., columns k0..k0+kb
      T* c = p + kb;                              // trailing matrix at (k0+kb, k0+kb)
      // The trailing SYRK's algorithmic work: outs outputs of the lower
      // triangle, each a kb-term dot product; bytes: read and write the lower
      // triangle of C once, read the panel once.
      if (la == nullptr) {
        const double outs = (double)m2 * (m2 + 1) / 2.0;
        LLH_PROF(kTrailingSyrk, 2.0 * outs * kb, es * 2.0 * outs + pes * (double)m2 * kb,
                 (trailing_syrk<T>(m2, kb, p, lda, c, info, half, s)));
        LLH_TRY(factor_steps<T>(a, lda, top_end(n, k0 + kb, kb2), k0 + kb, kb2, info, dinv, false, &stepped, s, prof,
                                diag_f64));
        LLH_TRY(factor_rows<T>(a, lda, n, k0 + kb, kb2, info, dinv, s, prof));
        continue;
      }
      // With half, the whole panel (m2 x kb) is rounded to f16 once, before the
      // fork: the look-ahead update and the SYRK both read the copy.
      bool half_ready = false;
      if constexpr (sizeof(T) == 4) {
        if (half != nullptr) {
          LLH_TRY(launch_convert_s2h(m2, kb, p, lda, half, kb, s));
          half_ready = true;
        }
      }
      LLH_TRY(hipEventRecord(la->fork, s));
      LLH_TRY(hipStreamWaitEvent(la->side, la->fork, 0));
      const int m3 = m2 - kb2;  // the rest of the trailing matrix
      const int end2 = top_end(n, k0 + kb, kb2), mt = end2 - k0 - kb, mr = n - end2;  // next panel's rows: steps, below
      {
        // the rows of the next panel's steps, then these, on the side stream
        const double outs = (double)mt * kb2 - (double)kb2 * (kb2 - 1) / 2.0;
        if (half_ready) {
          if constexpr (sizeof(T) == 4)
            LLH_PROF_ON(la->side, kPanelUpdate, 2.0 * outs * kb, 4.0 * 2.0 * outs + 2.0 * (double)mt * kb,
                        (launch_gemm_nt_h(true, mt, kb2, kb, -1.0f, half, kb, half, kb, 1.0f, c, lda, info,
                                          la->side)));
        } else {
          LLH_PROF_ON(la->side, kPanelUpdate, 2.0 * outs * kb, es * (2.0 * outs + (double)mt * kb),
                      (launch_gemm<T>(false, true, true, mt, kb2, kb, T(-1), p, lda, p, lda, T(1), c, lda, info,
                                      la->side)));
        }
        LLH_TRY(factor_steps<T>(a, lda, end2, k0 + kb, kb2, info, dinv, (mr > 0), &stepped, la->side, prof,
                                diag_f64));
      }
      if (mr > 0) {
        // its rows below, on s; then their solve, on the side stream
        const double outs = (double)mr * kb2;
        T* c2 = c + (int64_t)kb2 * lda;
        if (half_ready) {
          if constexpr (sizeof(T) == 4)
            LLH_PROF(kPanelUpdate, 2.0 * outs * kb, 4.0 * 2.0 * outs + 2.0 * ((double)mr + kb2) * kb,
                     (launch_gemm_nt_h(false, mr, kb2, kb, -1.0f, half + (int64_t)kb2 * kb, kb, half, kb, 1.0f, c2,
                                       lda, info, s)));
        } else {
          LLH_PROF(kPanelUpdate, 2.0 * outs * kb, es * (2.0 * outs + ((double)mr + kb2) * kb),
                   (launch_gemm<T>(false, true, false, mr, kb2, kb, T(-1), p + (int64_t)kb2 * lda, lda, p, lda, T(1),
                                   c2, lda, info, s)));
        }
        LLH_TRY(hipEventRecord(la->rows, s));
        LLH_TRY(hipStreamWaitEvent(la->side, la->rows, 0));
        LLH_TRY(factor_rows<T>(a, lda, n, k0 + kb, kb2, info, dinv, la->side, prof));
      }
      LLH_TRY(hipEventRecord(la->join, la->side));
      if (ff != nullptr) {
        LLH_TRY(hipStreamWaitEvent(la->fwd, la->join, 0));
        LLH_TRY(fwd_panel(k0 + kb, kb2));
      }
      if (m3 > 0) {
        const double outs = (double)m3 * (m3 + 1) / 2.0;
        T* p3 = p + (int64_t)kb2 * lda;
        T* c3 = c + (int64_t)kb2 * lda + kb2;
        if (half_ready) {
          if constexpr (sizeof(T) == 4)
            LLH_PROF(kTrailingSyrk, 2.0 * outs * kb, es * 2.0 * outs + 2.0 * (double)m3 * kb,
                     (launch_syrk_lower_h(m3, kb, -1.0f, half + (int64_t)kb2 * kb, kb, 1.0f, c3, lda, info, s)));
        } else {
          LLH_PROF(kTrailingSyrk, 2.0 * outs * kb, es * 2.0 * outs + pes * (double)m3 * kb,
                   (trailing_syrk<T>(m3, kb, p3, lda, c3, info, half, s)));
        }
      }
      LLH_TRY(hipStreamWaitEvent(s, la->join, 0));
    }
    if (ff != nullptr) {
      LLH_TRY(hipEventRecord(la->fwd_ev, la->fwd));
      LLH_TRY(hipStreamWaitEvent(s, la->fwd_ev, 0));
    }
  }
  if (zero_upper && n > small_max<T>()) LLH_TRY(launch_zero_triangle<T>(a, lda, n, true, info, s));
  return hipSuccess;
}

namespace {

// op(A) X = B with the inverses of the diagonal blocks, or by substitution (dinv
// null): one launch (launch_trsm_persistent) up to solve_split<T>(m) rows, otherwise by
// halves: the half that comes first, one product into the other half's rows, the other half.
template <typename T>
hipError_t trsm_split(bool upper_op, bool trans, int n, const T* a, int64_t lda, int m, T* b, int64_t ldb,
                      const T* dinv, bool dinv_t, SolveSync* sync, hipStream_t s, Profiler* prof,
                      const int32_t* gate) {
  const double es = (double)sizeof(T);
  if (n <= solve_split<T>(m)) {
    // the launch leaves the ticket at 0; the error word is the call's (solve_sync_begin)
    const int most = (int)std::min<int64_t>(sync->nmail * kSolveChunkHost, INT_MAX);
    for (int c = 0; c < m; c += most) {
      const int mc = std::min(most, m - c);
      // (before the values run out the words are cleared and they start anew: some 20
      // hours of solves without a pause)
      if (*sync->epoch > INT_MAX - solve_epochs(n)) {
        LLH_TRY(launch_fill_i32(sync->words + 2, 0, sync->nflags, s));
        LLH_TRY(launch_fill_i32(reinterpret_cast<int32_t*>(sync->mail), 0, 2 * solve_mail_words(sync->nmail), s));
        *sync->epoch = 1;
      }
      const int32_t epoch = *sync->epoch;
      *sync->epoch += solve_epochs(n);
      const double fl = (double)n * n * mc;
      LLH_PROF(kSolveGemm, fl, es * ((double)n * n / 2.0 + 2.0 * n * mc),
               (launch_trsm_persistent<T>(n, mc, a, lda, trans, !upper_op, dinv, dinv_t, b + c, ldb, sync->words,
                                          sync->words + 2, sync->mail, epoch, sync->words + 1, sync->spin_limit,
                                          gate, s)));
      if (m - c <= most) break;
    }
    return hipSuccess;
  }
  const int n1 = ((n + kNB - 1) / kNB + 1) / 2 * kNB, n2 = n - n1;
  const T* d2 = dinv == nullptr ? nullptr : dinv + (int64_t)(n1 / kNB) * kNB * kNB;
  const T* a22 = a + (int64_t)n1 * lda + n1;
  T* b2 = b + (int64_t)n1 * ldb;
  const double fl = 2.0 * n1 * n2 * m, by = es * ((double)n1 * n2 + 2.0 * n * m);
  if (!upper_op) {
    LLH_TRY(trsm_split<T>(upper_op, trans, n1, a, lda, m, b, ldb, dinv, dinv_t, sync, s, prof, gate));
    LLH_PROF(kSolveGemm, fl, by,
             (launch_gemm<T>(trans, false, false, n2, m, n1, T(-1), trans ? a + n1 : a + (int64_t)n1 * lda, lda, b,
                             ldb, T(1), b2, ldb, gate, s)));
    return trsm_split<T>(upper_op, trans, n2, a22, lda, m, b2, ldb, d2, dinv_t, sync, s, prof, gate);
  }
  LLH_TRY(trsm_split<T>(upper_op, trans, n2, a22, lda, m, b2, ldb, d2, dinv_t, sync, s, prof, gate));
  LLH_PROF(kSolveGemm, fl, by,
           (launch_gemm<T>(trans, false, false, n1, m, n2, T(-1), trans ? a + (int64_t)n1 * lda : a + n1, lda, b2,
                           ldb, T(1), b, ldb, gate, s)));
  return trsm_split<T>(upper_op, trans, n1, a, lda, m, b, ldb, dinv, dinv_t, sync, s, prof, gate);
}

}  // namespace

// Blocked solve of op(A) X = B (B row-major n x m, in place): trsm_split, or, without
// sync or beyond kSolveMaxCols columns, the substitution kNB rows at a time: solve the
// diagonal block, then subtract its contribution from the rows still to come with one
// GEMM (the column sweep of triangular.rs:113-125, done a block of rows at a time).
template <typename T>
hipError_t trsm_enqueue(bool upper_op, bool trans, int n, const T* a, int64_t lda, int m, T* b, int64_t ldb,
                        const T* dinv, bool dinv_t, T* dinv_work, SolveSync* sync, hipStream_t s,
                        Profiler* prof, const int32_t* gate) {
  if (n <= 0 || m <= 0) return hipSuccess;
  const double es = (double)sizeof(T);
  const bool inverses = m <= 64;
  if (sync != nullptr && sync->epoch != nullptr && m <= kSolveMaxCols && sync->nflags >= solve_flags<T>(n, m) &&
      sync->mail != nullptr && sync->nmail > 0 && (!inverses || dinv != nullptr || dinv_work != nullptr)) {
    if (!inverses) {
      dinv = nullptr;
    } else if (dinv == nullptr) {
      LLH_PROF(kSolveDiag, (double)n * kNB * kNB / 3.0, es * (double)n * kNB,
               (launch_trtri_blocks<T>(n, a, lda, trans, upper_op, dinv_work, gate, s)));
      dinv = dinv_work;
      dinv_t = false;
    }
    return trsm_split<T>(upper_op, trans, n, a, lda, m, b, ldb, dinv, dinv_t, sync, s, prof, gate);
  }
  const int nblk = (n + kNB - 1) / kNB;
  if (!upper_op) {  // forward
    for (int bi = 0; bi < nblk; ++bi) {
      const int i0 = bi * kNB, bs = std::min(kNB, n - i0);
      const T* tkk = a + (int64_t)i0 * lda + i0;
      LLH_PROF(kSolveDiag, (double)bs * bs * m, es * ((double)bs * bs / 2.0 + 2.0 * bs * m),
               (launch_trsv_block<T>(false, trans, bs, tkk, lda, m, b + (int64_t)i0 * ldb, ldb, gate, s)));
      const int rest = n - i0 - bs;
      if (rest <= 0) continue;
      // B[i0+bs:, :] -= op(A)[i0+bs:, i0:i0+bs] * X[i0:i0+bs, :]
      const T* blk = trans ? a + (int64_t)i0 * lda + (i0 + bs) : a + (int64_t)(i0 + bs) * lda + i0;
      LLH_PROF(kSolveGemm, 2.0 * rest * m * bs, es * ((double)rest * bs + 2.0 * rest * m + (double)bs * m),
               (launch_gemm<T>(trans, false, false, rest, m, bs, T(-1), blk, lda, b + (int64_t)i0 * ldb, ldb,
                               T(1), b + (int64_t)(i0 + bs) * ldb, ldb, gate, s)));
    }
  } else {  // backward
    for (int bi = nblk - 1; bi >= 0; --bi) {
      const int i0 = bi * kNB, bs = std::min(kNB, n - i0);
      const T* tkk = a + (int64_t)i0 * lda + i0;
      LLH_PROF(kSolveDiag, (double)bs * bs * m, es * ((double)bs * bs / 2.0 + 2.0 * bs * m),
               (launch_trsv_block<T>(true, trans, bs, tkk, lda, m, b + (int64_t)i0 * ldb, ldb, gate, s)));
      if (i0 == 0) continue;
      // B[:i0, :] -= op(A)[:i0, i0:i0+bs] * X[i0:i0+bs, :]
      const T* blk = trans ? a + (int64_t)i0 * lda : a + i0;
      LLH_PROF(kSolveGemm, 2.0 * i0 * m * bs, es * ((double)i0 * bs + 2.0 * i0 * m + (double)bs * m),
               (launch_gemm<T>(trans, false, false, i0, m, bs, T(-1), blk, lda, b + (int64_t)i0 * ldb, ldb,
                               T(1), b, ldb, gate, s)));
    }
  }
  return hipSuccess;
}

// The forward and back substitution with the factor L (lower triangle of a)
// and the inverses of its diagonal blocks (dinv, as the factor leaves them).
// A small one (solve_in_lds) is one single-workgroup launch with B in LDS and L
// streamed through registers (launch_solve_lds), otherwise the two one-launch
// triangles (trsm_enqueue).
//
// The one workgroup's time grows with n and m, the triangles' by a hop per 64 rows
// only.  Factor and solve, f64, one workgroup / triangles (us): n = 200 m = 1 112 / 133, m = 4
// 125 / 132, m = 8 140 / 132; n = 300 138 / 154, 158 / 153, 182 / 154; n = 400 203 / 200, 239 /
// 200, 284 / 201; n = 512 m = 1 239 / 225; f32 the same within 32 rows.
inline bool solve_in_lds(int n, int m) { return n + 32 * m <= 432 && m <= kSolveCols; }
static_assert(432 <= kSolveLdsMaxN, "the one-workgroup solve takes them");
template <typename T>
hipError_t solve_pair_enqueue(int n, const T* a, int64_t lda, int m, T* b, int64_t ldb, const T* dinv,
                              SolveSync* sync, hipStream_t s, Profiler* prof, const int32_t* gate) {
  const double es = (double)sizeof(T);
  if (solve_in_lds(n, m) && dinv != nullptr && lda <= INT32_MAX) {
    LLH_PROF(kSolveGemm, 2.0 * n * n * m, es * ((double)n * n + 2.0 * n * m),
             (launch_solve_lds<T>(n, m, a, lda, dinv, b, ldb, gate, s)));
    return hipSuccess;
  }
  LLH_TRY(trsm_enqueue<T>(false, false, n, a, lda, m, b, ldb, dinv, false, nullptr, sync, s, prof, gate));
  return trsm_enqueue<T>(true, true, n, a, lda, m, b, ldb, dinv, true, nullptr, sync, s, prof, gate);
}

template <typename T>
bool forward_fusable(int n, int m, const Lookahead* la) {
  return m > 0 && m <= 64 && n > panel_width(n, n, false) && n > kSolveLdsMaxN && n > small_max<T>() &&
         la != nullptr && la->fwd != nullptr && la->fwd_ev != nullptr;
}

// At n = 32768 with 16 right-hand sides the forward triangle after the factor
// would be 1.5 ms (512 hops); fused, each panel's 16-hop triangle and product
// run beside the trailing SYRK and only the last panel's, up to 64 hops, trail the factor.
template <typename T>
hipError_t factor_solve_enqueue(T* a, int64_t lda, int n, int m, T* b, int64_t ldb, T* dinv, T* y, SolveSync* sync,
                                int32_t* info, hipStream_t s, Profiler* prof, const Lookahead* la) {
  if (!forward_fusable<T>(n, m, la)) {
    LLH_TRY(potrf_enqueue<T>(a, lda, n, info, false, dinv, s, prof, false, la));
    if (m <= 0) return hipSuccess;
    return solve_pair_enqueue<T>(n, a, lda, m, b, ldb, dinv, sync, s, prof, info);
  }
  if (y == nullptr) return hipErrorInvalidValue;
  FwdFuse<T> ff;
  ff.b = b;
  ff.ldb = ldb;
  ff.y = y;
  ff.ldy = m;
  ff.m = m;
  ff.sync = sync;
  LLH_TRY(potrf_enqueue<T>(a, lda, n, info, false, dinv, s, prof, false, la, nullptr, &ff));
  LLH_TRY(launch_copy_rows_gated<T>(n, m, y, m, b, ldb, info, s));
  return trsm_enqueue<T>(true, true, n, a, lda, m, b, ldb, dinv, true, nullptr, sync, s, prof, info);
}

// A^-1 = L^-T L^-1 from the factor L (the lower triangle of a, lda) and the
// inverses of its diagonal blocks: W = L^-1 into the lower triangle of w (n x n,
// ldw), pairs of neighbouring diagonal blocks of h = 64, 128, ... rows combined as
// [[L11, 0], [L21, L22]]^-1 = [[W11, 0], [-W22 L21 W11, W22]], two launches a level;
// then W^T W into both triangles of x (ldx).  tmp: potri_tmp_elems(n) elements.
// About n^3/3 flops for W and n^3/3 for W^T W, against the 2n^3 of solving with the
// n columns of the identity.
template <typename T>
hipError_t potri_enqueue(int n, const T* a, int64_t lda, const T* dinv, T* w, int64_t ldw, T* x, int64_t ldx,
                         T* tmp, hipStream_t s) {
  if (n <= 0) return hipSuccess;
  LLH_TRY(launch_inv_diag<T>(n, dinv, w, ldw, s));
  for (int64_t h = kNB; h < n; h *= 2) LLH_TRY(launch_inv_level<T>(n, (int)h, a, lda, w, ldw, tmp, s));
  return launch_inv_wtw<T>(n, w, ldw, x, ldx, s);
}

template hipError_t potri_enqueue<double>(int, const double*, int64_t, const double*, double*, int64_t, double*,
                                          int64_t, double*, hipStream_t);
template hipError_t potri_enqueue<float>(int, const float*, int64_t, const float*, float*, int64_t, float*, int64_t,
                                         float*, hipStream_t);

template hipError_t potrf_enqueue<double>(double*, int64_t, int, int32_t*, bool, double*, hipStream_t,
                                          Profiler*, bool, const Lookahead*, _Float16*, const FwdFuse<double>*);
template hipError_t potrf_enqueue<float>(float*, int64_t, int, int32_t*, bool, float*, hipStream_t, Profiler*,
                                         bool, const Lookahead*, _Float16*, const FwdFuse<float>*);
template bool forward_fusable<double>(int, int, const Lookahead*);
template bool forward_fusable<float>(int, int, const Lookahead*);
template hipError_t factor_solve_enqueue<double>(double*, int64_t, int, int, double*, int64_t, double*, double*,
                                                 SolveSync*, int32_t*, hipStream_t, Profiler*, const Lookahead*);
template hipError_t factor_solve_enqueue<float>(float*, int64_t, int, int, float*, int64_t, float*, float*,
                                                SolveSync*, int32_t*, hipStream_t, Profiler*, const Lookahead*);
template hipError_t solve_pair_enqueue<double>(int, const double*, int64_t, int, double*, int64_t, const double*,
                                               SolveSync*, hipStream_t, Profiler*, const int32_t*);
template hipError_t solve_pair_enqueue<float>(int, const float*, int64_t, int, float*, int64_t, const float*,
                                              SolveSync*, hipStream_t, Profiler*, const int32_t*);
template hipError_t trsm_enqueue<double>(bool, bool, int, const double*, int64_t, int, double*, int64_t,
                                         const double*, bool, double*, SolveSync*, hipStream_t, Profiler*,
                                         const int32_t*);
template hipError_t trsm_enqueue<float>(bool, bool, int, const float*, int64_t, int, float*, int64_t,
                                        const float*, bool, float*, SolveSync*, hipStream_t, Profiler*,
                                        const int32_t*);

hipError_t solve_sync_begin(const SolveSync& sync, hipStream_t s) {
  if (sync.words == nullptr) return hipSuccess;
  return launch_fill_i32(sync.words + 1, 0, 1, s);
}

}  // namespace llh
