// Triangular solves on small diagonal blocks.
//
// trsv_block: the diagonal-block step of the blocked triangular solve: one
// thread owns one right-hand-side column, held in registers, swept exactly as
// triangular.rs:113-125 sweeps it (divide by the pivot, then update the rest of
// the column), restricted to b <= 64 rows.
#include "llh_common.h"
#include "llh_kernels.h"
#include "k_gemm_impl.h"
#include "k_trsm_impl.h"
#include "llh_wait.h"

#include <type_traits>
#include <utility>

namespace llh {
namespace {

template <typename T, bool UPPER_OP>
__global__ __launch_bounds__(64) void trsv_block_kernel(int b, bool trans, const T* __restrict__ Tm,
                                                        int64_t ldt, int m, T* __restrict__ Y, int64_t ldy,
                                                        const int32_t* __restrict__ gate) {
  if (gate != nullptr && *gate != kNoFail) return;
  // St[c * kNB + r] = op(T)[r, c], only op(T)'s triangle: column c of op(T) is
  // contiguous, which is what the column sweep reads.
  __shared__ __attribute__((aligned(16))) T St[kNB * kNB];
  const int tid = threadIdx.x;
  for (int e = tid; e < kNB * kNB; e += 64) {
    const int i = e / kNB, j = e % kNB;               // reads T[i, j], coalesced over j
    const int r = trans ? j : i, c = trans ? i : j;   // T[i, j] is op(T)[r, c]
    const bool in = r < b && c < b && (UPPER_OP ? c >= r : c <= r);
    St[c * kNB + r] = in ? Tm[(int64_t)i * ldt + j] : T(0);
  }
  __syncthreads();
  const int col = blockIdx.x * 64 + tid;
  if (col >= m) return;
  T y[kNB];
#pragma unroll
  for (int r = 0; r < kNB; ++r) y[r] = (r < b) ? Y[(int64_t)r * ldy + col] : T(0);
  if constexpr (!UPPER_OP) {
#pragma unroll
    for (int r = 0; r < kNB; ++r) {
      if (r < b) {
        y[r] = y[r] / St[r * kNB + r];
#pragma unroll
        for (int p = r + 1; p < kNB; ++p) y[p] -= y[r] * St[r * kNB + p];
      }
    }
  } else {
#pragma unroll
    for (int r = kNB - 1; r >= 0; --r) {
      if (r < b) {
        y[r] = y[r] / St[r * kNB + r];
#pragma unroll
        for (int p = 0; p < r; ++p) y[p] -= y[r] * St[r * kNB + p];
      }
    }
  }
#pragma unroll
  for (int r = 0; r < kNB; ++r)
    if (r < b) Y[(int64_t)r * ldy + col] = y[r];
}

// trtri64: one workgroup per diagonal block (trtri64_block, k_trsm_impl.h).
template <typename TS, typename T>
__global__ __launch_bounds__(256) void trtri64_kernel(int n, const TS* __restrict__ A, int64_t lda, bool trans,
                                                      bool upper, TS* __restrict__ out,
                                                      const int32_t* __restrict__ gate) {
  if (gate != nullptr && *gate != kNoFail) return;
  __shared__ T Ms[kNB * (kNB + 1)];
  __shared__ T Xs[kNB * (kNB + 1)];
  __shared__ T Ts[kNB * (kNB + 1)];
  const int o = blockIdx.x * kNB;
  trtri64_block<TS, TS, T>(min(kNB, n - o), A + (int64_t)o * lda + o, lda, trans, upper,
                       out + (int64_t)blockIdx.x * kNB * kNB, Ms, Xs, Ts);
}

// ---------------------------------------------------------------------------
// trsm_persistent: op(A) X = B in place for up to kSolveChunk right-hand-side
// columns per workgroup, one launch for the whole solve.
//
// Workgroups take tickets in launch order, every one of them, and the last sets the
// counter back (a launch of its own for that cost 5 us a solve); ticket t is (position
// p, column chunk q).  Position p is block row w = p (forward, op(A) lower) or w = nb-1-p
// (backward).  The workgroup accumulates sum_j op(A)_wj X_j over the blocks j
// that precede w in solve order, then solves op(A)_ww X_w = B_w - sum and
// publishes X_w.  A workgroup only ever waits for
// positions taken before its own, so the chain always advances whatever the
// residency.
//
// What bounds it: the chain of nb hops.  Only the last dependencies lie on it, so
// the workgroup does everything else before it waits for them.
//
// SUBST = false, up to 64 columns: X_w = inv(op(A)_ww) (B_w - sum) with the
// precomputed inverse of the diagonal block.  With l1 and l2 the
// blocks solved just before w (l1 last), it forms at the start
// G_i = inv(op(A)_ww) op(A)_w,li (in registers, as MFMA operands); after the other
// blocks, Z = inv(op(A)_ww) (B_w - sum_{j != l1, l2} op(A)_wj X_j); then Z -= G_2 X_l2
// and X_w = Z - G_1 X_l1.  A hop is then one transfer between CUs and one 64 x 64 x 16
// product on MFMA, 16 rows a wave, without a reduction.
//
// SUBST = true, more than 64 columns: each diagonal block is substituted, row by row
// (triangular.rs:113-125), as trsv_block does it, so that the
// residual stays that of a substitution whatever the block's condition, and an infinity
// or a NaN in a row of A or B reaches the rows after it only (an inverse's zeros would
// carry it to all 64: 0 x Inf).  Every block is walked, the wave partial sums are
// reduced, and each wave sweeps four columns, four rows of one a lane: 64 steps of a
// product with the pivot's reciprocal, a broadcast of it and up to four FMAs.
//
// The transfer is one store and one load: each 32-bit half of X_w travels in a 64-bit
// word beside a tag of the call and position (relaxed atomics of agent scope, which
// go past the L2s), so a reader polls the data itself instead of a flag, and neither
// side needs a fence (a release writes the whole L2 back, an acquire drops it).  The
// words lie in a ring of kMailRing blocks a chunk.  Only the kMailReach positions after
// a block read it there, and a position publishes after it has read its own
// dependencies, so a block's slot is free once its successor kMailRing later is
// reached (kMailReach < kMailRing).  Positions further behind read B itself, once the
// block's flag, raised after its stores have reached memory, holds the call's epoch.
//
// The walk over the other blocks is split by k: wave v multiplies columns
// [16 v, 16 v + 16) of each tile for all 64 rows, with both operands loaded straight
// into registers (tiles one block ahead), and polls for itself, so it has no barrier;
// the wave partial sums are reduced once.
//
// Against one flag per block between fences, with the products on the VALU (us a
// hop, n = 12000 and m = 16): f64 6.7 -> 2.8, f32 5.0 -> 2.0; whole solves (us): n = 4096,
// m = 64 f64 507 -> 195, f32 431 -> 156.  A hop with SUBST f64 5.0, f32 3.6 (n = 4096, m = 66);
// whole solves, against a launch per block and product: n = 4096, m = 300 f64 4461 -> 371,
// f32 3832 -> 286 (multiplying by the inverses would take 370 and 273).
//
// Why the line is at 64 columns: a solve of so few is little but the chain, whose hop is
// 2.8 against 5.0 us in f64, and its blocks have always been inverted; a wider one's
// substitution hides behind its products.
//
// The wait is bounded: past spin_limit polls (or once another workgroup has
// given up) the workgroup records an error and returns without publishing.
// A negative spin_limit makes every wait give up at once (a host-forced failure
// for tests of the error path; every workgroup still exits normally).  With a
// gate (the factor's status word) that holds a failed row, every workgroup
// returns at once and B is left untouched; where the gate is set while the launch runs,
// the waits end on it too, without an error (wait_step), and B may be partly solved.
constexpr int kSolveChunk = kSolveChunkHost;
constexpr int kFlagWindow = 64;  // flags checked ahead per wait
constexpr int kMailReach = 4;    // positions that read a block from the ring
static_assert(kMailReach < kMailRing, "a slot's readers have published before it is written again");
static_assert(kMailSlot >= 2 * kNB * kSolveChunkHost, "a block's words fit its slot");

// Relaxed loads and stores of agent scope, on the value's bits.
template <typename T>
__device__ __forceinline__ T agent_load(const T* p) {
  if constexpr (sizeof(T) == 8)
    return __builtin_bit_cast(T, __hip_atomic_load(reinterpret_cast<const uint64_t*>(p), __ATOMIC_RELAXED,
                                                   __HIP_MEMORY_SCOPE_AGENT));
  else
    return __builtin_bit_cast(T, __hip_atomic_load(reinterpret_cast<const uint32_t*>(p), __ATOMIC_RELAXED,
                                                   __HIP_MEMORY_SCOPE_AGENT));
}
template <typename T>
__device__ __forceinline__ void agent_store(T* p, T v) {
  if constexpr (sizeof(T) == 8)
    __hip_atomic_store(reinterpret_cast<uint64_t*>(p), __builtin_bit_cast(uint64_t, v), __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_AGENT);
  else
    __hip_atomic_store(reinterpret_cast<uint32_t*>(p), __builtin_bit_cast(uint32_t, v), __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_AGENT);
}

// The value of lane I of each group of 16 lanes, in all of its lanes.
template <int I, typename T>
__device__ __forceinline__ T row_value(T v) {
  constexpr int kBcast = 0x150 + I;  // DPP row_newbcast
  if constexpr (sizeof(T) == 8) {
    const uint64_t u = __builtin_bit_cast(uint64_t, v);
    const uint32_t lo = __builtin_amdgcn_mov_dpp((int)u, kBcast, 0xf, 0xf, false);
    const uint32_t hi = __builtin_amdgcn_mov_dpp((int)(u >> 32), kBcast, 0xf, 0xf, false);
    return __builtin_bit_cast(T, (uint64_t)hi << 32 | lo);
  } else {
    return __builtin_bit_cast(T, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), kBcast, 0xf, 0xf, false));
  }
}

template <typename T, bool VEC, bool trans, bool SUBST>
__global__ __launch_bounds__(256, 2) void trsm_persistent_kernel(
    int n, int m, const T* __restrict__ A, int64_t lda, bool lower_op, const T* __restrict__ Dinv,
    bool dinv_t, T* B, int64_t ldb, int32_t* ticket, int32_t* flags, uint64_t* mail, int32_t epoch, int32_t* err,
    int64_t spin_limit, const int32_t* __restrict__ gate) {
  using MF = Mfma<T>;
  using acc_t = typename MF::acc_t;
  // kFar (f64): G_2 waits in LDS, since with both in registers some are spilled (3.6 us
  // a hop instead of 2.9; one workgroup per CU instead: 476 us for 416 at n = 4096, m = 300)
  constexpr bool kFar = sizeof(T) == 8 && !SUBST;
  // a slab's row k, column c is at sidx(k, c).  In f32 rows 4 apart go to different banks;
  // with SUBST a lane reads 16-byte pieces of a row, and every row is shifted by one.
  constexpr int VL = 16 / sizeof(T), MC = kSolveChunk, S = kNB + 1, RSTEP = SUBST ? MC + VL : MC;
  constexpr int PAD = SUBST || kFar ? 0 : MC, SL = kNB * RSTEP + kNB / 4 * PAD, NK = kNB / 4, LS = kNB + VL;
  static_assert(MC == 16 && kNB == 64, "one 16-column chunk, four waves of 16 rows or columns");
  // a staged tile of op(A) for G, then the four wave partials, then X_l2 and X_l1
  __shared__ __attribute__((aligned(16))) T Wk[SUBST || 4 * SL > kNB * S ? 4 * SL : kNB * S];
  // B_w - sum; with SUBST the diagonal block instead, its rows and columns in solve order,
  // and its diagonal
  __shared__ __attribute__((aligned(16))) T Slab[SUBST ? kNB * LS : SL];
  __shared__ T Dg[SUBST ? kNB : 1];
  __shared__ T Far[kFar ? 4 * NK * 64 : 1];
  __shared__ int s_ticket, s_abort[3];
  const int tid = threadIdx.x, lane = tid & 63, fr = lane & 15, fq = lane >> 4;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int nb = (n + kNB - 1) / kNB, nq = (m + MC - 1) / MC;
  if (tid == 0) s_ticket = atomicAdd(ticket, 1);
  if (tid < 3) s_abort[tid] = 0;
  __syncthreads();
  const int tk = __builtin_amdgcn_readfirstlane(s_ticket);
  // (the last ticket: no workgroup takes another one, the next launch starts at 0)
  if (tk == nb * nq - 1 && tid == 0) atomicExch(ticket, 0);
  if (gate != nullptr && *gate != kNoFail) return;
  const int p = tk / nq, q = tk % nq;
  const int w = lower_op ? p : nb - 1 - p;
  const int w0 = w * kNB, bw = min(kNB, n - w0);
  const int c0 = q * MC, mc = min(MC, m - c0);
  auto jof = [&](int st) { return lower_op ? st : nb - 1 - st; };
  auto sidx = [](int k, int c) { return k * RSTEP + (k >> 2) * PAD + c; };
  // where this lane's entries of B_w are: rows 16 wv + row(lane, e), column fr; with SUBST
  // rows 16 e + fr in solve order, column 4 wv + fq
  auto xrow = [&](int e) {
    return SUBST ? (lower_op ? 16 * e + fr : kNB - 1 - 16 * e - fr) : 16 * wv + MF::row(lane, e);
  };
  const int xc = SUBST ? 4 * wv + fq : fr;

  // the diagonal block, or this wave's rows of its inverse, in the order of the products' k
  T iv[NK];
  T d[4], rd[4];  // with SUBST: the pivots of rows 16 e + fr in solve order, their reciprocals
  bool odd = false;
  if constexpr (SUBST) {
    T v[NK];
#pragma unroll
    for (int e = 0; e < NK; ++e) {
      const int i = (tid + 256 * e) / kNB, jj = (tid + 256 * e) % kNB, r = trans ? jj : i, c = trans ? i : jj;
      const bool in = r < bw && c < bw && (lower_op ? c <= r : c >= r);
      v[e] = in ? A[(int64_t)(w0 + i) * lda + w0 + jj] : T(r == c ? 1 : 0);
    }
#pragma unroll
    for (int e = 0; e < NK; ++e) {
      const int i = (tid + 256 * e) / kNB, jj = (tid + 256 * e) % kNB, r = trans ? jj : i, c = trans ? i : jj;
      const int to = lower_op ? r : kNB - 1 - r;
      Slab[to * LS + (lower_op ? c : kNB - 1 - c)] = v[e];
      if (r == c) Dg[to] = v[e];
    }
    __syncthreads();
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      d[e] = Dg[16 * e + fr];
      rd[e] = T(1) / d[e];
      odd = odd || (!__builtin_isnormal(rd[e]) && d[e] != T(0) && __builtin_isfinite(d[e]));
    }
  } else {
    const T* D = Dinv + (int64_t)w * kNB * kNB;
#pragma unroll
    for (int e = 0; e < NK; ++e) {
      const int k = 16 * (e / 4) + MF::row(lane, e % 4), r = 16 * wv + fr;
      iv[e] = D[dinv_t ? k * kNB + r : r * kNB + k];
    }
  }
  T bwr[4];  // B_w
#pragma unroll
  for (int e = 0; e < 4; ++e)
    bwr[e] = (xrow(e) < bw && xc < mc) ? B[(int64_t)(w0 + xrow(e)) * ldb + c0 + xc] : T(0);

  // g = this wave's rows of inv(op(A)_ww) op(A)_wj, j at position st, as the operand of
  // a product over k in the order of iv (computed transposed, which leaves it so)
  auto make_g = [&](int st, T (&g)[NK]) __attribute__((always_inline)) {
    const int j0 = jof(st) * kNB, bj = min(kNB, n - j0);
    __syncthreads();
    T v[NK];
#pragma unroll
    for (int e = 0; e < NK; ++e) {
      const int i = (tid + 256 * e) / kNB, jj = (tid + 256 * e) % kNB, r = trans ? jj : i, c = trans ? i : jj;
      const int64_t rr = w0 + min(r, bw - 1);
      v[e] = c < bj ? A[trans ? (int64_t)(j0 + c) * lda + rr : rr * lda + j0 + c] : T(0);
    }
#pragma unroll
    for (int e = 0; e < NK; ++e) {
      const int i = (tid + 256 * e) / kNB, jj = (tid + 256 * e) % kNB, r = trans ? jj : i, c = trans ? i : jj;
      Wk[r * S + c] = v[e];
    }
    __syncthreads();
#pragma unroll
    for (int kt = 0; kt < 4; ++kt) {
      acc_t t{};
#pragma unroll
      for (int e = 0; e < NK; ++e)
        t = MF::mma(Wk[(16 * (e / 4) + MF::row(lane, e % 4)) * S + 16 * kt + fr], iv[e], t);
#pragma unroll
      for (int e = 0; e < 4; ++e) g[4 * kt + e] = t[e];
    }
  };
  T g1[NK], g2[NK];
  if constexpr (!SUBST) {
    if (p > 0) make_g(p - 1, g1);
    if (p > 1) make_g(p - 2, g2);
  }
  T* const far = Far + (kFar ? wv * NK * 64 + lane : 0);
  if constexpr (kFar) {
#pragma unroll
    for (int e = 0; e < NK; ++e) far[64 * e] = g2[e];
  }

  // The row of block w that MFMA row f of row tile i stands for: for op(A) = A^T a lane's
  // rows of the tiles lie side by side in memory (16-byte loads; n = 12000, m = 16 f64 3.9 -> 2.5 us a
  // hop, f32 2.8 -> 2.0).
  auto arow = [&](int i, int f) __attribute__((always_inline)) {
    return trans ? i / VL * 16 * VL + f * VL + i % VL : 16 * i + f;
  };
  // this lane's values of op(A)[w0 + arow(i, fr), j0 + 16 wv + 4 fq + e], at 4 i + e
  typedef T vec_t __attribute__((ext_vector_type(VL)));
  auto fetch = [&](int st, T (&out)[NK]) __attribute__((always_inline)) {
    const int j0 = jof(st) * kNB, bj = min(kNB, n - j0), k0 = 16 * wv + 4 * fq;
    if (trans && VEC && bj == kNB && bw == kNB) {
      const T* col = A + (int64_t)(j0 + k0) * lda + w0 + VL * fr;
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int v = 0; v < 4 / VL; ++v) {
          const vec_t x = *reinterpret_cast<const vec_t*>(col + (int64_t)e * lda + 16 * VL * v);
#pragma unroll
          for (int c = 0; c < VL; ++c) out[4 * (VL * v + c) + e] = x[c];
        }
      return;
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int64_t r = w0 + min(arow(i, fr), bw - 1);
      if (!trans) {
        const T* row = A + r * lda + j0 + k0;
        if (VEC && bj == kNB) {
#pragma unroll
          for (int v = 0; v < 4 / VL; ++v) {
            const vec_t x = *reinterpret_cast<const vec_t*>(row + v * VL);
#pragma unroll
            for (int e = 0; e < VL; ++e) out[4 * i + v * VL + e] = x[e];
          }
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e) out[4 * i + e] = (k0 + e < bj) ? row[e] : T(0);
        }
      } else {
        const T* col = A + (int64_t)(j0 + k0) * lda + r;
#pragma unroll
        for (int e = 0; e < 4; ++e) out[4 * i + e] = (k0 + e < bj) ? col[(int64_t)e * lda] : T(0);
      }
    }
  };
  // rows 16 wv + 4 fq + e of X_j, column fr, from B
  auto loadx = [&](int st, T (&out)[4]) __attribute__((always_inline)) {
    const int j0 = jof(st) * kNB, bj = min(kNB, n - j0), k0 = 16 * wv + 4 * fq;
#pragma unroll
    for (int e = 0; e < 4; ++e)
      out[e] = (k0 + e < bj && fr < mc) ? agent_load(&B[(int64_t)(j0 + k0 + e) * ldb + c0 + fr]) : T(0);
  };
  // one more poll of a wait: false once it gives up or leaves
  auto go_on = [&](int64_t& it, int stage) -> bool {
    const Wait next = wait_step(
        it, spin_limit, kNoFail, [&] { return agent_load(err); },
        [&] { return gate != nullptr ? agent_load(gate) : kNoFail; });
    if (next == Wait::kGoOn) return true;
    if (lane == 0) {
      if (next == Wait::kGiveUp) atomicExch(err, 1);
      s_abort[stage] = 1;
    }
    return false;
  };
  // wait until block st's flag is raised, then take every later flag already
  // raised (up to the window); false when the wait gave up
  int ready = 0;
  auto wait_for = [&](int st) -> bool {
    const int32_t* f = &flags[jof(st) * nq + q];
    int64_t it = 0;
    bool go = spin_limit >= 0 || go_on(it, 0);
    while (go && __hip_atomic_load(f, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != epoch) {
      go = go_on(it, 0);
      __builtin_amdgcn_s_sleep(1);
    }
    if (!go) return false;
    const int t2 = st + 1 + lane;
    const bool up = lane < kFlagWindow - 1 && t2 < p &&
                    __hip_atomic_load(&flags[jof(min(t2, p - 1)) * nq + q], __ATOMIC_RELAXED,
                                      __HIP_MEMORY_SCOPE_AGENT) == epoch;
    const uint64_t down = ~(uint64_t)__ballot(up);  // (lane 63 is never up)
    ready = __builtin_amdgcn_readfirstlane(st + 1 + __builtin_ctzll(down));
    asm volatile("" ::: "memory");
    return true;
  };
  // words o[e] of block st from the ring, once all of them carry its tag
  uint64_t* const ring = mail + (int64_t)q * kMailRing * kMailSlot;
  auto take = [&](int st, int o0, int step, T (&out)[4], int stage) -> bool {
    const uint64_t* box = ring + (st % kMailRing) * kMailSlot + o0;
    const uint32_t tag = (uint32_t)epoch + (uint32_t)(st / kMailRing);
    int64_t it = 0;
    if (spin_limit < 0 && !go_on(it, stage)) return false;
    for (;;) {
      uint64_t lo[4], hi[4];
      bool got = true;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        lo[e] = agent_load(box + step * e);
        if constexpr (sizeof(T) == 8) hi[e] = agent_load(box + step * e + kNB * MC);
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        got = got && (uint32_t)(lo[e] >> 32) == tag;
        if constexpr (sizeof(T) == 8) {
          got = got && (uint32_t)(hi[e] >> 32) == tag;
          out[e] = __builtin_bit_cast(double, (hi[e] << 32) | (uint32_t)lo[e]);
        } else {
          out[e] = __builtin_bit_cast(float, (uint32_t)lo[e]);
        }
      }
      if (__ballot(!got) == 0) return true;
      if (!go_on(it, stage)) return false;
    }
  };

  // the walk over the blocks before w, or before l2
  const int nwalk = SUBST ? p : max(p - 2, 0);
  acc_t acc[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) acc[i] = acc_t{};
  {
    T a_cur[NK], a_nxt[NK], x_cur[4], x_nxt[4];
    bool x_pre = false;
    if (nwalk > 0) fetch(0, a_cur);
    for (int st = 0; st < nwalk; ++st) {
      if (x_pre) {
#pragma unroll
        for (int e = 0; e < 4; ++e) x_cur[e] = x_nxt[e];
      } else if (st >= ready && st >= p - kMailReach) {
        if (!take(st, (16 * wv + 4 * fq) * MC + fr, MC, x_cur, 0)) break;
      } else {
        if (st >= ready && !wait_for(st)) break;
        loadx(st, x_cur);
      }
      if (st + 1 < nwalk) fetch(st + 1, a_nxt);
      x_pre = st + 1 < nwalk && st + 1 < ready;
      if (x_pre) loadx(st + 1, x_nxt);
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[i] = MF::mma(a_cur[4 * i + e], x_cur[e], acc[i]);
#pragma unroll
      for (int e = 0; e < NK; ++e) a_cur[e] = a_nxt[e];
    }
  }

  __syncthreads();  // every wave is done with the staged tile
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int e = 0; e < 4; ++e) Wk[wv * SL + sidx(arow(i, MF::row(lane, e)), fr)] = acc[i][e];
  __syncthreads();
  if (s_abort[0]) return;
  // B_w - sum, the wave partials reduced
  T rhs[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const int o = sidx(xrow(e), xc);
    const T sum = Wk[o] + Wk[SL + o] + Wk[2 * SL + o] + Wk[3 * SL + o];
    rhs[e] = (xrow(e) < bw && xc < mc) ? bwr[e] - sum : T(0);
  }
  T out[4];  // X_w
  if constexpr (SUBST) {
    // row 16 e + fr, column fq of the wave's four: the broadcast of a row's value to its
    // column's other rows stays within 16 lanes
    auto sweep = [&](auto divide) __attribute__((always_inline)) {
      static_for(std::make_integer_sequence<int, 4>{}, [&](auto bc) __attribute__((always_inline)) {
        constexpr int b = decltype(bc)::value;
        T sum[4] = {T(0), T(0), T(0), T(0)};  // of these 16 columns, for the rows of later blocks
        static_for(std::make_integer_sequence<int, 16 / VL>{}, [&](auto gc) __attribute__((always_inline)) {
          constexpr int i0 = decltype(gc)::value * VL;
          vec_t l[4];
#pragma unroll
          for (int e = b; e < 4; ++e)
            l[e] = *reinterpret_cast<const vec_t*>(&Slab[(16 * e + fr) * LS + 16 * b + i0]);
          static_for(std::make_integer_sequence<int, VL>{}, [&](auto vc) __attribute__((always_inline)) {
            constexpr int v = decltype(vc)::value, i = i0 + v;
            const T q = row_value<i>(decltype(divide)::value ? rhs[b] / d[b] : rhs[b] * rd[b]);
            const T u = __builtin_elementwise_fma(-l[b][v], q, rhs[b]);
            rhs[b] = fr > i ? u : rhs[b];
#pragma unroll
            for (int e = b + 1; e < 4; ++e) sum[e] = __builtin_elementwise_fma(l[e][v], q, sum[e]);
          });
        });
#pragma unroll
        for (int e = b + 1; e < 4; ++e) rhs[e] -= sum[e];
      });
    };
    // (pivots whose reciprocal is no normal number are divided by; those of 0 and
    // infinity give the quotient's infinities, zeros and NaNs as they are)
    if (__ballot(odd) == 0)
      sweep(std::false_type{});
    else
      sweep(std::true_type{});
    // through LDS (this wave's columns of the first partial), so that a store takes whole rows
#pragma unroll
    for (int e = 0; e < 4; ++e) Wk[sidx(xrow(e), xc)] = rhs[e] / d[e];
    __syncthreads();
#pragma unroll
    for (int e = 0; e < 4; ++e) out[e] = Wk[sidx(tid / MC + kNB / 4 * e, tid % MC)];
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e) Slab[sidx(xrow(e), fr)] = rhs[e];
    __syncthreads();
    // f x slab, in f32 as four sums of 16 terms (less rounding than one of 64)
    auto product = [&](const T (&f)[NK], const T* slab) __attribute__((always_inline)) -> acc_t {
      constexpr int NP = sizeof(T) == 4 ? 4 : 1;
      acc_t t[NP];
#pragma unroll
      for (int i = 0; i < NP; ++i) t[i] = acc_t{};
#pragma unroll
      for (int e = 0; e < NK; ++e)
        t[e % NP] = MF::mma(f[e], slab[sidx(16 * (e / 4) + MF::row(lane, e % 4), fr)], t[e % NP]);
      if constexpr (NP == 4) return (t[0] + t[1]) + (t[2] + t[3]);
      return t[0];
    };
    acc_t x = product(iv, Slab);  // Z
    // x -= G X for the dependency at position st, 16 of whose rows each wave takes
    auto apply_g = [&](int st, const T (&g)[NK], int stage) __attribute__((always_inline)) -> bool {
      T y[4];
      T* const slab = Wk + (stage - 1) * SL;
      if (take(st, 16 * MC * wv + lane, 4 * MC, y, stage)) {
#pragma unroll
        for (int e = 0; e < 4; ++e) slab[sidx(16 * wv + 4 * e + fq, fr)] = y[e];
      }
      __syncthreads();
      if (s_abort[stage]) return false;
      const acc_t t = product(g, slab);
#pragma unroll
      for (int e = 0; e < 4; ++e) x[e] -= t[e];
      return true;
    };
    if (p > 1) {
      if constexpr (kFar) {
#pragma unroll
        for (int e = 0; e < NK; ++e) g2[e] = far[64 * e];
      }
      if (!apply_g(p - 2, g2, 1)) return;
    }
    if (p > 0 && !apply_g(p - 1, g1, 2)) return;
#pragma unroll
    for (int e = 0; e < 4; ++e) out[e] = x[e];
  }
  // row and column of out[e]
  auto orow = [&](int e) { return SUBST ? tid / MC + kNB / 4 * e : 16 * wv + MF::row(lane, e); };
  const int oc = SUBST ? tid % MC : fr;
  if (p + 1 < nb) {
    uint64_t* box = ring + (p % kMailRing) * kMailSlot;
    const uint64_t tag = (uint64_t)((uint32_t)epoch + (uint32_t)(p / kMailRing)) << 32;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int r = orow(e);
      const T v = r < bw ? out[e] : T(0);
      if constexpr (sizeof(T) == 8) {
        const uint64_t u = __builtin_bit_cast(uint64_t, v);
        agent_store(box + r * MC + oc, tag | (uint32_t)u);
        agent_store(box + kNB * MC + r * MC + oc, tag | (u >> 32));
      } else {
        agent_store(box + r * MC + oc, tag | __builtin_bit_cast(uint32_t, v));
      }
    }
  }
#pragma unroll
  for (int e = 0; e < 4; ++e)
    if (orow(e) < bw && oc < mc) agent_store(&B[(int64_t)(w0 + orow(e)) * ldb + c0 + oc], out[e]);
  if (p + kMailReach + 1 >= nb) return;  // no position reads this flag
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this wave's stores have reached memory
  __syncthreads();
  if (tid == 0) __hip_atomic_store(&flags[w * nq + q], epoch, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

}  // namespace

template <typename T>
hipError_t launch_trsv_block(bool upper_op, bool trans, int b, const T* Tm, int64_t ldt, int m, T* Y,
                             int64_t ldy, const int32_t* gate, hipStream_t s) {
  if (m <= 0 || b <= 0) return hipSuccess;
  if (b > kNB) return hipErrorInvalidValue;
  const dim3 grid((m + 63) / 64);
  if (upper_op)
    hipLaunchKernelGGL((trsv_block_kernel<T, true>), grid, dim3(64), 0, s, b, trans, Tm, ldt, m, Y, ldy, gate);
  else
    hipLaunchKernelGGL((trsv_block_kernel<T, false>), grid, dim3(64), 0, s, b, trans, Tm, ldt, m, Y, ldy, gate);
  return hipGetLastError();
}

template <typename TS, typename T>
hipError_t launch_trtri_blocks(int n, const TS* A, int64_t lda, bool trans, bool upper, TS* out,
                               const int32_t* gate, hipStream_t s) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL((trtri64_kernel<TS, T>), dim3((n + kNB - 1) / kNB), dim3(256), 0, s, n, A, lda, trans,
                     upper, out, gate);
  return hipGetLastError();
}

template <typename T>
hipError_t launch_trsm_persistent(int n, int m, const T* A, int64_t lda, bool trans, bool lower_op,
                                  const T* Dinv, bool dinv_t, T* B, int64_t ldb, int32_t* ticket,
                                  int32_t* flags, uint64_t* mail, int32_t epoch, int32_t* err,
                                  int64_t spin_limit, const int32_t* gate, hipStream_t s) {
  if (n <= 0 || m <= 0) return hipSuccess;
  const int nb = (n + kNB - 1) / kNB, nq = (m + kSolveChunk - 1) / kSolveChunk;
  const bool vec = (reinterpret_cast<uintptr_t>(A) % 16 == 0) && ((lda * sizeof(T)) % 16 == 0);
  auto go = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3(nb * nq), dim3(256), 0, s, n, m, A, lda, lower_op, Dinv, dinv_t, B, ldb, ticket,
                       flags, mail, epoch, err, spin_limit, gate);
  };
  if (Dinv == nullptr) {
    if (vec) trans ? go(trsm_persistent_kernel<T, true, true, true>) : go(trsm_persistent_kernel<T, true, false, true>);
    else trans ? go(trsm_persistent_kernel<T, false, true, true>) : go(trsm_persistent_kernel<T, false, false, true>);
  } else {
    if (vec) trans ? go(trsm_persistent_kernel<T, true, true, false>) : go(trsm_persistent_kernel<T, true, false, false>);
    else trans ? go(trsm_persistent_kernel<T, false, true, false>) : go(trsm_persistent_kernel<T, false, false, false>);
  }
  return hipGetLastError();
}

template hipError_t launch_trtri_blocks<double, double>(int, const double*, int64_t, bool, bool, double*,
                                                        const int32_t*, hipStream_t);
template hipError_t launch_trtri_blocks<float, float>(int, const float*, int64_t, bool, bool, float*,
                                                      const int32_t*, hipStream_t);
template hipError_t launch_trtri_blocks<float, double>(int, const float*, int64_t, bool, bool, float*,
                                                       const int32_t*, hipStream_t);
template hipError_t launch_trsm_persistent<double>(int, int, const double*, int64_t, bool, bool, const double*,
                                                   bool, double*, int64_t, int32_t*, int32_t*, uint64_t*, int32_t,
                                                   int32_t*, int64_t, const int32_t*, hipStream_t);
template hipError_t launch_trsm_persistent<float>(int, int, const float*, int64_t, bool, bool, const float*, bool,
                                                  float*, int64_t, int32_t*, int32_t*, uint64_t*, int32_t, int32_t*,
                                                  int64_t, const int32_t*, hipStream_t);
template hipError_t launch_trsv_block<double>(bool, bool, int, const double*, int64_t, int, double*, int64_t,
                                              const int32_t*, hipStream_t);
template hipError_t launch_trsv_block<float>(bool, bool, int, const float*, int64_t, int, float*, int64_t,
                                             const int32_t*, hipStream_t);

}  // namespace llh
