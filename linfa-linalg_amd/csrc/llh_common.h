// Shared definitions for the linfa-linalg-hip kernels and host drivers (gfx950).
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstdint>
#include <type_traits>
#include <utility>

namespace llh {

// Status word written by the factor kernels: the first failing row of the
// `d <= 0` pivot test (cholesky.rs:69), or kNoFail.
constexpr int32_t kNoFail = 0x7fffffff;

// Block sizes of the blocked right-looking POTRF: kNB is the width of the
// diagonal block factored in LDS and of the panel solved row by row; the outer
// panel width, the rank of the trailing SYRK update on MFMA, is kNBO, or
// kNBO_LARGE for an order of at least kNBO_LARGE_N when the SYRK runs on f64 or
// f32 operands (outer_width()).  Wider panels give each output tile more MFMA
// k-slabs per read-modify-write of C but a longer panel chain.  Measured: solve n =
// 32768 f64 194.7 / 195.9 / 198.6 ms at 1024 / 768 / 1536, FP32 refined 137.0 / 138.5 /
// 137.8; potrf n = 16384 f64 29.5 / 29.7 ms at 512 / 1024; the f16-operand factor, whose SYRK is fast and
// whose panel chain sets the pace, 87 / 95 ms at 512 / 1024 (n = 32768), and later
// FP16+IR 88.5 / 78.1 / 70.8 ms at 256 / 384 / 512 (narrower panels pass over the
// f32 trailing matrix more often).
constexpr int kNB = 64;
constexpr int kNBO = 512;
constexpr int kNBO_LARGE = 1024;
constexpr int kNBO_LARGE_N = 24576;
inline int outer_width(int n, bool half_syrk) { return (!half_syrk && n >= kNBO_LARGE_N) ? kNBO_LARGE : kNBO; }

// The last kStepTail columns are one panel (their updates ride on the step
// launches below), those before it outer_width panels.  Measured (potrf, us) with a tail of 2048 / 4096 / 6144:
// f64 n = 3000 1106 / 952, 5003 2561 / 2580 / 2601, 8192 5894 / 5952 / 6930; f32
// n = 3000 835 / 756, 5003 1960 / 1890 / 1886, 8192 3882 / 3898 / 4455.
constexpr int kStepTail = 4096;
inline int panel_width(int rem, int n, bool half_syrk) { return rem <= kStepTail ? rem : outer_width(n, half_syrk); }

// The panel step at block column k0 applies step_rank columns before it to later block
// columns, all of them or, with step_ahead, the next one (k_step.hip); T: the type its
// diagonal block is factored in.
template <typename T>
__host__ __device__ inline bool step_ahead(int k0, int p0) { return sizeof(T) == 4 && (k0 - p0) / kNB % 2 != 0; }
template <typename T>
__host__ __device__ inline int step_rank(int k0, int p0) { return sizeof(T) == 8 || step_ahead<T>(k0, p0) ? kNB : 2 * kNB; }

// A panel of at most so many rows is stepped through with all of them: every step's
// launch solves the rows below as well.  With more, the steps take the panel's top
// block alone, beside the trailing update, and the rows below follow in one launch:
// the repeated work and the rank-64 updates of many rows would take more from the
// trailing update than the shorter chain gives.  Measured (potrf, ms) with bounds of
// 0 / 6144 / 8192 / 12288 rows: f64 n = 6000 3.50 / 3.28 / 3.28 / 3.29, 8192 6.18 / 5.98 /
// 5.81 / 5.81, 12000 13.7 / 13.6 / 13.5 / 13.5, 20000 50.2 / 50.3 / 50.0 / 50.1; f32
// n = 8192 4.00 / 3.92 / 3.87 / 3.88, 12000 8.43 / 8.45 / 8.40 / 8.55, 16384 17.5 / 17.4 /
// 17.4 / 17.7.
constexpr int kStepRows = 8192;

// Right-hand-side columns per workgroup of the one-launch triangular solve, and
// the bound on its flag waits (2^22 polls: well over 0.1 s, far above any real wait).
constexpr int kSolveChunkHost = 16;
constexpr int64_t kSpinLimit = 1ll << 22;
// The blocks that the solve's workgroups hand to their successors: a ring of kMailRing
// blocks of kMailSlot 64-bit words (a 32-bit half and its tag) per column chunk, for
// up to kMailChunks chunks a launch (16 MB).
constexpr int kMailRing = 8;
constexpr int kMailSlot = 2 * kNB * kSolveChunkHost;
constexpr int kMailChunks = 128;
inline int64_t solve_mail_words(int64_t chunks) { return chunks * kMailRing * kMailSlot; }
// Tags that a launch of n rows takes: one per lap of the ring.
inline int solve_epochs(int n) { return ((n + kNB - 1) / kNB + kMailRing - 1) / kMailRing; }

// Rows that one launch of the triangular solve takes for m right-hand sides
// (trsm_split): all of them up to 64 columns, where the chain of 64-row hops
// bounds it; with more columns n * m = 6M, about as many as keep its products
// shorter than that chain, the rest as products with larger tiles between launches.
// Measured (us, L / L^T) at 1.5M, 3M, 6M, 12M: f64 n = 4096 m = 1500 1393 / 1347, 1116 /
// 1047, 957 / 885, 1001 / 925, n = 12000 m = 500 3730 / 3560, 2894 / 2800, 2462 / 2380,
// 2622 / 2579; f32 n = 4096 m = 1500 892 / 932, 765 / 747, 690 / 592, 678 / 541, n = 12000
// m = 500 2391 / 2427, 1916 / 1921, 1630 / 1512, 1995 / 1433, m = 1500 4622 / 4568, 4298 /
// 4016, 4133 / 3701, 3901 / 3419.
constexpr int kSolveMaxCols = 32768;
template <typename T>
inline int solve_split(int m) {
  if (m <= 64) return INT32_MAX;
  const int rows = 6000000 / m / kNB * kNB;
  return rows > kNB ? rows : kNB;
}
// Flags that the largest of those launches needs for order n.
template <typename T>
inline int64_t solve_flags(int n, int m) {
  const int64_t nb = (n + kNB - 1) / kNB, per = (int64_t)solve_split<T>(m) / kNB;
  return (nb < per ? nb : per) * ((m + kSolveChunkHost - 1) / kSolveChunkHost);
}

// Largest n the single-workgroup LDS kernel takes (the packed lower triangle of
// an f64 matrix must fit in 160 KiB of LDS with room to spare).
constexpr int kSmallMaxD = 128;
constexpr int kSmallMaxS = 176;

// Exact-order arithmetic.  The files that use these helpers are compiled with
// -ffp-contract=off and open with `#pragma clang fp contract(off)`, so every
// `s += x*y` stays a separately rounded multiply and add, as the reference's
// compiled Rust is.  IEEE division and square root are correctly rounded on
// gfx950 for f64 and, without fast-math flags, for f32.
template <typename T>
__device__ __forceinline__ T sqrt_rn(T a);
template <>
__device__ __forceinline__ double sqrt_rn<double>(double a) { return __builtin_sqrt(a); }
template <>
__device__ __forceinline__ float sqrt_rn<float>(float a) { return __builtin_sqrtf(a); }

// Calls f(std::integral_constant<int, I>) for I = 0 .. n-1: loops are
// expanded at compile time, so every index into the register arrays is a
// constant (a rolled loop would move them to scratch memory).
template <typename F, int... I>
__device__ __forceinline__ void static_for(std::integer_sequence<int, I...>, F&& f) {
  (f(std::integral_constant<int, I>{}), ...);
}

}  // namespace llh
