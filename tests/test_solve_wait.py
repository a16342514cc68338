"""The rule of the one-launch triangular solve's waits (csrc/llh_wait.h), compiled for the
host: a wait ends on its bound, on another workgroup's error and on the factor's gate.
On the GPU, failing factors that a substitution runs beside."""
import os
import subprocess
import time

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "linfa-linalg_amd", "csrc")

PROGRAM = r"""
#include <cstdio>

#include "llh_wait.h"

using namespace llh;

// Workgroups of one chain.  Each takes its ticket, reads the gate as `sees` tells and
// leaves or goes on; one that goes on publishes once the position before it has, and
// polls until then.  From poll `set_at` on the gate word itself holds a failed row.
// Returns the polls of the longest wait, or -1 where an error was recorded.
static int64_t chain(int n, const bool* sees, int64_t set_at, int64_t limit, bool* published) {
  constexpr int32_t kClear = 0x7fffffff;
  int64_t longest = 0;
  for (int p = 0; p < n; ++p) {
    published[p] = false;
    if (sees[p]) continue;  // left on the gate: its position is never published
    if (p > 0 && !published[p - 1]) {
      int64_t polls = 0;
      Wait w = Wait::kGoOn;
      while ((w = wait_step(polls, limit, kClear, [] { return 0; }, [&] { return polls >= set_at ? 5 : kClear; })) ==
             Wait::kGoOn) {
      }
      longest = polls > longest ? polls : longest;
      if (w == Wait::kGiveUp) return -1;
      continue;
    }
    published[p] = true;
  }
  return longest;
}

int main() {
  constexpr int64_t kLimit = 1ll << 22;
  constexpr int kN = 6;
  bool published[kN];
  // every way in which some positions have seen the gate and others have not
  for (int mask = 0; mask < 1 << kN; ++mask) {
    bool sees[kN];
    for (int p = 0; p < kN; ++p) sees[p] = mask >> p & 1;
    const int64_t polls = chain(kN, sees, 100, kLimit, published);
    if (polls < 0 || polls > 108) return std::printf("mask %d: %lld polls\n", mask, (long long)polls), 1;
  }
  int64_t polls = 0;
  const auto none = [] { return 0; };
  const auto clear = [] { return 7; };
  if (wait_step(polls, -1, 7, none, clear) != Wait::kGiveUp) return 2;  // a forced failure
  for (polls = 0; wait_step(polls, 20, 7, none, clear) == Wait::kGoOn;) {
  }
  if (polls != 21) return 3;  // the bound
  polls = 0;
  Wait w = Wait::kGoOn;
  while ((w = wait_step(polls, 20, 7, [] { return 1; }, clear)) == Wait::kGoOn) {
  }
  if (w != Wait::kGiveUp || polls != 8) return 4;  // another workgroup's error
  return 0;
}
"""


def test_waits_end(tmp_path):
    src, exe = tmp_path / "wait.cpp", tmp_path / "wait"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-I", CSRC, "-o", str(exe), str(src)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, (r.returncode, r.stdout)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", ["float64", "float32"])
# rows in the second panel, among its last columns, and in the last panel
@pytest.mark.parametrize("f", [512, 600, 1023, 1700, 5199])
def test_failure_beside_the_forward_substitution(f, dtype):
    """The factor fails while an earlier panel's substitution runs beside it."""
    import torch

    import linfa_linalg_hip as llh
    n, m = 5200, 64
    g = torch.Generator(device="cuda").manual_seed(f)
    b = torch.randn(n, n, dtype=torch.float64, device="cuda", generator=g)
    a = b @ b.T / n
    a.diagonal().add_(1.0)
    l = torch.linalg.cholesky(a[: f + 1, : f + 1])
    a[f, f] = (l[f, :f] ** 2).sum() - 0.5
    a = a.to(getattr(torch, dtype))
    rhs = torch.randn(n, m, dtype=a.dtype, device="cuda", generator=g)
    for _ in range(3):
        x = rhs.clone()
        t = time.perf_counter()
        with pytest.raises(llh.NotPositiveDefinite) as e:
            llh.device.solvec(a.clone(), x)
        assert time.perf_counter() - t < 0.5  # the factor takes milliseconds, a wait's bound seconds
        assert e.value.column == f and torch.equal(x, rhs)
