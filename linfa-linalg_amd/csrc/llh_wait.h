// The rule of a bounded wait inside a kernel: constexpr, so that the host tests run it.
#pragma once

#include <cstdint>

namespace llh {

enum class Wait {
  kGoOn,    // poll again
  kGiveUp,  // the bound is reached, or another workgroup has given up: record the error
  kLeave,   // the gate holds a failed row: no error, what is waited for may never come
};

// After a poll that found nothing.  A workgroup takes its ticket whatever the gate holds
// and then leaves where it holds a failed row, while a later one may still have read it
// clear (the factor runs beside the solve): the wait of that one ends on the gate too, or
// it would poll to the bound.  error and gate load the words past the L2s; they are
// looked at every eighth poll.
template <typename Error, typename Gate>
constexpr Wait wait_step(int64_t& polls, int64_t limit, int32_t clear, Error&& error, Gate&& gate) {
  if (limit < 0 || ++polls > limit) return Wait::kGiveUp;
  if ((polls & 7) != 0) return Wait::kGoOn;
  if (gate() != clear) return Wait::kLeave;
  return error() != 0 ? Wait::kGiveUp : Wait::kGoOn;
}

}  // namespace llh
