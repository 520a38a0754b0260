// Which 16-byte block (32 inner indices) of a nibble column k_onehot_digits
// loads. Host code too: the bounds are tested on the CPU.
#pragma once

#include <cstdint>

#if defined(__HIPCC__)
#define ACKVQ_HOST_DEVICE __host__ __device__
#else
#define ACKVQ_HOST_DEVICE
#endif

namespace ackvq {

// Lane half h's block of step s (64 inner indices, a block a half) in a column
// of `blocks` blocks: block 2 s + h, or the last one past the end, whose value
// goes unused (an odd column's last step has no second half, and the loop loads
// one step ahead).
ACKVQ_HOST_DEVICE inline constexpr uint32_t digit_block(uint32_t s, uint32_t h, uint32_t blocks) {
  return 2 * s + h < blocks ? 2 * s + h : blocks - 1;
}

}  // namespace ackvq
