// Ordering of (logit, column) pairs shared by the argmax kernels.
#pragma once

#include "common.h"

namespace oxr {

// Order-preserving key of a bf16 logit (as fp32 bits) and its column: larger
// value wins, then lower column.  NaN sorts above everything (torch argmax
// returns the first NaN); -0 and +0 compare equal.
__device__ __forceinline__ uint64_t argmax_key(uint32_t fbits, uint32_t col) {
  uint32_t key;
  if ((fbits & 0x7fffffffu) > 0x7f800000u) key = 0xffffffffu;
  else {
    if ((fbits & 0x7fffffffu) == 0u) fbits = 0u;
    key = (fbits & 0x80000000u) ? ~fbits : (fbits | 0x80000000u);
  }
  return ((uint64_t)key << 32) | (uint32_t)(~col);
}

}  // namespace oxr
