// Host-side passes over the arrays of a run -- copies into and out of page-locked memory, fp32 <-> bf16 -- shared out
// among a few threads where they are long.
#pragma once

#include <cstddef>
#include <cstdint>

namespace pmlc::rt {

void hostCopy(void* dst, const void* src, size_t bytes);
// fp32 -> bf16 storage, round to nearest even; any NaN becomes 0x7fc0
void hostToBf16(uint16_t* dst, const float* src, size_t n);
void hostFromBf16(float* dst, const uint16_t* src, size_t n);

}  // namespace pmlc::rt
