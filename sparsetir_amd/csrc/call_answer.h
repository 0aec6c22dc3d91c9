// What the kernels of a call write into host memory, one 8-byte store per bucket that needs no order with another:
// the ELL rows of the bucket below the number of the call.  The host watches for its number.
#pragma once
#include <cstdint>

namespace stir {

constexpr int kCallShift = 40;  // rows of a bucket are fewer
constexpr uint32_t kCallNumbers = 1u << (64 - kCallShift);

// The number of the next call: never 0, which is what an answer that was not written yet reads as.
inline uint32_t next_call(uint32_t number) {
  number = (number + 1) % kCallNumbers;
  return number ? number : 1;
}

// Before the launch: an answer of this number that is left from kCallNumbers calls ago must not pass for this call's.
inline void forget_answers(uint64_t* answers, int count) {
  for (int b = 0; b < count; ++b) __atomic_store_n(answers + b, uint64_t(0), __ATOMIC_RELAXED);
}

inline bool answered(const uint64_t* answer, uint32_t number) {
  return (__atomic_load_n(answer, __ATOMIC_ACQUIRE) >> kCallShift) == number;
}

inline int64_t answered_rows(uint64_t answer) { return (int64_t)(answer & ((uint64_t(1) << kCallShift) - 1)); }

}  // namespace stir
