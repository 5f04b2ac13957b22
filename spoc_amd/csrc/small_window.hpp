// The host's side of a small download (get_small in transfer.cpp): a window of pinned memory into which a kernel puts every
// 32-bit word together with the number of its call, in one store of 8 bytes.  No HIP here.
#pragma once
#include <chrono>
#include <cstddef>
#include <cstdint>
#include <cstring>

#include "transfer.hpp"

namespace sarek_hip {

constexpr size_t kWindowWords = kSmallBytes / 4;

// The number of the next call, never 0, which an empty window holds.  When the numbers start again the window is emptied: a word
// that no call has written since its number was used last would be taken for the data of the call that bears it now.
inline uint32_t next_number(uint64_t *window, uint32_t &count) {
  if (++count == 0) {
    std::memset(window, 0, kWindowWords * sizeof(uint64_t));
    count = 1;
  }
  return count;
}

constexpr int kNotDelivered = -1;

// `bytes` (at most kSmallBytes) of call `number` into dst, when all of its words are there.  They are looked for until `look` has
// passed, then once more after wait(), which returns 0 when the kernel has ended.  0; what wait() returned; or kNotDelivered
// where the kernel has ended and a word is missing.  dst is written where 0 is returned and nowhere else.
template <class Wait>
int gather_words(void *dst, const uint64_t *window, size_t bytes, uint32_t number, std::chrono::microseconds look, Wait wait) {
  uint32_t data[kWindowWords];
  const auto until = std::chrono::steady_clock::now() + look;
  bool waited = false;
  for (size_t i = 0; i < (bytes + 3) / 4; ++i) {
    uint64_t word;
    while ((word = __atomic_load_n(window + i, __ATOMIC_RELAXED)) >> 32 != number) {
      if (waited) return kNotDelivered;
      for (int k = 0; k < 64 && __atomic_load_n(window + i, __ATOMIC_RELAXED) >> 32 != number; ++k) __builtin_ia32_pause();
      if (std::chrono::steady_clock::now() > until) {
        if (const int rc = wait(); rc != 0) return rc;
        waited = true;
      }
    }
    data[i] = static_cast<uint32_t>(word);
  }
  std::memcpy(dst, data, bytes);
  return 0;
}

}  // namespace sarek_hip
