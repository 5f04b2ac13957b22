// Transfers of small vectors, beside the general ones of the C ABI (transfer.cpp).
#pragma once
#include <cstddef>

namespace sarek_hip {
constexpr size_t kSmallBytes = 3072;
// Both work on the default stream of the current device, which `dst` (put) and `src` (get) must lie on, and return
// SAREK_HIP_E_UNSUPPORTED, nothing done, where the general copy has to be taken.
// put_small: `src` may change as soon as it returns; `dst` holds the data for whatever the default stream is given next.
int put_small(void *dst, const void *src, size_t bytes);
// get_small: what the default stream was given before it has run, and the data is in `dst`, when it returns.
int get_small(void *dst, const void *src, size_t bytes, int dev);
}  // namespace sarek_hip
