// The host's side of a small download, with a window in ordinary memory and threads in the kernel's place.
#include <cstdio>
#include <thread>
#include <vector>

#include "small_window.hpp"

using namespace sarek_hip;
using std::chrono::microseconds;
using std::chrono::milliseconds;

namespace {
uint64_t window[kWindowWords];
int failures = 0;

void expect(bool ok, const char *what) {
  if (!ok) std::printf("failed: %s\n", what), ++failures;
}

void put(uint32_t number, size_t first, size_t last) {
  for (size_t i = first; i < last; ++i)
    __atomic_store_n(window + i, static_cast<uint64_t>(number) << 32 | (0x01010101u * (i % 200 + 1) ^ number), __ATOMIC_RELAXED);
}

bool holds(const std::vector<unsigned char> &dst, uint32_t number, size_t bytes) {
  for (size_t i = 0; i < dst.size(); ++i) {
    const uint32_t word = 0x01010101u * (i / 4 % 200 + 1) ^ number;
    if (dst[i] != (i < bytes ? static_cast<unsigned char>(word >> (i % 4 * 8)) : 0xEE)) return false;
  }
  return true;
}

bool untouched(const std::vector<unsigned char> &dst) {
  for (unsigned char c : dst)
    if (c != 0xEE) return false;
  return true;
}
}  // namespace

int main() {
  uint32_t count = 0;
  int waits = 0;
  auto ended = [&] { return ++waits, 0; };
  for (size_t bytes : {size_t{1}, size_t{3}, size_t{4}, size_t{5}, size_t{1024}, kSmallBytes - 1, kSmallBytes}) {
    const size_t words = (bytes + 3) / 4;
    std::vector<unsigned char> dst(kSmallBytes + 8, 0xEE);
    // all there; word by word while the host looks; by the time the wait ends
    uint32_t number = next_number(window, count);
    put(number, 0, words);
    expect(gather_words(dst.data(), window, bytes, number, milliseconds(2), ended) == 0 && waits == 0 && holds(dst, number, bytes), "there");
    number = next_number(window, count);
    std::thread late([&] {
      for (size_t i = words; i-- > 0;) put(number, i, i + 1);
    });
    const int rc = gather_words(dst.data(), window, bytes, number, std::chrono::seconds(20), ended);
    late.join();
    expect(rc == 0 && waits == 0 && holds(dst, number, bytes), "while it looks");
    number = next_number(window, count);
    expect(gather_words(dst.data(), window, bytes, number, microseconds(50), [&] { return put(number, 0, words), ++waits, 0; }) == 0 &&
               waits == 1 && holds(dst, number, bytes), "after the wait");
    // the last word never comes: the call ends, and dst is as it was; the same where the wait fails
    std::vector<unsigned char> kept(kSmallBytes + 8, 0xEE);
    number = next_number(window, count);
    put(number, 0, words - 1);
    expect(gather_words(kept.data(), window, bytes, number, microseconds(50), ended) == kNotDelivered && waits == 2 && untouched(kept), "never");
    number = next_number(window, count);
    put(number, 0, words - 1);
    expect(gather_words(kept.data(), window, bytes, number, microseconds(50), [] { return 7; }) == 7 && untouched(kept), "wait failed");
    waits = 0;
  }
  // the numbers start again: what an old call with the same number left is not this call's
  put(1, 0, kWindowWords);
  count = 0xFFFFFFFFu;
  const uint32_t number = next_number(window, count);
  std::vector<unsigned char> kept(16, 0xEE);
  expect(number == 1 && gather_words(kept.data(), window, 16, number, microseconds(50), ended) == kNotDelivered && untouched(kept), "numbers start again");
  if (failures == 0) std::printf("small window ok\n");
  return failures;
}
