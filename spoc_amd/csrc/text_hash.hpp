// Hash of a kernel text, for the tables that are looked up by text at every launch.
#pragma once
#include <cstdint>
#include <cstring>
#include <string>
#include <string_view>

namespace sarek_hip {

// Four lanes of eight bytes a step: a 3 KB text takes 0.1 us (one lane, whose multiplications wait for each other: 0.45;
// the standard library's: 0.4), a launch 2.8.
inline uint64_t hash_text(const char *p, size_t n) {
  constexpr uint64_t kMul = 0xFF51AFD7ED558CCDull;
  uint64_t h[4] = {0x9E3779B97F4A7C15ull ^ n, 0xC2B2AE3D27D4EB4Full, 0x165667B19E3779F9ull, 0x27D4EB2F165667C5ull};
  uint64_t w[4];
  while (n >= 32) {
    std::memcpy(w, p, 32);
    for (int i = 0; i < 4; ++i) {
      h[i] = (h[i] ^ w[i]) * kMul;
      h[i] ^= h[i] >> 32;
    }
    p += 32;
    n -= 32;
  }
  std::memset(w, 0, 32);
  std::memcpy(w, p, n);
  uint64_t r = 0;
  for (int i = 0; i < 4; ++i) {
    r = (r ^ h[i] ^ w[i]) * 0xC4CEB9FE1A85EC53ull;
    r ^= r >> 29;
  }
  return r;
}

struct TextHash {
  using is_transparent = void;
  size_t operator()(std::string_view v) const { return hash_text(v.data(), v.size()); }
};

}  // namespace sarek_hip
