// Numbers by which the count words of a launch (shares, gang ranges) are told from whatever else their workspace holds.
//
// A count word is launch number << 16 | parts done, and a word that does not carry the launch's number counts as zero,
// so a workspace needs no clearing.  That is only as good as the numbers are unlike data: counted from 1, launch n took
// any token id or offset between n << 16 and (n + 1) << 16 for its own count, and merged partials that were not there.
// A number therefore starts with eleven ones behind a zero, which makes the word a NaN to whoever wrote it as doubles, as
// pairs of floats or as bf16 or half, and more than 2^62 as a 64-bit integer; the other 36 bits start anywhere, differently in every
// process, and move by a large odd step, so they pass through all 2^36 values before one comes again.
#pragma once
#include <stdint.h>
#include <sys/random.h>
#include <time.h>

#include <atomic>

namespace msgl {

constexpr int kLaunchBits = 36;
constexpr uint64_t kLaunchMark = 0x7ffull << kLaunchBits;
constexpr uint64_t kLaunchStep = 0x9e3779b97f4a7c15ull;  // odd; 2^64 / golden ratio

inline uint64_t launch_seed() {
  uint64_t seed = 0;
  if (getrandom(&seed, sizeof seed, GRND_NONBLOCK) == (ssize_t)sizeof seed) return seed;
  timespec t{};
  clock_gettime(CLOCK_MONOTONIC, &t);  // an address (of this call's stack) and the clock instead
  return ((uint64_t)t.tv_sec * 1000000000ull + (uint64_t)t.tv_nsec) * kLaunchStep ^ reinterpret_cast<uintptr_t>(&t);
}

inline uint64_t next_launch_number() {
  static std::atomic<uint64_t> next{launch_seed()};
  return kLaunchMark | (next.fetch_add(kLaunchStep, std::memory_order_relaxed) & ((1ull << kLaunchBits) - 1));
}

}  // namespace msgl
