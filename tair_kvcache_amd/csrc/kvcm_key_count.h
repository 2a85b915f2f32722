// kvcm_key_count.h -- how many keys a request has and where they go, for offsets that may hold anything: every operation is
// defined for all values, and no sum wraps. Plain C++, no HIP (constexpr functions are device functions too): kvcm_hash.hip
// includes it, and so do the host sanitizer runs (tests/cpp/sanitize).
#pragma once

#include <stdint.h>

namespace kvcm {

constexpr int64_t kUnknown = INT64_MAX;  // the caller did not say how large an array is: its offsets are taken as they are

constexpr int64_t distance(int64_t from, int64_t to) {  // no signed overflow
    return static_cast<int64_t>(static_cast<uint64_t>(to) - static_cast<uint64_t>(from));
}

// whether [at, at + n) is a non-empty part of [0, size)
constexpr bool inside(int64_t at, int64_t n, int64_t size) { return at >= 0 && n > 0 && n <= size - at; }

constexpr int64_t keys_of(int64_t len, int32_t block_size) {
    if (static_cast<uint64_t>(len) >> 32 == 0) {  // 32-bit division: a fifth of the instructions
        return static_cast<uint32_t>(len) / static_cast<uint32_t>(block_size);
    }
    return len > 0 ? len / block_size : 0;
}

// Keys of one request; `bad` is set when the tokens they are made of are not all there.
constexpr int64_t keys_of_request(int64_t at, int64_t next, int32_t block_size, int64_t n_tokens, bool &bad) {
    const int64_t count = keys_of(distance(at, next), block_size);
    bad |= n_tokens != kUnknown && count > 0 && !inside(at, count * block_size, n_tokens);
    return count;
}

// Sums of counts end at kMostKeys, where they stay: requests whose tokens are not there are counted as well, and two of them
// would take a sum beyond 63 bits and back to where another request's keys lie, or in front of all of them. Sound requests
// never get there. The result does not depend on the order in which counts (0 or more) are added up.
constexpr int64_t kMostKeys = int64_t{1} << 62;
constexpr int64_t add_keys(int64_t a, int64_t b) {
    const uint64_t sum = static_cast<uint64_t>(a) + static_cast<uint64_t>(b);
    return sum < static_cast<uint64_t>(kMostKeys) ? static_cast<int64_t>(sum) : kMostKeys;
}

// Whether `count` keys behind `before` others (a sum) lie within the first `room`.
constexpr bool keys_fit(int64_t before, int64_t count, int64_t room) {
    const int64_t end = add_keys(before, count);
    return end < kMostKeys && end <= room;
}

}  // namespace kvcm
