// kvcm_key_count.h -- how many keys a request has and where they go, for offsets that may hold anything: every operation is
// defined for all values, and no sum wraps. Plain C++, no HIP (constexpr functions are device functions too): kvcm_hash.hip
// includes it, and so do the host sanitizer runs (tests/cpp/sanitize).
//
// Requests whose tokens are not there are counted as well, and a few of them would take a sum beyond 63 bits and back to where
// another request's keys lie, or in front of all of them. So a request counts for kMostKeys at most, which is more than any memory
// holds: where that matters a sum is kMostKeys or more, and nothing fits behind it. The counts of 2^21 requests, a thread's share of
// all there can be, then add up to 2^62 without a look at every sum (saturating each of them cost 0.4 to 1.5 us of a launch that
// makes offsets), and are brought down to kMostKeys before a thousand such shares, or the 8192 requests of a workgroup, come on top.
#pragma once

#include <stdint.h>

namespace kvcm {

constexpr int64_t kUnknown = INT64_MAX;  // the caller did not say how large an array is: its offsets are taken as they are

constexpr int64_t distance(int64_t from, int64_t to) {  // no signed overflow
    return static_cast<int64_t>(static_cast<uint64_t>(to) - static_cast<uint64_t>(from));
}

// whether [at, at + n) is a non-empty part of [0, size)
constexpr bool inside(int64_t at, int64_t n, int64_t size) { return at >= 0 && n > 0 && n <= size - at; }

constexpr int64_t kMostKeys = int64_t{1} << 41;

constexpr int64_t keys_of(int64_t len, int32_t block_size) {
    if (static_cast<uint64_t>(len) >> 32 == 0) {  // 32-bit division: a fifth of the instructions
        return static_cast<uint32_t>(len) / static_cast<uint32_t>(block_size);
    }
    const int64_t count = len > 0 ? len / block_size : 0;
    return count < kMostKeys ? count : kMostKeys;
}

// Keys of one request; `bad` is set when the tokens they are made of are not all there.
constexpr int64_t keys_of_request(int64_t at, int64_t next, int32_t block_size, int64_t n_tokens, bool &bad) {
    const int64_t count = keys_of(distance(at, next), block_size);
    bad |= n_tokens != kUnknown && count > 0 && !inside(at, count * block_size, n_tokens);
    return count;
}

// What a sum that has gone on adding says: itself, or kMostKeys.
constexpr int64_t at_most_all_keys(int64_t sum) { return sum < kMostKeys ? sum : kMostKeys; }

// The room to ask keys_fit for, of a buffer of `keys` keys: nothing fits behind kMostKeys, however large the caller says it is.
constexpr int64_t room_for_keys(int64_t keys) { return keys < kMostKeys ? keys : kMostKeys - 1; }

// Whether `count` keys behind `before` others lie within that room.
constexpr bool keys_fit(int64_t before, int64_t count, int64_t room) { return before + count <= room; }

}  // namespace kvcm
