// kvcm_internal.h -- shared by the translation units of libkvcm_hip.so (not installed).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "kvcm_hip.h"

namespace kvcm {

constexpr uint64_t kGolden = 0x9e3779b97f4a7c15ULL;

inline int32_t launch_status() {
    hipError_t e = hipGetLastError();
    return e == hipSuccess ? KVCM_OK : static_cast<int32_t>(e);
}

// Whether work on `s` is being recorded into a graph. The null stream never is, and must not be asked: the question alone is
// an error while another stream is being captured.
inline bool is_capturing(hipStream_t s) {
    hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
    return s && (hipStreamIsCapturing(s, &status) != hipSuccess || status != hipStreamCaptureStatusNone);
}

// n / d for n < 2^31 as a multiply and a shift: mul = ceil(2^(31+L) / d), L = ceil(log2 d).
struct FastDiv {
    uint32_t mul;
    uint32_t shift;
};

inline FastDiv make_fastdiv(uint32_t d) {
    uint32_t L = 0;
    while ((uint64_t{1} << L) < d) {
        ++L;
    }
    const uint64_t pow = uint64_t{1} << (31 + L);
    return FastDiv{static_cast<uint32_t>((pow + d - 1) / d), 31 + L};
}

__device__ inline uint32_t fast_div(uint32_t n, FastDiv f) {
    return static_cast<uint32_t>((static_cast<uint64_t>(n) * f.mul) >> f.shift);
}

// One hashInt64Func step (kv_cache_manager/manager/hash_util.h:8-12) with the token term pre-added:
// a = value + 0x9e3779b97f4a7c15. Unsigned arithmetic wraps mod 2^64; the right shift is arithmetic.
__host__ __device__ inline uint64_t hash_step_preadded(uint64_t h, uint64_t a) {
    return h ^ (a + (h << 12) + static_cast<uint64_t>(static_cast<int64_t>(h) >> 32));
}

}  // namespace kvcm
