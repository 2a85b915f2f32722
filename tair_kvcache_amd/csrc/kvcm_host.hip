// kvcm_host.hip -- the entry points of libkvcm_hip.so that are host code and nothing else: version, error text, the wait for
// a value that a kernel writes into host memory, and the per-block hash over iov CRCs. Kept apart from the kernels so that a plain host compiler can build this file (and
// kvcm_file.hip, kvcm_host_idx.h) for the sanitizer runs of tests/cpp/sanitize.
#include "kvcm_internal.h"

#include <sched.h>
#include <sys/prctl.h>
#include <time.h>

namespace {

// The kernel may round a thread's sleep up by its timer slack, 50 us unless somebody has changed it: more than the naps below
// are meant to last. Set to the least while it exists.
class ShortTimerSlack {
   public:
    ShortTimerSlack() : before_(prctl(PR_GET_TIMERSLACK, 0, 0, 0, 0)) { prctl(PR_SET_TIMERSLACK, 1, 0, 0, 0); }
    ~ShortTimerSlack() {
        if (before_ > 0) {
            prctl(PR_SET_TIMERSLACK, static_cast<unsigned long>(before_), 0, 0, 0);
        }
    }
    ShortTimerSlack(const ShortTimerSlack &) = delete;
    ShortTimerSlack &operator=(const ShortTimerSlack &) = delete;

   private:
    const int before_;
};

}  // namespace

extern "C" {

int32_t kvcm_hip_version(void) { return 200; }  // 0.2.0: host-index gather/scatter added, test hook gone

const char *kvcm_hip_error_string(int32_t code) {
    switch (code) {
        case KVCM_OK:
            return "ok";
        case KVCM_ERR_INVALID_ARG:
            return "invalid argument";
        case KVCM_ERR_ALIGNMENT:
            return "misaligned address or stride";
        case KVCM_ERR_TOO_LARGE:
            return "size exceeds the launch geometry";
        case KVCM_ERR_IO:
            return "file input/output error";
        case KVCM_ERR_OUT_OF_RANGE:
            return "index out of range";
        default:
            return code > 0 ? hipGetErrorString(static_cast<hipError_t>(code)) : "unknown kvcm error";
    }
}

// The value arrives a few microseconds after the kernel that writes it has started, so the thread looks for it without
// sleeping at first (sleeping and being woken costs more than the wait), gives its core away between looks after a
// while, and only then -- there is other work in front -- takes naps and asks the stream whether anything will still come.
// Behind 1.4 and 6.7 ms of other work a ragged hash_tokens returns 11-18 us after that work has ended (35-49 us with the
// default timer slack; 20 us where the number was copied back and the stream synchronised).
int32_t kvcm_wait_value(const int64_t *h_value, kvcm_stream_t stream) {
    if (!h_value) {
        return KVCM_ERR_INVALID_ARG;
    }
    const auto arrived = [h_value] { return __atomic_load_n(h_value, __ATOMIC_ACQUIRE) != KVCM_PENDING; };
    for (int i = 0; i < 4096; ++i) {
        if (arrived()) {
            return KVCM_OK;
        }
        if (i == 0 && kvcm::is_capturing(static_cast<hipStream_t>(stream))) {  // nothing runs before the graph does
            return static_cast<int32_t>(hipErrorStreamCaptureUnsupported);
        }
        if (i >= 1024) {
            sched_yield();
        } else {
            __builtin_ia32_pause();
        }
    }
    const ShortTimerSlack slack;
    for (;;) {
        const hipError_t e = hipStreamQuery(static_cast<hipStream_t>(stream));
        if (arrived()) {
            return KVCM_OK;
        }
        if (e != hipErrorNotReady) {
            return e == hipSuccess ? static_cast<int32_t>(hipErrorUnknown) : static_cast<int32_t>(e);
        }
        const struct timespec nap = {0, 20000};
        nanosleep(&nap, nullptr);
    }
}

int32_t kvcm_blocks_hash_from_crcs(const uint32_t *crcs, int64_t n_crcs, int32_t iovs_per_block, int64_t *out_hashes) {
    if (iovs_per_block <= 0 || n_crcs < 0 || (n_crcs > 0 && (!crcs || !out_hashes))) {
        return KVCM_ERR_INVALID_ARG;
    }
    int64_t nb = 0;
    for (int64_t off = 0; off + iovs_per_block <= n_crcs; off += iovs_per_block) {
        uint64_t h = 0;
        for (int32_t i = 0; i < iovs_per_block; ++i) {
            h = kvcm::hash_step_preadded(h, static_cast<uint64_t>(crcs[off + i]) + kvcm::kGolden);
        }
        out_hashes[nb++] = static_cast<int64_t>(h);
    }
    return KVCM_OK;
}

}  // extern "C"
