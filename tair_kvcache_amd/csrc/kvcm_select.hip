// kvcm_select.hip -- which blocks of a batch have to be moved: first occurrences of block keys inside a
// batch of requests, and the ascending index list of the blocks a mask leaves to save.
//
// The reference decides this on the host: the manager answers StartWriteCache with a block mask and the connector
// turns it into a Python list (kv_cache_manager/py_connector/vllm/v1_connector.py:835-850); requests of one batch that
// share a prefix are not compared with each other at all. Here both steps stay on the device, next to the keys
// (kvcm_hip_hash_tokens) and to the index kernels that consume the list.
//
// Small integer kernels, nowhere near a bandwidth bound: n is the number of block keys of a batch (thousands).
#include <atomic>
#include <climits>
#include <mutex>

#include "kvcm_internal.h"

namespace kvcm {
namespace {

// Table of kvcm_hip_first_occurrence_static: room for 2^20 keys (capacity 2 n, one int32 per slot = 8 MiB).
// Every device that the library runs on holds its own copy, at its own address, until the process ends.
constexpr int64_t kStaticMaxKeys = int64_t{1} << 20;
constexpr int64_t kStaticCapacity = 2 * kStaticMaxKeys;
static __device__ __align__(256) int32_t scratch[kStaticCapacity];

// Device address of `scratch` per device: in host code the array's name is only a handle for the runtime's symbol
// calls, never an address a kernel may be given.
constexpr int kMaxDevices = 64;
std::atomic<int32_t *> g_scratch_ptr[kMaxDevices];
std::mutex g_scratch_mutex;

// The current device's copy of `scratch`; looked up once per device. Returns a kvcm / HIP code.
int32_t static_scratch(int32_t **out) {
    int dev = -1;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) {
        return static_cast<int32_t>(e);
    }
    if (dev < 0 || dev >= kMaxDevices) {
        return KVCM_ERR_TOO_LARGE;
    }
    int32_t *p = g_scratch_ptr[dev].load(std::memory_order_acquire);
    if (!p) {
        std::lock_guard<std::mutex> guard(g_scratch_mutex);
        p = g_scratch_ptr[dev].load(std::memory_order_relaxed);
        if (!p) {
            void *addr = nullptr;
            e = hipGetSymbolAddress(&addr, HIP_SYMBOL(scratch));
            if (e != hipSuccess) {
                return static_cast<int32_t>(e);
            }
            if (!addr) {
                return static_cast<int32_t>(hipErrorInvalidSymbol);
            }
            p = static_cast<int32_t *>(addr);
            g_scratch_ptr[dev].store(p, std::memory_order_release);
        }
    }
    *out = p;
    return KVCM_OK;
}

constexpr int kSelThreads = 1024;  // 16 waves: one workgroup scans 1024 flags or counts per pass
constexpr int kSelWaves = kSelThreads / 64;

__global__ __launch_bounds__(256) void fill_i32_kernel(int32_t *__restrict__ p, int64_t n, int32_t v) {
    int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
    if (i < n) {
        p[i] = v;
    }
}

__device__ inline int32_t table_load(const int32_t *p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Keys beyond which a probe looks at its slot before it tries to claim it. Claim at once / look first, us:
//                            2^16         2^18         5 * 2^16     3 * 2^17     2^19         2^20
// first, all different   26.4 / 25.1  44.5 / 44.0  42.0 / 50.3  46.9 / 47.2  71.9 / 65.6  117.0 / 105.2
// first, each 8 times    11.8 / 13.7  21.2 / 23.7  26.3 / 29.8  28.9 / 32.1  35.3 / 31.7   62.4 / 42.2
// list, all different    18.4 / 18.7  36.0 / 45.1  43.8 / 54.5  52.6 / 49.4  64.1 / 58.8  100.2 / 98.3
// list, each 8 times     14.1 / 15.1  24.5 / 26.7  28.3 / 32.0  31.9 / 35.5  38.8 / 34.8   70.5 / 49.3
// The columns of 2^16 and 2^18 keys are at two slots per key for first occurrences, four for the list. In a table that full
// (less than 2.5 slots per key) claims that fail cost more than looks from 2^17 keys on where keys are different: 2^18 of them
// 42.5 to 49.8 / 41.6 to 46, by their values.
constexpr int64_t kLookFirstBeyond = 3 << 17;
constexpr int64_t kLookFirstBeyondFull = 1 << 17;
bool look_first(int64_t n, int64_t slots) { return n > (2 * slots < 5 * n ? kLookFirstBeyondFull : kLookFirstBeyond); }

// Open addressing, linear probing, one int32 per slot: -1 = empty, otherwise an index whose key owns the slot.
// A slot claimed for key K is only ever lowered (atomicMin) by indices that hold the same K, so whatever index a
// probe reads from a slot names that slot's key; after the launch the slot holds the smallest such index.
__global__ __launch_bounds__(256) void insert_kernel(const int64_t *__restrict__ keys, int32_t n,
                                                     int32_t *table, uint32_t mask, int shift,
                                                     int32_t *__restrict__ slot_of, bool look_first) {
    int32_t i = blockIdx.x * 256 + threadIdx.x;
    if (i >= n) {
        return;
    }
    const int64_t k = keys[i];
    uint32_t s = static_cast<uint32_t>((static_cast<uint64_t>(k) * kGolden) >> shift) & mask;
    for (;;) {
        // Few keys: claimed or looked at in one trip to memory. Many: the atomics are the bound, and a look saves those that
        // find the slot taken.
        int32_t o = look_first ? table_load(table + s) : -1;
        if (o < 0) {
            o = atomicCAS(table + s, -1, i);
            if (o < 0) {
                break;  // claimed
            }
        }
        if (keys[o] == k) {
            if (o > i) {  // what a slot holds only ever falls: a smaller index that is there already stays or gives way to a
                atomicMin(table + s, i);  // yet smaller one, and needs no atomic from the 30 requests that share a prefix
            }
            break;
        }
        s = (s + 1) & mask;
    }
    slot_of[i] = static_cast<int32_t>(s);
}

__global__ __launch_bounds__(256) void resolve_kernel(int32_t *__restrict__ first_idx, const int32_t *__restrict__ table,
                                                      int32_t n, uint8_t *__restrict__ is_repeat) {
    int32_t i = blockIdx.x * 256 + threadIdx.x;
    if (i >= n) {
        return;
    }
    int32_t f = table[first_idx[i]];
    first_idx[i] = f;
    if (is_repeat) {
        is_repeat[i] = f != i;
    }
}

__device__ inline bool wanted(const uint8_t *__restrict__ a, const uint8_t *__restrict__ b, int32_t i) {
    return a[i] == 0 && (b == nullptr || b[i] == 0);
}

// Rank of this thread among the workgroup's set flags, and the workgroup's total. All threads call.
__device__ inline int32_t flag_rank(bool flag, int32_t *wave_totals, int32_t *total) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const uint64_t ballot = __ballot(flag);
    if (lane == 0) {
        wave_totals[wave] = __popcll(ballot);
    }
    __syncthreads();
    int32_t before = 0, all = 0;
    for (int w = 0; w < kSelWaves; w++) {
        int32_t c = wave_totals[w];
        before += w < wave ? c : 0;
        all += c;
    }
    *total = all;
    return before + __popcll(ballot & ((1ull << lane) - 1));
}

__global__ __launch_bounds__(kSelThreads) void count_kernel(const uint8_t *__restrict__ a, const uint8_t *__restrict__ b,
                                                            int32_t n, int32_t *__restrict__ group_count) {
    __shared__ int32_t wave_totals[kSelWaves];
    int32_t i = blockIdx.x * kSelThreads + threadIdx.x, total;
    flag_rank(i < n && wanted(a, b, i), wave_totals, &total);
    if (threadIdx.x == 0) {
        group_count[blockIdx.x] = total;
    }
}

// One workgroup: counts[0..G) -> exclusive prefix sums in place, grand total to *d_total.
__global__ __launch_bounds__(kSelThreads) void scan_kernel(int32_t *__restrict__ counts, int32_t G,
                                                           int32_t *__restrict__ d_total) {
    __shared__ int32_t wave_totals[kSelWaves];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    int32_t carry = 0;
    for (int32_t base = 0; base < G; base += kSelThreads) {
        const int32_t i = base + threadIdx.x;
        const int32_t v = i < G ? counts[i] : 0;
        int32_t incl = v;
        for (int d = 1; d < 64; d <<= 1) {
            int32_t up = __shfl_up(incl, d, 64);
            incl += lane >= d ? up : 0;
        }
        if (lane == 63) {
            wave_totals[wave] = incl;
        }
        __syncthreads();
        int32_t before = 0, all = 0;
        for (int w = 0; w < kSelWaves; w++) {
            int32_t c = wave_totals[w];
            before += w < wave ? c : 0;
            all += c;
        }
        if (i < G) {
            counts[i] = carry + before + incl - v;
        }
        carry += all;
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        *d_total = carry;
    }
}

__global__ __launch_bounds__(kSelThreads) void write_kernel(const uint8_t *__restrict__ a, const uint8_t *__restrict__ b,
                                                            int32_t n, const int32_t *__restrict__ group_offset,
                                                            int32_t *__restrict__ indices) {
    __shared__ int32_t wave_totals[kSelWaves];
    int32_t i = blockIdx.x * kSelThreads + threadIdx.x, total;
    const bool flag = i < n && wanted(a, b, i);
    const int32_t rank = flag_rank(flag, wave_totals, &total);
    if (flag) {
        indices[group_offset[blockIdx.x] + rank] = i;
    }
}

// The list of a batch of more keys than part_kernel takes, in four launches (fill, insert, choose, list) where first occurrences and mask compaction in a row
// take six. Bound by latency: every launch is a chain of two or three trips to memory, and what counts is how many follow
// each other. 256 keys per workgroup, so that 32 768 keys make 128 workgroups.
constexpr int kListThreads = 256;
constexpr int kListWaves = kListThreads / 64;
// Keys up to which a workgroup adds up the counts of all workgroups in front of it itself (16 per thread at most) instead of
// waiting for a scan of its own.
constexpr int64_t kListMaxKeys = int64_t{1} << 20;

// One bit per key: first occurrence and not saved yet. The bits of a wave go out as one word, a workgroup's total beside them.
__global__ __launch_bounds__(kListThreads) void choose_kernel(const int32_t *__restrict__ slot_of, const int32_t *__restrict__ table,
                                                              const uint8_t *__restrict__ saved, int32_t n,
                                                              uint64_t *__restrict__ words, int32_t *__restrict__ group_count) {
    __shared__ int32_t wave_totals[kListWaves];
    const int32_t i = blockIdx.x * kListThreads + threadIdx.x;
    bool flag = false;
    if (i < n) {
        const int32_t slot = slot_of[i];
        flag = !(saved && saved[i]) && table[slot] == i;
    }
    const uint64_t ballot = __ballot(flag);
    const int wave = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0) {
        words[blockIdx.x * kListWaves + wave] = ballot;
        wave_totals[wave] = __popcll(ballot);
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        int32_t all = 0;
        for (int w = 0; w < kListWaves; ++w) {
            all += wave_totals[w];
        }
        group_count[blockIdx.x] = all;
    }
}

__global__ __launch_bounds__(kListThreads) void list_kernel(const uint64_t *__restrict__ words, const int32_t *__restrict__ group_count,
                                                            int32_t *__restrict__ indices, int32_t *__restrict__ d_count) {
    __shared__ int32_t wave_sums[kListWaves];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int32_t group = blockIdx.x;
    uint64_t word[kListWaves];
#pragma unroll
    for (int w = 0; w < kListWaves; ++w) {
        word[w] = words[group * kListWaves + w];
    }
    int32_t sum = 0;
#pragma unroll 4
    for (int32_t g = threadIdx.x; g < group; g += kListThreads) {
        sum += group_count[g];
    }
    for (int d = 1; d < 64; d <<= 1) {
        sum += __shfl_xor(sum, d, 64);
    }
    if (lane == 0) {
        wave_sums[wave] = sum;
    }
    __syncthreads();
    int32_t before = 0, own = 0;
    uint64_t mine = 0;
#pragma unroll
    for (int w = 0; w < kListWaves; ++w) {
        before += wave_sums[w] + (w < wave ? __popcll(word[w]) : 0);
        own += w >= wave ? __popcll(word[w]) : 0;
        mine = w == wave ? word[w] : mine;
    }
    if (mine >> lane & 1) {
        indices[before + __popcll(mine & ((1ull << lane) - 1))] = group * kListThreads + static_cast<int32_t>(threadIdx.x);
    }
    if (group == static_cast<int32_t>(gridDim.x) - 1 && threadIdx.x == 0) {
        *d_count = before + own;  // thread 0: nothing of its own group lies before it
    }
}

// The list of up to kPartMaxKeys keys in two launches. Every workgroup reads ALL keys and takes those whose hash value falls into
// its part, so a part's table fits the LDS: no table in memory to clear, no chain of probes through memory, and nobody waits for
// anybody. Bound: every compute unit reads every key (64 bytes a clock from its L2) and looks at it, about 70 clocks for 64 keys of
// a wave; the keys that are taken wait in LDS until 64 of them can be entered at a time, because a branch for the few lanes whose
// key it is costs a wave as much as 64 of them (32 768 keys 12.4 to 15.0, so 9.2 to 9.7 us). Two launches against four, us, all
// different / each 8 times: 1000 keys 11.3 / 12.0 -> 6.7 / 6.6, 16 384 14.2 / 11.7 -> 7.8 / 7.7, 32 768 13.9 / 11.8 -> 9.7 / 9.2,
// 65 536 16.3 / 14.3 -> 13.3 / 12.8; 100 000 keys 20.9 / 17.1 and 17.8 / 17.7, 131 072 23.0 / 18.5 and 21.3 / 21.0, so beyond 65 536
// the table in memory stays.
constexpr int kPartThreads = 1024;
constexpr int64_t kPartMaxKeys = int64_t{1} << 16;
constexpr uint64_t kNoKey = 0x8000000000000000ull;  // an empty slot; a key of this value is kept apart

struct PartShape {
    int log2_parts, log2_slots;
};

// One part per compute unit where there are keys for it, and eight slots per key of an even share.
PartShape part_shape(int64_t n) {
    PartShape p{n > 4096 ? 8 : n > 512 ? 6 : 4, 8};
    while ((int64_t{1} << (p.log2_slots + p.log2_parts)) < 8 * n) {
        ++p.log2_slots;
    }
    return p;
}

// Both halves times odd constants, modulo 2^32; the upper bits choose the part, the next ones the slot. In 64-bit multiply-adds,
// which issue at the full rate (a 32-bit multiplication takes four times as long).
__device__ __forceinline__ uint32_t part_hash(uint64_t k) {
    uint64_t x, carry;
    asm("v_mad_u64_u32 %0, %1, %2, %3, 0" : "=v"(x), "=s"(carry) : "v"(static_cast<uint32_t>(k)), "s"(0x9e3779b1u));
    asm("v_mad_u64_u32 %0, %1, %2, %3, %4" : "=v"(x), "=s"(carry) : "v"(static_cast<uint32_t>(k >> 32)), "s"(0x85ebca77u), "v"(x));
    return static_cast<uint32_t>(x);
}

// All bits of a key into all bits of the result (the finalizer of MurmurHash3): whatever pattern brings keys into one part, this
// one spreads them.
__device__ __forceinline__ uint64_t mix_key(uint64_t k) {
    k = (k ^ (k >> 33)) * 0xff51afd7ed558ccdull;
    k = (k ^ (k >> 33)) * 0xc4ceb9fe1a85ec53ull;
    return k ^ (k >> 33);
}

// flags[i] = keys[i] is a first occurrence and not saved yet. Exactly one write per key: whoever learns that an index is not the
// smallest of its key clears it -- its own, or the one it has just replaced -- and what is left in the table at the end is set.
__global__ __launch_bounds__(kPartThreads) void part_kernel(const uint64_t *__restrict__ keys, int32_t n, int log2_parts, int log2_slots,
                                                            const uint8_t *__restrict__ saved, uint8_t *__restrict__ flags) {
    extern __shared__ __attribute__((aligned(16))) uint64_t s_key[];
    const uint32_t slots = 1u << log2_slots, mask = slots - 1;
    int32_t *const s_first = reinterpret_cast<int32_t *>(s_key + slots);  // smallest index of the slot's key
    __shared__ int32_t s_first_no_key, s_full, s_hits;
    __shared__ uint64_t s_wait_key[kPartThreads / 64][2 * 64];
    __shared__ int32_t s_wait_idx[kPartThreads / 64][2 * 64];
    const uint32_t lane = threadIdx.x & 63u, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const auto clear = [&] {
        for (uint32_t i = threadIdx.x; i < slots; i += kPartThreads) {
            s_key[i] = kNoKey;
            s_first[i] = INT32_MAX;
        }
    };
    const auto write_out = [&] {
        for (uint32_t s = threadIdx.x; s <= slots; s += kPartThreads) {
            const int32_t f = s < slots ? s_first[s] : s_first_no_key;
            if (f != INT32_MAX) {
                flags[f] = !(saved && saved[f]);
            }
        }
    };
    clear();
    if (threadIdx.x == 0) {
        s_first_no_key = INT32_MAX;
        s_full = s_hits = 0;
    }
    __syncthreads();
    const auto put = [&](int32_t *first, int32_t i) {
        const int32_t was = atomicMin(first, i);
        if (was != INT32_MAX) {
            flags[was < i ? i : was] = 0;
        }
    };
    const auto probe = [&](uint64_t k, int32_t i, uint32_t s) {  // false: all slots hold other keys
        for (uint32_t tries = 0; tries < slots; ++tries) {
            const uint64_t o = atomicCAS(reinterpret_cast<unsigned long long *>(s_key + s), kNoKey, k);
            if (o == kNoKey || o == k) {
                put(s_first + s, i);
                return true;
            }
            s = (s + 1) & mask;
        }
        return false;
    };
    const auto take = [&](uint64_t k, int32_t i) {
        if (k == kNoKey) {
            put(&s_first_no_key, i);
        } else if (__hip_atomic_load(&s_full, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) == 0 &&
                   !probe(k, i, (part_hash(k) << log2_parts) >> (32 - log2_slots))) {
            __hip_atomic_store(&s_full, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        }
    };
    uint64_t *const wait_key = s_wait_key[wave];
    int32_t *const wait_idx = s_wait_idx[wave];
    uint32_t waiting = 0;
    const auto enter = [&](uint32_t count) {  // the last `count` keys that wait
        __builtin_amdgcn_wave_barrier();
        waiting -= count;
        if (lane < count) {
            take(wait_key[waiting + lane], wait_idx[waiting + lane]);
        }
        __builtin_amdgcn_wave_barrier();
    };
    const auto look = [&](uint64_t k, int32_t i, bool there) {
        const bool hit = part_hash(k) >> (32 - log2_parts) == blockIdx.x && there;
        const uint64_t hits = __ballot(hit);
        if (hits) {
            if (hit) {
                const uint32_t at = waiting + __builtin_amdgcn_mbcnt_hi(static_cast<uint32_t>(hits >> 32),
                                                                        __builtin_amdgcn_mbcnt_lo(static_cast<uint32_t>(hits), 0));
                wait_key[at] = k;
                wait_idx[at] = i;
            }
            waiting += __popcll(hits);
            if (waiting >= 64) {
                enter(64);
            }
        }
    };
    typedef uint64_t u64x2 __attribute__((ext_vector_type(2)));
    typedef u64x2 u64x2_a8 __attribute__((aligned(8)));
    constexpr int kAhead = 4;
    constexpr int32_t kStep = 2 * kPartThreads;
    for (int32_t base = 0; base < n; base += kAhead * kStep) {
        u64x2 k[kAhead];
        const int32_t first = base + static_cast<int32_t>(threadIdx.x) * 2;
        if (base + kAhead * kStep <= n) {
#pragma unroll
            for (int a = 0; a < kAhead; ++a) {
                k[a] = *reinterpret_cast<const u64x2_a8 *>(keys + first + a * kStep);
            }
#pragma unroll
            for (int a = 0; a < kAhead; ++a) {
                look(k[a].x, first + a * kStep, true);
                look(k[a].y, first + a * kStep + 1, true);
            }
        } else {
#pragma unroll
            for (int a = 0; a < kAhead; ++a) {
                const int32_t i = first + a * kStep;
                k[a] = u64x2{i < n ? keys[i] : 0, i + 1 < n ? keys[i + 1] : 0};
            }
#pragma unroll
            for (int a = 0; a < kAhead; ++a) {
                if (base + a * kStep < n) {
                    look(k[a].x, first + a * kStep, first + a * kStep < n);
                    look(k[a].y, first + a * kStep + 1, first + a * kStep + 1 < n);
                }
            }
        }
    }
    enter(waiting);
    __syncthreads();
    if (s_full == 0) {
        write_out();
        return;
    }
    // More different keys than slots, all of one part: keys with a pattern that the sum of products maps to one place. Their part is
    // gone through once more, as many times over as bring the number of keys down to half the slots, a share of the mixed keys
    // at a time. What has been cleared so far stays so (a smaller index of that key is known), everything else is decided again.
    // 65 536 keys, each twice, all of one part 2.1 ms, with one slot to start from 4.8; 8192 of the latter 0.47 (looked for one by one,
    // in the keys in front of each, 5.8 and the square of that for more). The look at s_full per key that is entered takes 0.5 %.
    const auto mine = [&](uint64_t k) { return k != kNoKey && part_hash(k) >> (32 - log2_parts) == blockIdx.x; };
    int32_t hits = 0;
    for (int32_t i = threadIdx.x; i < n; i += kPartThreads) {
        hits += mine(keys[i]);
    }
    atomicAdd(&s_hits, hits);
    __syncthreads();
    int log2_shares = 1;
    while ((s_hits >> log2_shares) > static_cast<int32_t>(slots / 2)) {
        ++log2_shares;
    }
    for (uint32_t share = 0; share < 1u << log2_shares; ++share) {
        clear();
        __syncthreads();
        for (int32_t i = threadIdx.x; i < n; i += kPartThreads) {
            const uint64_t k = keys[i], m = mix_key(k);
            if (static_cast<uint32_t>(m >> 32) >> (32 - log2_shares) == share && mine(k) && !probe(k, i, static_cast<uint32_t>(m) & mask)) {
                int32_t j = 0;  // made against this function, too: looked for one by one
                while (j < i && keys[j] != k) {
                    ++j;
                }
                flags[i] = j == i && !(saved && saved[i]);
            }
        }
        __syncthreads();
        write_out();
        __syncthreads();
    }
}

// The ascending list of the set flags. A workgroup takes 1024 of them, four per thread, and counts all flags in front of its own.
constexpr int kPartListThreads = 256;
__global__ __launch_bounds__(kPartListThreads) void part_list_kernel(const uint32_t *__restrict__ flags4, int32_t n,
                                                                     int32_t *__restrict__ indices, int32_t *__restrict__ d_count) {
    __shared__ int32_t s_before[kPartListThreads / 64], s_own[kPartListThreads / 64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int32_t first = (blockIdx.x * kPartListThreads + threadIdx.x) * 4;
    uint32_t mine = first < n ? flags4[first / 4] : 0;
    if (first + 4 > n && first < n) {
        mine &= (1u << 8 * (n - first)) - 1;
    }
    int32_t before = 0;
    typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
    typedef u32x4 u32x4_a8 __attribute__((aligned(8)));
    const u32x4_a8 *const front = reinterpret_cast<const u32x4_a8 *>(flags4);
#pragma unroll 4
    for (int32_t i = threadIdx.x; i < static_cast<int32_t>(blockIdx.x) * kPartListThreads / 4; i += kPartListThreads) {
        const u32x4 f = front[i];
        before += __popc(f.x) + __popc(f.y) + __popc(f.z) + __popc(f.w);
    }
    const int32_t own = __popc(mine);
    int32_t incl = own;
    for (int d = 1; d < 64; d <<= 1) {
        const int32_t up = __shfl_up(incl, d, 64);
        incl += lane >= d ? up : 0;
        before += __shfl_xor(before, d, 64);
    }
    if (lane == 63) {
        s_before[wave] = before;
        s_own[wave] = incl;
    }
    __syncthreads();
    int32_t at = incl - own;
    for (int w = 0; w < kPartListThreads / 64; ++w) {
        at += s_before[w] + (w < wave ? s_own[w] : 0);
    }
#pragma unroll
    for (int b = 0; b < 4; ++b) {
        if (mine >> 8 * b & 1) {
            indices[at++] = first + b;
        }
    }
    if (blockIdx.x == gridDim.x - 1 && threadIdx.x == kPartListThreads - 1) {
        *d_count = at;
    }
}

constexpr int64_t kMaxKeys = int64_t{1} << 30;

int64_t list_groups(int64_t n) { return (n + kListThreads - 1) / kListThreads; }

int64_t table_capacity(int64_t n) {
    int64_t cap = 1024;
    while (cap < 2 * n) {
        cap <<= 1;
    }
    return cap;
}

// Slots of the table of one list. Up to 2^18 keys four to eight per key: every probe is two trips to memory one after the
// other, and the launch lasts as long as its unluckiest key. Beyond, 2.5 to 5 per key: the table no longer lies in the caches,
// and clearing it counts as well (three / six slots per key: 327 680 keys 43.8 / 50, 655 360 70.8 / 71.5 us).
int64_t list_capacity(int64_t n) {
    const int64_t cap = table_capacity(n);
    return n <= int64_t{1} << 18 || 2 * cap < 5 * n ? 2 * cap : cap;
}

// An empty table of `cap` slots (a power of two, >= 2 n) and the keys into it; the fill is a kernel, so the sequence may be
// recorded into a graph.
void launch_insert(const int64_t *d_keys, int32_t n, int32_t *table, int64_t cap, int32_t *slot_of, hipStream_t s) {
    int log2cap = 0;
    while ((int64_t{1} << log2cap) < cap) {
        log2cap++;
    }
    fill_i32_kernel<<<static_cast<unsigned>(cap / 256), 256, 0, s>>>(table, cap, -1);
    insert_kernel<<<(static_cast<unsigned>(n) + 255) / 256, 256, 0, s>>>(d_keys, n, table, static_cast<uint32_t>(cap - 1), 64 - log2cap,
                                                                       slot_of, look_first(n, cap));
}

int32_t launch_first_occurrence(const int64_t *d_keys, int64_t n, int32_t *table, int64_t cap, int32_t *d_first_idx,
                                uint8_t *d_is_repeat, hipStream_t s) {
    const int32_t n32 = static_cast<int32_t>(n);
    launch_insert(d_keys, n32, table, cap, d_first_idx, s);
    resolve_kernel<<<static_cast<unsigned>((n + 255) / 256), 256, 0, s>>>(d_first_idx, table, n32, d_is_repeat);
    return launch_status();
}

}  // namespace
}  // namespace kvcm

extern "C" {

int64_t kvcm_hip_first_occurrence_workspace_bytes(int64_t n) {
    if (n < 0 || n > kvcm::kMaxKeys) {
        return KVCM_ERR_TOO_LARGE;
    }
    return kvcm::table_capacity(n) * 4;
}

int32_t kvcm_hip_first_occurrence(const int64_t *d_keys, int64_t n, void *d_workspace, int64_t workspace_bytes,
                                  int32_t *d_first_idx, uint8_t *d_is_repeat, kvcm_stream_t stream) {
    if (n < 0) {
        return KVCM_ERR_INVALID_ARG;
    }
    if (n == 0) {
        return KVCM_OK;
    }
    if (n > kvcm::kMaxKeys) {
        return KVCM_ERR_TOO_LARGE;
    }
    if (!d_keys || !d_workspace || !d_first_idx) {
        return KVCM_ERR_INVALID_ARG;
    }
    const int64_t cap = kvcm::table_capacity(n);
    if (workspace_bytes < cap * 4) {
        return KVCM_ERR_INVALID_ARG;
    }
    if (reinterpret_cast<uintptr_t>(d_workspace) % 4 != 0) {
        return KVCM_ERR_ALIGNMENT;
    }
    return kvcm::launch_first_occurrence(d_keys, n, static_cast<int32_t *>(d_workspace), cap, d_first_idx, d_is_repeat,
                                         static_cast<hipStream_t>(stream));
}

int64_t kvcm_hip_first_occurrence_static_max_keys(void) { return kvcm::kStaticMaxKeys; }

int32_t kvcm_hip_first_occurrence_static(const int64_t *d_keys, int64_t n, int32_t *d_first_idx, uint8_t *d_is_repeat,
                                         kvcm_stream_t stream) {
    if (n < 0) {
        return KVCM_ERR_INVALID_ARG;
    }
    if (n > kvcm::kStaticMaxKeys) {
        return KVCM_ERR_TOO_LARGE;
    }
    if (n > 0 && (!d_keys || !d_first_idx)) {
        return KVCM_ERR_INVALID_ARG;
    }
    // also for n == 0: a call with no keys is how a caller does the per-device set-up ahead of time
    int32_t *table = nullptr;
    const int32_t rc = kvcm::static_scratch(&table);
    if (rc != KVCM_OK) {
        return rc;
    }
    if (n == 0) {
        return KVCM_OK;
    }
    // the table keeps the last call's contents: the fill kernel clears the slots this call probes
    return kvcm::launch_first_occurrence(d_keys, n, table, kvcm::table_capacity(n), d_first_idx, d_is_repeat,
                                         static_cast<hipStream_t>(stream));
}

int64_t kvcm_hip_mask_to_indices_workspace_bytes(int64_t n) {
    if (n < 0 || n > kvcm::kMaxKeys) {
        return KVCM_ERR_TOO_LARGE;
    }
    return ((n + kvcm::kSelThreads - 1) / kvcm::kSelThreads + 1) * 4;
}

int32_t kvcm_hip_mask_to_indices(const uint8_t *d_mask, const uint8_t *d_mask2, int64_t n, void *d_workspace,
                                 int64_t workspace_bytes, int32_t *d_indices, int32_t *d_count,
                                 kvcm_stream_t stream) {
    if (n < 0 || !d_count) {
        return KVCM_ERR_INVALID_ARG;
    }
    if (n > kvcm::kMaxKeys) {
        return KVCM_ERR_TOO_LARGE;
    }
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (n == 0) {
        kvcm::fill_i32_kernel<<<1, 256, 0, s>>>(d_count, 1, 0);
        return kvcm::launch_status();
    }
    if (!d_mask || !d_workspace || !d_indices) {
        return KVCM_ERR_INVALID_ARG;
    }
    const int64_t G = (n + kvcm::kSelThreads - 1) / kvcm::kSelThreads;
    if (workspace_bytes < (G + 1) * 4) {
        return KVCM_ERR_INVALID_ARG;
    }
    if (reinterpret_cast<uintptr_t>(d_workspace) % 4 != 0) {
        return KVCM_ERR_ALIGNMENT;
    }
    int32_t *counts = static_cast<int32_t *>(d_workspace);
    const int32_t n32 = static_cast<int32_t>(n), G32 = static_cast<int32_t>(G);
    kvcm::count_kernel<<<G32, kvcm::kSelThreads, 0, s>>>(d_mask, d_mask2, n32, counts);
    kvcm::scan_kernel<<<1, kvcm::kSelThreads, 0, s>>>(counts, G32, d_count);
    kvcm::write_kernel<<<G32, kvcm::kSelThreads, 0, s>>>(d_mask, d_mask2, n32, counts, d_indices);
    return kvcm::launch_status();
}

int64_t kvcm_hip_select_save_max_keys(void) { return kvcm::kListMaxKeys; }

int64_t kvcm_hip_select_save_workspace_bytes(int64_t n) {
    if (n < 0 || n > kvcm::kListMaxKeys) {
        return KVCM_ERR_TOO_LARGE;
    }
    // words first (8-byte aligned), then table, slots and counts; up to kPartMaxKeys keys the first n bytes are flags instead
    return kvcm::list_groups(n) * (kvcm::kListWaves * 8 + 4) + (kvcm::list_capacity(n) + n) * 4;
}

int32_t kvcm_hip_select_save(const int64_t *d_keys, const uint8_t *d_saved, int64_t n, void *d_workspace,
                             int64_t workspace_bytes, int32_t *d_indices, int32_t *d_count, kvcm_stream_t stream) {
    if (n <= 0 || !d_keys || !d_workspace || !d_indices || !d_count) {
        return KVCM_ERR_INVALID_ARG;
    }
    if (n > kvcm::kListMaxKeys) {
        return KVCM_ERR_TOO_LARGE;
    }
    if (workspace_bytes < kvcm_hip_select_save_workspace_bytes(n)) {
        return KVCM_ERR_INVALID_ARG;
    }
    if (reinterpret_cast<uintptr_t>(d_workspace) % 8 != 0) {
        return KVCM_ERR_ALIGNMENT;
    }
    const hipStream_t s = static_cast<hipStream_t>(stream);
    if (n <= kvcm::kPartMaxKeys) {
        const kvcm::PartShape p = kvcm::part_shape(n);
        uint8_t *const flags = static_cast<uint8_t *>(d_workspace);
        kvcm::part_kernel<<<1u << p.log2_parts, kvcm::kPartThreads, 12u << p.log2_slots, s>>>(
            reinterpret_cast<const uint64_t *>(d_keys), static_cast<int32_t>(n), p.log2_parts, p.log2_slots, d_saved, flags);
        kvcm::part_list_kernel<<<static_cast<unsigned>((n + 1023) / 1024), kvcm::kPartListThreads, 0, s>>>(
            reinterpret_cast<const uint32_t *>(flags), static_cast<int32_t>(n), d_indices, d_count);
        return kvcm::launch_status();
    }
    const int64_t groups = kvcm::list_groups(n), cap = kvcm::list_capacity(n);
    uint64_t *words = static_cast<uint64_t *>(d_workspace);
    int32_t *table = reinterpret_cast<int32_t *>(words + groups * kvcm::kListWaves);
    int32_t *slot_of = table + cap, *counts = slot_of + n;
    const int32_t n32 = static_cast<int32_t>(n);
    const unsigned grid = static_cast<unsigned>(groups);
    kvcm::launch_insert(d_keys, n32, table, cap, slot_of, s);
    kvcm::choose_kernel<<<grid, kvcm::kListThreads, 0, s>>>(slot_of, table, d_saved, n32, words, counts);
    kvcm::list_kernel<<<grid, kvcm::kListThreads, 0, s>>>(words, counts, d_indices, d_count);
    return kvcm::launch_status();
}

}  // extern "C"
