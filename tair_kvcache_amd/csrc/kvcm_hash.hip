// kvcm_hash.hip -- block keys of token-ID sequences, batched over requests.
//
// Function: GenKeyVector (kv_cache_manager/manager/cache_manager.cc:76-87) over hashInt64Array
// (kv_cache_manager/manager/hash_util.h:14-24): ONE running 64-bit state per request goes through every
// token, h <- h ^ (v + C + (h << 12) + (h >> 32)), and is emitted at every block boundary. The step mixes
// + and ^, so a request is a serial chain of len dependent steps; the parallelism is across requests.
//
// Two kernels, by number of requests. Up to kLeanUpTo (4096) hash_lean_kernel: 16 requests per workgroup, so that there is one for
// each compute unit; its design and what bounds it stand above it. Beyond, hash_tokens_kernel:
// Design (gfx950, wave64): a workgroup owns 64 requests and is role-split.
//   wave 0      "chain wave": lane = request. Keeps the state in VGPRs and does nothing but the recurrence,
//               reading pre-added terms a = v + C from LDS (one ds_read_b128 per 2 steps, prefetched a whole
//               tile ahead into a second register set). A wave issues one instruction every 4 clocks, so the step is
//               written for their number: 5 instructions (see chain_step).
//   waves 1..3  "loader waves": stream the 64 requests' tokens from HBM in [64 requests x 64 tokens] tiles with
//               16-byte buffer loads (512-byte row segments), add C, and write them transposed into a 2-slot LDS
//               ring. Each loader wave owns every third tile and keeps its loads in flight for about three
//               tile periods, so HBM latency stays off the chain. In launches of thousands of requests they also
//               write the keys out: the chain wave leaves them in an LDS buffer, and whole 512-byte rows per
//               request go to memory (kKeysSpread / kKeysBurst) instead of one 8-byte store per key and lane.
//               With 4-byte tokens such launches use tiles of 128 RAW tokens (512-byte row segments here too): the
//               loaders store what they loaded and the chain wave converts, one step ahead of its use.
// Roofline: HBM for many requests (8*block_size + 8 bytes per key); for few requests the bound is the
// instruction issue of the chain wave, which no amount of bandwidth removes.
#include "kvcm_internal.h"
#include "kvcm_key_count.h"

#include <climits>

namespace kvcm {
namespace {

#ifndef KVCM_HASH_LOADERS
#define KVCM_HASH_LOADERS 3
#endif
#ifndef KVCM_HASH_RAW_AHEAD
#define KVCM_HASH_RAW_AHEAD 1
#endif
#ifndef KVCM_HASH_TILE_TOKENS
#define KVCM_HASH_TILE_TOKENS 64
#endif

// Loader waves. Three, so that the four waves of a workgroup sit on the four SIMDs of a CU: the chain wave needs about
// 280 VGPRs (two register sets of 64 pre-added terms) and must not share its SIMD's register file. More loaders were
// measured with 32-token tiles (where the registers fit): no gain at 16 384 requests, 5 % slower for one batch.
constexpr int kLoaders = KVCM_HASH_LOADERS;
constexpr int kThreads = 64 * (1 + kLoaders);
constexpr int kReqs = 64;                     // requests per workgroup = lanes of the chain wave
constexpr int kTT = KVCM_HASH_TILE_TOKENS;    // tokens per request per tile
constexpr int kRing = 2;                      // LDS tiles in the ring: prefetched from, written to (the tile that is
                                              // computed on already sits in the chain wave's registers)
constexpr int kPad = 2;                       // keeps rows 16-byte aligned (b128 reads) and spreads banks
// Raw tiles (4-byte tokens, many requests in flight): a ring slot holds [64 requests x 128 RAW int32 tokens] -- the same
// bytes as 64 pre-added 64-bit terms -- so that a request's share of a tile is 512 contiguous bytes of the token stream
// instead of 256 (the memory system serves 256-byte pieces at little more than half the rate of 512-byte ones), and the
// chain wave sign-extends and adds the constant itself, one instruction per step beside the chain.
constexpr int tile_tokens(bool raw) { return raw ? 2 * kTT : kTT; }
constexpr int kRowVecs = kTT / 2;  // 16-byte pieces of one request's row of a tile, either format
// Staged keys (many requests in flight; block sizes 1, 8, 16, 32, 64 and 128): the keys of a GROUP of tiles collect in LDS
// and leave as whole rows of 512 bytes per request, see hash_tokens_kernel. A group is as many tiles as yield 64 keys per
// request: key_group_tiles(block size), i.e. one tile at block size 1, sixteen at block size 16, 128 at block size 128.
constexpr int kKeysPerGroup = 64;
constexpr int key_group_tiles(int bs, int tok = kTT) { return bs >= 1 && bs <= 2 * kTT ? kKeysPerGroup * bs / tok : 16; }
constexpr int kKeyGroupTiles = key_group_tiles(16);  // the spread form exists for block size 16 only
static_assert(key_group_tiles(1) == 1 && key_group_tiles(16) == 16 && key_group_tiles(128) == 128, "64 keys per group");
constexpr int kKeyPad = 2;
constexpr int kKeyRow = kKeysPerGroup + kKeyPad;  // one request's row of the LDS key buffer

// Workgroup barrier that waits only for this wave's LDS traffic. __syncthreads() would also drain the
// loader waves' outstanding global loads, which must stay in flight across barriers.
// Spelled with builtins so that the compiler's own wait-count bookkeeping sees the LDS wait: after it the chain
// wave's prefetched tile counts as arrived and its steps run without further waits.
__device__ __forceinline__ void lds_barrier() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0); vmcnt and expcnt left at their maxima
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

// One step of the recurrence with the token term pre-added (a = v + C): h ^= a + (h << 12) + sar(h, 32).
// The wave that sets the pace issues one vector instruction every 4 clocks, dependent on its predecessor or not (64 steps in
// a row take 20.9 clocks each, 8.7 ns), so what counts is the number of instructions: these five, and everything else that
// takes an issue slot of this wave -- LDS reads, key stores, waits, loop control. sar(h, 32) is the sign-extended upper
// half, and v_mad_i64_i32 (hi * 1 + a) adds it to `a` in ONE instruction; v_lshlrev_b64, v_lshl_add_u64 and two v_xor_b32
// are the rest (forms with v_mad_u64_u32 for the shift, or in 32-bit halves with carries, take as many or more: 37 to 46
// clocks measured step by step where this one took 25).
__device__ __forceinline__ uint64_t chain_step(uint64_t h, uint64_t a) {
    uint64_t a_plus_sar, carry_out;
    asm("v_mad_i64_i32 %0, %1, %2, 1, %3"
        : "=v"(a_plus_sar), "=s"(carry_out)
        : "v"(static_cast<uint32_t>(h >> 32)), "v"(a));
    return h ^ (a_plus_sar + (h << 12));
}

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

// sign-extended 32-bit token + C in one instruction (the compiler's own form is a shift for the sign and a 64-bit
// add): with 32-bit tokens the loader wave whose turn it is has twice as many tokens to convert per load, and its
// store phase must stay shorter than the chain wave's tile
__device__ __forceinline__ uint64_t pre_add_i32(uint32_t token) {
    uint64_t sum, carry_out;
    asm("v_mad_i64_i32 %0, %1, %2, 1, %3" : "=v"(sum), "=s"(carry_out) : "v"(token), "s"(kGolden));
    return sum;
}

// Maximum / minimum of a 32-bit value over the 64 lanes of a wave, returned as a wave-uniform value. Data-parallel
// primitives within rows of 16 lanes, then across rows: six steps of one or two instructions, against six round trips
// through the LDS crossbar for the shuffle form (0.5 us at the head of a kernel that lasts 50).
template <bool MAX>
__device__ __forceinline__ uint32_t wave_reduce_u32(uint32_t v) {
#define KVCM_DPP_STEP(CTRL)                                                                                       \
    {                                                                                                             \
        const uint32_t o = static_cast<uint32_t>(__builtin_amdgcn_update_dpp(static_cast<int>(v), static_cast<int>(v), \
                                                                             CTRL, 0xf, 0xf, false));             \
        v = MAX ? (o > v ? o : v) : (o < v ? o : v);                                                              \
    }
    KVCM_DPP_STEP(0x111)  // row_shr:1   a lane without a source keeps its own value
    KVCM_DPP_STEP(0x112)  // row_shr:2
    KVCM_DPP_STEP(0x114)  // row_shr:4
    KVCM_DPP_STEP(0x118)  // row_shr:8   lane 15 of every row now holds the row's result
    KVCM_DPP_STEP(0x142)  // row_bcast:15
    KVCM_DPP_STEP(0x143)  // row_bcast:31  lane 63 holds the wave's
#undef KVCM_DPP_STEP
    return static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(v), 63));
}
__device__ __forceinline__ uint32_t wave_max_u32(uint32_t v) { return wave_reduce_u32<true>(v); }
__device__ __forceinline__ uint32_t wave_min_u32(uint32_t v) { return wave_reduce_u32<false>(v); }

// What a loader wave needs to know about its workgroup.
template <typename TokT>
struct LoaderCtx {
    const TokT *tokens;
    const int64_t *s_start;  // LDS: first token of each of the 64 requests
    int64_t last_token;      // index of the last token of the whole batch (clamp target)
    int64_t wg_first_token;  // first token of the workgroup's first request
    uint32_t wg_bytes;       // bytes from there to the end of the batch, saturated at 2^32 - 1
};

// Loader, fast form: 16-byte BUFFER loads. One load instruction covers 64 / kLPR request rows with kLPR lanes
// each, so a tile takes kNL loads per lane (32 for int64 tokens, 16 for int32). The buffer resource spans from the
// workgroup's first token to the end of the batch: the hardware returns zeros past the end instead of faulting, so
// the loads need no clamp, and a load costs two instructions (offset add + buffer_load_dwordx4). Positions past a
// request's own last hashed token read a neighbour's tokens; the chain wave never consumes those entries.
template <typename TokT, bool RAW = false>
struct BufferLoader {
    static_assert(!RAW || sizeof(TokT) == 4, "raw tiles hold 4-byte tokens");
    static constexpr int kEPL = 16 / sizeof(TokT);  // tokens per load
    static constexpr int kLPR = tile_tokens(RAW) / kEPL;  // lanes per request row
    static constexpr int kRPW = 64 / kLPR;          // request rows per load instruction
    static constexpr int kNL = kReqs / kRPW;        // loads per lane per tile
    __amdgpu_buffer_rsrc_t rsrc;
    uint32_t rel[kNL];  // byte offset of this lane's piece of row j, tile 0
    u32x4 regs[kNL];
    uint32_t lane;

    __device__ __forceinline__ void setup(const LoaderCtx<TokT> &c, uint32_t lane_) {
        lane = lane_;
        rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<TokT *>(c.tokens + c.wg_first_token), 0, c.wg_bytes,
                                                 0x00020000);
        const uint32_t sub = lane / kLPR, piece = lane % kLPR;
#pragma unroll
        for (int j = 0; j < kNL; ++j) {
            rel[j] = static_cast<uint32_t>((c.s_start[j * kRPW + sub] - c.wg_first_token) * sizeof(TokT)) + piece * 16u;
        }
    }
    __device__ __forceinline__ void issue(int64_t t0) {
        issue_half<0>(t0);
        issue_half<1>(t0);
    }
    template <int HALF>
    __device__ __forceinline__ void issue_half(int64_t t0) {
        const uint32_t tile_off = static_cast<uint32_t>(t0 * sizeof(TokT));
#pragma unroll
        for (int j = HALF * (kNL / 2); j < (HALF + 1) * (kNL / 2); ++j) {
            // aux = 2: the non-temporal bit (sc0, sc1 and both were measured as well: only nt matters). Tokens are
            // read once. Timed the way the kernel is used -- on tokens that are not in the 256 MiB memory-side cache,
            // which holds other dirty data -- the bit is worth 30 to 45 % from 4096 requests up, for either token
            // width (8192 x 4096 8-byte tokens: 68 us against 96; 16 384 x 4096 4-byte tokens: 83 against 125) and
            // 5 % for one batch. Launched over and over on the same 256 MiB or less, the kernel without the bit reads
            // that cache instead of HBM and looks 10 to 25 % faster than with it: a benchmark's artefact.
            regs[j] = __builtin_amdgcn_raw_buffer_load_b128(rsrc, rel[j] + tile_off, 0, 2);
        }
    }
    // Adds the golden-ratio constant (the token term of the step is v + C) and writes the tile transposed.
    __device__ __forceinline__ void store(uint64_t (*tile)[kTT + kPad]) const {
        const uint32_t sub = lane / kLPR, piece = lane % kLPR;
        // One wait for all the loads of the tile (they were requested two tile periods ago) instead of one in front
        // of every LDS write: this phase has to fit into the chain wave's tile, and every instruction of it counts.
        __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0); lgkmcnt and expcnt left at their maxima
#pragma unroll
        for (int j = 0; j < kNL; ++j) {
            const u32x4 v = regs[j];
            if (RAW) {
                reinterpret_cast<u32x4 *>(&tile[j * kRPW + sub][0])[piece] = v;  // as it came: the chain wave converts
                continue;
            }
            ulonglong2 *dst = reinterpret_cast<ulonglong2 *>(&tile[j * kRPW + sub][piece * kEPL]);
            if (sizeof(TokT) == 8) {
                dst[0] = make_ulonglong2(((static_cast<uint64_t>(v.y) << 32) | v.x) + kGolden,
                                         ((static_cast<uint64_t>(v.w) << 32) | v.z) + kGolden);
            } else {
                dst[0] = make_ulonglong2(pre_add_i32(v.x), pre_add_i32(v.y));
                dst[1] = make_ulonglong2(pre_add_i32(v.z), pre_add_i32(v.w));
            }
        }
    }
};

// Offsets need not ascend: a request may begin in front of its workgroup's first token. So loads count from the first token of
// all wherever 32 bits reach the last one, and only in larger arrays from the workgroup's first. There a request may be out of reach,
// in front of it or 4 GiB and more behind it; hash_lean_kernel looks at each, hash_tokens_kernel (where that costs block size 1 up to
// 2 %) at where the workgroup's last one ends.
constexpr uint64_t kBufferReach = 0xFFF00000u;
template <typename TokT>
__device__ __forceinline__ bool within_reach(int64_t total) { return static_cast<uint64_t>(total) < kBufferReach / sizeof(TokT); }
template <typename TokT>
__device__ __forceinline__ bool out_of_reach(int64_t start, int64_t ntok, int64_t first) {
    return ntok > 0 && (start < first || !within_reach<TokT>(start - first + ntok));
}

// Loader, general form: one element per load through global addresses, positions clamped to the last token of
// the batch. Used when a 32-bit buffer offset does not reach one of the workgroup's requests.
template <typename TokT, bool RAW = false>
struct GlobalLoader {
    static constexpr int kTok = tile_tokens(RAW);
    static constexpr int kPerLane = kReqs * kTok / 64;  // tile elements per loader lane
    LoaderCtx<TokT> c;
    TokT regs[kPerLane];
    uint32_t lane;

    __device__ __forceinline__ void setup(const LoaderCtx<TokT> &c_, uint32_t lane_) {
        c = c_;
        lane = lane_;
    }
    __device__ __forceinline__ void issue(int64_t t0) {
        issue_half<0>(t0);
        issue_half<1>(t0);
    }
    template <int HALF>
    __device__ __forceinline__ void issue_half(int64_t t0) {
#pragma unroll
        for (int j = HALF * (kPerLane / 2); j < (HALF + 1) * (kPerLane / 2); ++j) {
            const uint32_t e = lane + 64u * j;
            const int64_t pos = c.s_start[e / kTok] + t0 + (e % kTok);
            regs[j] = c.tokens[pos < c.last_token ? pos : c.last_token];
        }
    }
    __device__ __forceinline__ void store(uint64_t (*tile)[kTT + kPad]) const {
#pragma unroll
        for (int j = 0; j < kPerLane; ++j) {
            const uint32_t e = lane + 64u * j;
            if (RAW) {
                reinterpret_cast<uint32_t *>(&tile[e / kTok][0])[e % kTok] = static_cast<uint32_t>(regs[j]);
            } else {
                tile[e / kTok][e % kTok] = static_cast<uint64_t>(static_cast<int64_t>(regs[j])) + kGolden;
            }
        }
    }
};

// A request's place among the keys, as the loaders that write staged keys need it.
struct KeyRow {
    int64_t first;   // index of its first key
    int64_t count;   // keys it has; 0 for a row without a request
};

// What a loader wave needs to write out a group of staged keys (KS kernels only).
struct KeyDrain {
    const uint64_t *s_keys;      // LDS: [2][request][kKeyRow] keys of the group being filled and of the one before
    const KeyRow *s_keyrow;      // LDS: where each request's keys go, and how many it has
    int64_t *keys;
};

// Sixteen bytes of staged keys -> global. The chain wave fills rows to the end of the group whether the request still has
// tokens or not; what lies behind a request's last key stays here. POLICY: 0 written through at system scope, 1 non-temporal.
template <int POLICY>
__device__ __forceinline__ void store_keys(const KeyDrain &kd, const KeyRow &row, int32_t group, uint32_t piece, const u32x4 &v) {
    const int64_t at = static_cast<int64_t>(group) * kKeysPerGroup + piece * 2;
    int64_t *dst = kd.keys + row.first + at;
    if (at + 2 <= row.count) {
        if (POLICY == 0) {
            asm volatile("global_store_dwordx4 %0, %1, off sc0 sc1" : : "v"(dst), "v"(v) : "memory");
        } else {
            typedef u32x4 u32x4_a8 __attribute__((aligned(8)));
            __builtin_nontemporal_store(v, reinterpret_cast<u32x4_a8 *>(dst));
        }
    } else if (at < row.count) {
        *dst = static_cast<int64_t>((static_cast<uint64_t>(v.y) << 32) | v.x);
    }
}

// One group of staged keys, LDS -> global: every store instruction writes two requests' rows of 512 bytes, whole cache
// lines, non-temporal. Written as 8-byte stores from the chain wave (one line per lane, a sixteenth of it at a time)
// the 32 MiB of keys of a 16 384-request batch cost 20 us of a 107 us launch -- not for their bytes but for what they do
// to the memory system in the middle of the token stream; the same stores into a buffer that stays in the L2 cost
// nothing, and so do they as one burst after the last token. Whole rows at intervals of sixteen tiles recover a third
// of that.
// A group is 32 such store instructions; `step` (0..15) selects two of them, so that the work spreads over the sixteen
// tiles that follow the group instead of holding one loader back from its next barrier.
constexpr int kDrainSteps = kKeyGroupTiles;
constexpr int kDrainPerStep = kReqs * kKeysPerGroup / 128 / kDrainSteps;
__device__ __forceinline__ void drain_keys(const KeyDrain &kd, int32_t group, int32_t step, uint32_t lane) {
    const uint32_t buf = static_cast<uint32_t>(group) & 1u;
#pragma unroll
    for (int j = 0; j < kDrainPerStep; ++j) {
        const uint32_t c = static_cast<uint32_t>(step * kDrainPerStep + j) * 64u + lane;  // 16-byte piece of the group's keys
        const uint32_t row = c / (kKeysPerGroup / 2), piece = c % (kKeysPerGroup / 2);
        const u32x4 v = *reinterpret_cast<const u32x4 *>(kd.s_keys + (buf * kReqs + row) * kKeyRow + piece * 2);
        store_keys<1>(kd, kd.s_keyrow[row], group, piece, v);
    }
}

// Half of a closed group (`part` = 0 or 1: every other store instruction), in bursts of eight row pieces: all LDS reads
// of a burst are under way before its first store goes out, so the loader is back at its loads after about 0.2 us.
// Written through at system scope: 97-99 us for 16 384 x 4096 tokens where the same stores take 101-105 us non-temporal, 104
// plain, 100-101 with sc1 alone (65 536 x 4096: 385-388 against 399-403 us).
__device__ __forceinline__ void drain_half(const KeyDrain &kd, int32_t group, int32_t part, uint32_t lane) {
    const uint32_t buf = static_cast<uint32_t>(group) & 1u;
    constexpr int kBurst = 8;
    static_assert((kDrainSteps * kDrainPerStep / 2) % kBurst == 0, "whole bursts");
#pragma unroll 1
    for (int32_t base = 0; base < kDrainSteps * kDrainPerStep / 2; base += kBurst) {
        KeyRow to[kBurst];
        u32x4 v[kBurst];
        uint32_t piece[kBurst];
#pragma unroll
        for (int i = 0; i < kBurst; ++i) {
            const uint32_t c = static_cast<uint32_t>((base + i) * 2 + part) * 64u + lane;
            const uint32_t row = c / (kKeysPerGroup / 2);
            piece[i] = c % (kKeysPerGroup / 2);
            to[i] = kd.s_keyrow[row];
            v[i] = *reinterpret_cast<const u32x4 *>(kd.s_keys + (buf * kReqs + row) * kKeyRow + piece[i] * 2);
        }
#pragma unroll
        for (int i = 0; i < kBurst; ++i) {
            store_keys<0>(kd, to[i], group, piece[i], v[i]);
        }
    }
}

// How a kernel's keys reach memory: from the chain wave, one at a time (kKeysDirect); staged in LDS and written by the
// loaders a sixteenth of a group per tile (kKeysSpread); staged and written a whole group at once, right after the
// barrier that closes it (kKeysBurst); the host chooses by token width and number of requests (the timings stand at
// launch_hash). Writes that all workgroups issue at the same moments disturb the token stream less than writes spread
// evenly through it, as long as the loaders do not fall behind while they issue them.
constexpr int kKeysDirect = 0, kKeysSpread = 1, kKeysBurst = 2;
// A workgroup of a spread kernel whose requests are shorter than this many tiles stores its keys directly: what the last
// group costs after the loop (about 1.5 us) is more than staging saves on 2048 tokens.
constexpr int kSpreadFromTiles = 32;
// Block size 1, 8-byte elements (the prefix chain): a workgroup in which nobody fills a tile stores its keys directly (1000 sequences
// of 4 to 64 digests 5.8 us, staged 6.2), and so does one of few equally long requests, the last of a launch, because a store takes
// the longer the more lanes it has (4096 digests each, 31 requests direct / staged 78 / 97, 32: 80 / 93, 48: 106 / 89, 64: 146 / 86).
// Where requests end at different places staging pays from two of them on: 4 requests of 64 to 4096 digests 155 / 100.
__device__ __forceinline__ bool chain_stays_direct(uint32_t requests, uint32_t ntiles, uint32_t whole) {
    return whole + 1 >= ntiles && (requests <= 32 || whole == 0);
}

// The steps [first_step, kDrainSteps) of a group that belong to loader `me` (step % kLoaders == me), all LDS reads
// under way before the first store: nothing else is left to do when this runs, so round trips would add up.
__device__ __forceinline__ void drain_tail(const KeyDrain &kd, int32_t group, int32_t first_step, int32_t me,
                                           uint32_t lane) {
    const uint32_t buf = static_cast<uint32_t>(group) & 1u;
    constexpr int kMaxSteps = (kDrainSteps + kLoaders - 1) / kLoaders;
    constexpr int kN = kMaxSteps * kDrainPerStep;
    const int32_t s0 = first_step + (me - first_step % kLoaders + kLoaders) % kLoaders;
    KeyRow to[kN];
    u32x4 v[kN];
    uint32_t piece[kN];
#pragma unroll
    for (int i = 0; i < kN; ++i) {
        const int32_t step = s0 + (i / kDrainPerStep) * kLoaders;
        to[i].count = 0;
        if (step < kDrainSteps) {
            const uint32_t c = static_cast<uint32_t>(step * kDrainPerStep + i % kDrainPerStep) * 64u + lane;
            const uint32_t row = c / (kKeysPerGroup / 2);
            piece[i] = c % (kKeysPerGroup / 2);
            to[i] = kd.s_keyrow[row];
            v[i] = *reinterpret_cast<const u32x4 *>(kd.s_keys + (buf * kReqs + row) * kKeyRow + piece[i] * 2);
        }
    }
#pragma unroll
    for (int i = 0; i < kN; ++i) {
        store_keys<1>(kd, to[i], group, piece[i], v[i]);
    }
}

// A loader wave's whole life. Loader lw owns tiles lw, lw + kLoaders, ...; tile t lives in ring slot t % kRing.
// Tiles 0 and 1 are published before the first barrier: the chain wave computes on tile k while its LDS reads of
// tile k+1 are already in flight, so tile k+2 is what gets written during iteration k (its slot held tile k-1,
// which the chain wave pulled into registers an iteration ago). A loader issues the loads of its next tile right
// AFTER the barrier that published its previous one, so they stay in flight for kLoaders - 1 tile periods while the
// data waits in the loader's registers, not in LDS: more loaders = more bytes in flight per CU at no LDS cost.
// staged: the workgroup's keys pass through LDS and leave through the loaders; apart: reads and writes take turns.
template <typename Loader, typename TokT, int KS, int G, int TOK>
__device__ __forceinline__ void run_loader(const LoaderCtx<TokT> &ctx, uint64_t (*s_tile)[kReqs][kTT + kPad],
                                           int64_t lw, int64_t ntiles, uint32_t lane, const KeyDrain &kd, bool staged,
                                           bool apart) {
    static_assert(kRing == 2 && kLoaders >= 3, "two ring slots: prefetched from, written to");
    // the burst drain splits a closed group between the kLoaders - 1 loaders whose tile is not due, as halves
    static_assert(KS != kKeysBurst || kLoaders == 3, "drain_half deals a group out to exactly two loaders");
    static_assert((G & (G - 1)) == 0 && (KS != kKeysSpread || G == kKeyGroupTiles), "groups of 2^n tiles; spread: 16");
    Loader ld;
    ld.setup(ctx, lane);
    // 32-bit counters: the loop control stays in scalar registers (there are no ordered 64-bit scalar compares); a
    // request of 2^37 tokens does not fit the memory of the device
    const int32_t nt = static_cast<int32_t>(ntiles), me = static_cast<int32_t>(lw);
    if (me < nt) {
        ld.issue(static_cast<int64_t>(me) * TOK);
    }
    if (me < 2 && me < nt) {
        ld.store(s_tile[me]);
    }
    lds_barrier();
    if (me < 2 && me + kLoaders < nt) {
        ld.issue(static_cast<int64_t>(me + kLoaders) * TOK);
    }
    // tile 2 goes where tile 0 lies: not before the chain wave has pulled tile 0 into its registers
    lds_barrier();
    int32_t turn = 2 % kLoaders;  // loader whose tile is due: (k + 2) % kLoaders
    int slot = 2 % kRing;         // ring slot of that tile: (k + 2) % kRing
    bool was_mine = false;
    for (int32_t k = 0; k < nt; ++k) {
        const int32_t nxt = k + 2;  // tile that must be in LDS when this iteration ends
        const bool my_turn = turn == me;
        const bool mine = my_turn && nxt < nt;
        if (mine) {
            ld.store(s_tile[slot]);
        }
        if (KS == kKeysSpread && staged && k >= kKeyGroupTiles &&
            (turn == 0 ? kLoaders - 1 : turn - 1) == me) {
            // The group of staged keys before the one this tile belongs to was closed by an earlier barrier, and its
            // buffer is not written again before the barrier that ends this group: a sixteenth of it leaves per tile,
            // here, in front of the barrier, through the loader that published a tile an iteration ago and has nothing
            // to do until the barrier (its own next wait for memory is two tiles away, so the stores are not waited for).
            drain_keys(kd, k / kKeyGroupTiles - 1, k & (kKeyGroupTiles - 1), lane);
        }
        turn = turn + 1 == kLoaders ? 0 : turn + 1;
        slot = slot + 1 == kRing ? 0 : slot + 1;
        lds_barrier();
        // the loads of this loader's next tile go out in two halves, one tile period apart: a burst of 32 load
        // instructions sits in the CU's memory pipeline in front of the chain wave's key stores
        // (which of the two forms runs is a compile-time matter: with both in one loop body the compiler waits for
        // all outstanding loads where the paths meet, and a kernel that does so takes 80 us for a batch instead of 58)
        if (KS == kKeysSpread || (KS == kKeysBurst && sizeof(TokT) == 8)) {
            // no key stores of the chain wave to keep out of the way of: 2 to 5 % faster from 4096 requests than in
            // halves (spread form); in the burst form of 8-byte tokens 4 % at 10 240 and 12 288 requests, 7 to 10 % for
            // the prefix chain up to 2048 chains, nothing at 16 384. Raw tiles of 4-byte tokens lose 5 % by it at
            // 16 384 requests (66.8 against 63.6 us) and keep the halves.
            if (mine && nxt + kLoaders < nt) {
                ld.issue(static_cast<int64_t>(nxt + kLoaders) * TOK);
            }
        } else {
            if (mine && nxt + kLoaders < nt) {
                ld.template issue_half<0>(static_cast<int64_t>(nxt + kLoaders) * TOK);
            }
            if (was_mine && nxt - 1 + kLoaders < nt) {
                ld.template issue_half<1>(static_cast<int64_t>(nxt - 1 + kLoaders) * TOK);
            }
        }
        was_mine = mine;
        if (KS == kKeysBurst && staged && ((k & (G - 1)) == G - 1 || k == nt - 1) && turn != me) {
            // The barrier above closed a group of G tiles, or what there is of the last one. The loader whose tile is due
            // next leaves it alone (its next wait for memory would wait for these stores as well); the other two write half
            // of it each.
            if (G == 1 && apart) {
                __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): keys leave when the next tile's tokens are in
            }
            drain_half(kd, k / G, (me - turn + kLoaders) % kLoaders - 1, lane);
        }
    }
    if (KS == kKeysSpread && staged) {
        // What the loop did not reach: the rest of the last group but one, and all of the last group, the steps dealt out
        // to the loaders; no barrier follows, and nobody writes the buffers any more.
        const int32_t last = (nt - 1) / kKeyGroupTiles;
        if (last >= 1) {
            drain_tail(kd, last - 1, nt - last * kKeyGroupTiles, me, lane);
        }
        drain_tail(kd, last, 0, me, lane);
    }
}

// One group of a lane's row of a tile, LDS -> registers. The scheduler keeps the group where it stands: a lone wave issues a
// 16-byte read every 6 clocks in groups of 8, every 8.4 in groups of 32 (no more than 15 can be outstanding) and every 12
// when they stand alone between the steps. Two groups per tile against one, the whole kernel: 160 requests of up to 8192
// 4-byte tokens 103.9 / 109.3 us, 64 x 4096 8-byte tokens 52.1 / 52.1; four groups 103.3 and 52.9.
constexpr int kReadGroups = 2;
template <int N>
__device__ __forceinline__ void read_row_part(ulonglong2 (&a)[kRowVecs], const uint64_t *row_ptr, int group) {
    const ulonglong2 *row = reinterpret_cast<const ulonglong2 *>(row_ptr) + group * N;
#pragma unroll
    for (int i = 0; i < N; ++i) {
        a[group * N + i] = row[i];
    }
    __builtin_amdgcn_sched_barrier(0);
}

// The chain wave's work on one tile: kTT steps from the lane's pre-added terms `a`, a key at every block
// boundary. MASKED = some lane may have run out of tokens inside this tile (ragged batch). Such a lane keeps stepping
// -- on a neighbour's tokens or on zeros, whatever the loaders fetched past its end -- because masking the steps would
// cost the wave a compare, two exec writes and a branch per chunk; its state is dead from there on, and only its KEY
// STORES are masked. The common case of equally long requests takes the unmasked path, which has no per-lane compare.
// BS > 0 = the block size is this compile-time constant (a divisor or a multiple of the tile): the places where a key
// is due are then known when the code is written, and the scalar bookkeeping (add, compare, branch per chunk: one
// instruction slot in sixteen of the wave that sets the pace) disappears from the loop.
// STAGED (unmasked tiles, block size a compile-time constant up to two tiles): the tile's keys go to the lane's row of the LDS key buffer, `staged_row`
// pointing at the tile's first key there; a loader wave writes the rows out (drain_keys).
template <int CHUNK, bool MASKED, int BS, bool STAGED = false, bool RAW = false>
__device__ __forceinline__ void run_tile(const ulonglong2 (&a)[kRowVecs], ulonglong2 (&next)[kRowVecs],
                                         const uint64_t *next_row, uint64_t &h, int64_t t0, int64_t my_ntok,
                                         int32_t &since_key, int32_t block_size, int64_t *__restrict__ keys,
                                         int64_t &key_pos, uint64_t *staged_row = nullptr) {
    constexpr int TOK = tile_tokens(RAW);  // steps per tile
    static_assert(!STAGED || (!MASKED && BS >= 1 && BS <= 2 * kTT), "keys are staged for whole tiles of blocks up to two tiles");
    static_assert(BS == 0 || (BS % CHUNK == 0 && (TOK % BS == 0 || BS % TOK == 0)), "block size fits the tiling");
    // tokens of this lane that are hashed and lie in this tile or before its end: a block that ends at position p of
    // the tile belongs to the lane iff p <= left (my_ntok is a multiple of the block size)
    const int64_t left64 = my_ntok - t0;
    const int32_t left = MASKED ? static_cast<int32_t>(left64 < TOK ? (left64 > 0 ? left64 : 0) : TOK) : TOK;
    // raw tiles: four 4-byte tokens per 16-byte piece; sign-extension + C is one v_mad_i64_i32 off the chain, issued
    // KVCM_HASH_RAW_AHEAD steps before the step that consumes it
    const auto raw_token = [&](int s) -> uint32_t {
        const uint64_t pair = (s & 2) ? a[s / 4].y : a[s / 4].x;
        return static_cast<uint32_t>((s & 1) ? pair >> 32 : pair);
    };
    constexpr int kAhead = KVCM_HASH_RAW_AHEAD;
    uint64_t pre[kAhead > 0 ? kAhead : 1];
    if (RAW) {
#pragma unroll
        for (int i = 0; i < kAhead; ++i) {
            pre[i] = pre_add_i32(raw_token(i));
        }
    }
    uint64_t held = 0;
#pragma unroll
    for (int c = 0; c < TOK; c += CHUNK) {
        if (c % (TOK / kReadGroups) == 0) {
            read_row_part<kRowVecs / kReadGroups>(next, next_row, c / (TOK / kReadGroups));
        }
#pragma unroll
        for (int s = c; s < c + CHUNK; ++s) {
            if (RAW && kAhead > 0) {
                const uint64_t now = pre[s % kAhead];
                if (s + kAhead < TOK) {
                    pre[s % kAhead] = pre_add_i32(raw_token(s + kAhead));
                }
                h = chain_step(h, now);
            } else if (RAW) {
                h = chain_step(h, pre_add_i32(raw_token(s)));
            } else {
                h = chain_step(h, (s & 1) ? a[s / 2].y : a[s / 2].x);
            }
        }
        bool key_due;
        if (BS == 0) {
            since_key += CHUNK;
            key_due = since_key == block_size;
            if (key_due) {
                since_key = 0;
            }
        } else if (BS <= TOK) {
            key_due = (c + CHUNK) % BS == 0;  // tiles start on block boundaries
        } else {
            key_due = c + CHUNK == TOK && (t0 + TOK) % BS == 0;
        }
        if (key_due) {
            // Where a tile holds an even number of keys they leave two at a time, 16 bytes per lane: every lane's key lies
            // in a cache line of its own, and it is the lines that a store takes its time for, not the bytes (a store of
            // 64 lanes into 64 lines costs the chain 35 clocks; 64 requests of 4096 tokens 54.5 -> 52.2 us).
            constexpr bool kPaired = !MASKED && BS >= 1 && TOK % (2 * (BS > 0 ? BS : 1)) == 0;
            const int key_in_tile = BS > TOK ? 0 : (c + CHUNK) / (BS > 0 ? BS : 1) - 1;
            if (kPaired && key_in_tile % 2 == 0) {
                held = h;
            } else if (kPaired && STAGED) {
                *reinterpret_cast<ulonglong2 *>(staged_row + key_in_tile - 1) = make_ulonglong2(held, h);
            } else if (kPaired) {
                typedef uint64_t u64x2 __attribute__((ext_vector_type(2)));
                typedef u64x2 u64x2_a8 __attribute__((aligned(8)));  // one store: wide accesses need dword alignment only
                *reinterpret_cast<u64x2_a8 *>(keys + key_pos - 1) = u64x2{held, h};
            } else if (STAGED) {
                staged_row[key_in_tile] = h;
            } else if (!MASKED || c + CHUNK <= left) {
                keys[key_pos] = static_cast<int64_t>(h);
            }
            key_pos += 1;
        }
    }
}

// R requests of the same length, one behind the other (the kernel's token_offsets is NULL): nothing has to be read before
// the first tokens, and the key offsets, which follow from the sizes, are written on the side where the caller wants them
// -- one launch instead of eight (the offsets were computed by seven small launches in front of this one: 42 us of host
// time for a launch that lasts 9).
struct Uniform {
    int64_t tokens;            // tokens per request
    int64_t keys;              // tokens / block size
    int64_t *key_offsets_out;  // [R + 1], or NULL
};

// What the arrays hold, for launches with offsets: a request that names tokens or key slots beyond it is left out, and no
// load leaves the tokens, whatever the offsets say.
struct Extent {
    int64_t tokens;
    int64_t keys;
};

// Block size 1 writes as much as it reads. Where every request of a workgroup starts at the same place of a 32 KiB period, their
// pieces meet in the same channels of memory, and with a workgroup on every CU reads and writes are better kept apart: a loader
// waits for its tokens before it writes keys. us with / without that wait: 16 384 sequences of 4096 digests 220 / 231, of 8192:
// 427 / 489, 65 536 of 4096: 799 / 858, 16 384 of 8192 4-byte tokens 352 / 410; but of 2048 (16 KiB apart) 128 / 121, of 6144
// (48 KiB) 339 / 330, of 4000 to 4160: 330 / 320, and 8192 sequences of 4096, half the CUs, 154 / 122.
constexpr uint32_t kApartPeriod = 32768;
constexpr uint32_t kApartFromWorkgroups = 240;

// CHUNK = steps between two looks at the block boundary: 8 when block_size % 8 == 0 (a lane is then
// active for whole chunks or not at all), otherwise 1. BS = block size when it is 1, 8, 16, 32, 64 or 128, otherwise 0.
// KS != kKeysDirect ("keys staged", the block sizes with a kernel of their own; chosen by the host where the keys' way to memory
// bounds the launch: many requests, or a key after every token): the chain wave writes its keys into an LDS buffer instead of to memory, whether
// a request still has tokens or not, and after every group of tiles the loader waves write out what there is of it as rows
// of up to 512 bytes, spread over the next group's tiles (block size 16) or at once.
template <typename TokT, int CHUNK, int BS, int KS = kKeysDirect, bool RAW = false>
__global__ __launch_bounds__(kThreads) void hash_tokens_kernel(const TokT *__restrict__ tokens,
                                                              const int64_t *__restrict__ token_offsets, int32_t R,
                                                              int32_t block_size, uint64_t seed,
                                                              int64_t *__restrict__ keys,
                                                              const int64_t *__restrict__ key_offsets,
                                                              const Uniform uni, const Extent have,
                                                              int32_t force_global_loads) {
    __shared__ __attribute__((aligned(16))) uint64_t s_tile[kRing][kReqs][kTT + kPad];
    __shared__ int64_t s_start[kReqs];
    __shared__ int64_t s_ntok[kReqs];
    static_assert(!KS || (BS >= 1 && BS <= 2 * kTT), "keys are staged for block sizes up to two tiles");
    static_assert(KS != kKeysSpread || BS == 16, "the spread form exists for 16-token blocks");
    constexpr int TOK = tile_tokens(RAW);        // tokens per request per tile
    constexpr int G = key_group_tiles(BS, TOK);  // tiles per group of staged keys
    static_assert(!KS || G >= 1, "a group of staged keys is at least one tile");
    constexpr int kDiv = BS > 0 ? BS : 1;  // the first key of tile t of a group lies at position t * TOK / BS of the row
    __shared__ __attribute__((aligned(16))) uint64_t s_keys[KS ? 2 * kReqs * kKeyRow : 2];
    __shared__ __attribute__((aligned(16))) KeyRow s_keyrow[KS ? kReqs : 1];

    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int64_t r = static_cast<int64_t>(blockIdx.x) * kReqs + lane;

    // Everything that has to come from memory before the first tile can be requested is asked for here, by all four
    // waves at once: one trip to memory instead of three in a row (a 64 x 4096 batch is only ~50 us long).
    int64_t my_ntok = 0, key_pos = 0;
    LoaderCtx<TokT> ctx;
    bool buffer_loads = false;
    int64_t first_start = 0;
    const int64_t r_first = static_cast<int64_t>(blockIdx.x) * kReqs;
    if (wave == 0) {
        int64_t start;
        if (token_offsets) {
            start = token_offsets[r_first];  // rows past R and requests without keys idle at the first row
            start = start < 0 && have.tokens != kUnknown ? 0 : start;
            if (r < R) {
                const int64_t at = token_offsets[r], n = distance(at, token_offsets[r + 1]);
                // a division by a constant where there is one: by a variable it takes longer than the loads in front of it
                const int32_t bs = BS > 0 ? BS : block_size;
                const int64_t nkeys = n / bs;  // a trailing partial block yields no key
                key_pos = key_offsets ? key_offsets[r] : r * (distance(token_offsets[0], token_offsets[1]) / bs);
                if (inside(key_pos, nkeys, have.keys) && (have.tokens == kUnknown || inside(at, nkeys * bs, have.tokens))) {
                    start = at;
                    my_ntok = nkeys * bs;
                }
            }
        } else {
            start = r_first * uni.tokens;
            if (r < R) {
                start = r * uni.tokens;
                my_ntok = uni.keys * block_size;
                key_pos = key_offsets ? key_offsets[r] : r * uni.keys;
            }
            my_ntok = key_pos < 0 ? 0 : my_ntok;  // a negative key offset: no keys are wanted for this request
        }
        s_start[lane] = start;
        s_ntok[lane] = my_ntok;
        if (KS) {
            s_keyrow[lane] = KeyRow{key_pos, my_ntok / kDiv};  // no tokens, no keys: rows past R among them
        }
    } else {
        ctx.tokens = tokens;
        ctx.s_start = s_start;
        const int64_t r_end = r_first + kReqs < R ? r_first + kReqs : R;
        const bool known = token_offsets && have.tokens != kUnknown;
        const int64_t total = !token_offsets ? R * uni.tokens : known ? have.tokens : token_offsets[R];
        ctx.last_token = total - 1;  // >= 0 whenever a tile is loaded: some request has a full block then
        first_start = token_offsets ? token_offsets[r_first] : r_first * uni.tokens;
        ctx.wg_first_token = within_reach<TokT>(total) ? 0 : first_start;
        if (known && (ctx.wg_first_token < 0 || ctx.wg_first_token > total)) {
            ctx.wg_first_token = ctx.wg_first_token < 0 ? 0 : total;
        }
        const uint64_t to_end = static_cast<uint64_t>(total - ctx.wg_first_token) * sizeof(TokT);
        ctx.wg_bytes = to_end > 0xFFFFFFFFull ? 0xFFFFFFFFu : static_cast<uint32_t>(to_end);
        const int64_t end_token = token_offsets ? token_offsets[r_end] : r_end * uni.tokens;
        const uint64_t wg_span = static_cast<uint64_t>(distance(ctx.wg_first_token, end_token)) * sizeof(TokT);
        buffer_loads = !force_global_loads && (within_reach<TokT>(total) || wg_span < kBufferReach);
        if (uni.key_offsets_out && wave == kLoaders) {  // the last loader: its first tile is the one needed last
            if (r < R) {
                uni.key_offsets_out[r] = r * uni.keys;
            }
            if (r_end == R && lane == 0) {
                uni.key_offsets_out[R] = R * uni.keys;
            }
        }
    }
    __syncthreads();

    // Tiles of the longest request (how long the workgroup runs) and whole tiles of the shortest (from where on some
    // lane has run out): max and min over the 64 lanes of per-lane tile counts, which fit 32 bits (a request of 2^37
    // tokens does not fit the memory of the device). Rows past R in the last workgroup count for neither.
    const int64_t lane_ntok = s_ntok[lane];
    const uint32_t ntiles_u = wave_max_u32(static_cast<uint32_t>((lane_ntok + TOK - 1) / TOK));
    const uint32_t full_u = wave_min_u32(r < R ? static_cast<uint32_t>(lane_ntok / TOK) : 0xFFFFFFFFu);
    const int64_t ntiles = ntiles_u;  // uniform over the workgroup
    if (ntiles == 0) {
        return;
    }
    // tiles [0, n_full) are those in which no request has run out of tokens
    const int32_t n_full = static_cast<int32_t>(full_u < ntiles_u ? full_u : ntiles_u);
    // whether this workgroup's keys are staged
    const bool staged =
        KS == kKeysSpread  ? ntiles_u >= static_cast<uint32_t>(kSpreadFromTiles)
        : KS != kKeysBurst ? false
        : BS == 1 && sizeof(TokT) == 8
            ? !chain_stays_direct(static_cast<uint32_t>(R - r_first < kReqs ? R - r_first : kReqs), ntiles_u, full_u)
            : true;
    if (wave != 0) {
        // ---------------------------------------------------------------- loader waves
        const KeyDrain kd{s_keys, s_keyrow, keys};
        const bool apart = BS == 1 && KS == kKeysBurst && gridDim.x >= kApartFromWorkgroups &&
                           __all((static_cast<uint32_t>(s_start[lane] - first_start) * sizeof(TokT)) % kApartPeriod == 0);
        if (buffer_loads) {
            run_loader<BufferLoader<TokT, RAW>, TokT, KS, G, TOK>(ctx, s_tile, wave - 1, ntiles, lane, kd, staged, apart);
        } else {
            run_loader<GlobalLoader<TokT, RAW>, TokT, KS, G, TOK>(ctx, s_tile, wave - 1, ntiles, lane, kd, staged, apart);
            // vmcnt(0), for the compiler's books: it lays this path out in front of the other one and would otherwise take
            // the registers of these loads for pending there, and wait for ALL outstanding loads -- the next tile's -- in
            // front of every group of keys that is written out (prefix chain, 64 x 4096: 113 us with that wait, 86 without)
            __builtin_amdgcn_s_waitcnt(0x0F70);
        }
        return;
    }

    // -------------------------------------------------------------------- chain wave
    uint64_t h = seed;
    int32_t since_key = 0;  // uniform: all lanes step in lockstep from token 0
    lds_barrier();
    if (r >= R) {
        // A lane without a request leaves here; the wave goes on without it (every workgroup has at least one request,
        // so the wave still meets every barrier). This keeps the unmasked path, whose key stores are unconditional,
        // usable when R is not a multiple of 64.
        return;
    }
    ulonglong2 cur[kRowVecs], nxt[kRowVecs];
    read_row_part<kRowVecs>(cur, &s_tile[0][lane][0], 0);
    lds_barrier();  // tile 0 is in registers: its slot may take tile 2
    // Loop control in 32-bit scalars (there are no ordered 64-bit scalar compares, and every vector compare is an issue
    // slot of this wave). A request of 2^37 tokens does not fit the memory of the device, so the tile count fits 32 bits.
    const int32_t nt = static_cast<int32_t>(ntiles);
    const auto staged_row = [&](int32_t k) -> uint64_t * {
        return KS ? s_keys + ((k / G & 1) * kReqs + lane) * kKeyRow + (k & (G - 1)) * TOK / kDiv : nullptr;
    };
    int ring = 0;
    for (int32_t k = 0; k < nt; k += 2) {
        // even tile: compute on `cur`, prefetch the odd tile into `nxt`; then the other way round
        int ring1 = ring + 1 == kRing ? 0 : ring + 1;
        const uint64_t *const row1 = &s_tile[ring1][lane][0];  // behind the last tile: read and not used
        if (KS && staged) {
            run_tile<CHUNK, false, BS, KS != kKeysDirect, RAW>(cur, nxt, row1, h, static_cast<int64_t>(k) * TOK, my_ntok,
                                                               since_key, block_size, keys, key_pos, staged_row(k));
        } else if (k < n_full) {
            run_tile<CHUNK, false, BS, false, RAW>(cur, nxt, row1, h, static_cast<int64_t>(k) * TOK, my_ntok, since_key,
                                                   block_size, keys, key_pos);
        } else {
            run_tile<CHUNK, true, BS, false, RAW>(cur, nxt, row1, h, static_cast<int64_t>(k) * TOK, my_ntok, since_key,
                                                  block_size, keys, key_pos);
        }
        lds_barrier();
        if (k + 1 >= nt) {
            break;
        }
        ring = ring1 + 1 == kRing ? 0 : ring1 + 1;
        const uint64_t *const row2 = &s_tile[ring][lane][0];
        if (KS && staged) {
            run_tile<CHUNK, false, BS, KS != kKeysDirect, RAW>(nxt, cur, row2, h, static_cast<int64_t>(k + 1) * TOK, my_ntok,
                                                               since_key, block_size, keys, key_pos, staged_row(k + 1));
        } else if (k + 1 < n_full) {
            run_tile<CHUNK, false, BS, false, RAW>(nxt, cur, row2, h, static_cast<int64_t>(k + 1) * TOK, my_ntok, since_key,
                                                   block_size, keys, key_pos);
        } else {
            run_tile<CHUNK, true, BS, false, RAW>(nxt, cur, row2, h, static_cast<int64_t>(k + 1) * TOK, my_ntok, since_key,
                                                  block_size, keys, key_pos);
        }
        lds_barrier();
    }
}

// ------------------------------------------------------------------------------------------- key offsets

// Where every request's keys go: exclusive prefix sums of len / block_size, and the total -- the latter straight into host
// memory, so that a caller who has to size something by it waits for THIS kernel (a few us) and not for the hash kernel
// behind it. Bound by latency: a workgroup scans kOffsetsPerWg requests, eight per thread (their nine offsets are in flight
// together), and adds up everything in front of its range itself instead of waiting for a pass of partial sums: one launch,
// no workspace. 160 requests 3.2 us against 7.5 us on the device (and 3.6 against 22 on the host) for five launches of a
// general prefix sum; 8192 requests 8.5 against 12.5, 16 384 10.1 against 12.8, then the re-reading shows: 65 536 20 / 13.
// From kOffsetsRereadUpTo requests on a launch in front leaves the sum of every workgroup's range (`sums`).
constexpr int kOffsetsThreads = 1024;
constexpr int kOffsetsPerThread = 8;
constexpr int64_t kOffsetsPerWg = kOffsetsThreads * kOffsetsPerThread;
constexpr int32_t kOffsetsRereadUpTo = 32768;
int64_t offsets_groups(int32_t R) { return (R + kOffsetsPerWg - 1) / kOffsetsPerWg; }

// For launches that count their keys themselves (hash_lean_kernel): where the offsets and the total go, or NULL twice.
struct CountOut {
    int64_t *key_offsets;  // [R + 1]
    int64_t *h_total;      // pinned
    FastDiv by_block;      // n / block size for n < 2^31
};

// ------------------------------------------------------------------------------------------- few requests per workgroup

// The kernel for launches that leave compute units idle when 64 requests share a workgroup (up to kLeanUpTo requests): 16 requests
// per workgroup, four waves on the four SIMDs of a compute unit.
//   wave 0     "chain wave": nothing but the recurrence, 32 steps at a time from terms read 32 steps ahead (two register sets of
//              64 registers: no accumulation registers), and every 16 steps the state, which is left in LDS two at a time.
//   waves 1, 2 loaders: 16 x 64 tokens as 16-byte buffer loads, two tiles each under way, C added, rows into an LDS ring.
//   wave 3     writer: picks the keys out of the states and stores them.
// Where keys lie between the states (block sizes that 16 does not divide, EVERY), the loader whose turn it is not goes through the
// tile again: 64 lanes of 16 steps each, from the states in front of them, and leaves the state after every step in the place of
// its term. So a key costs the chain nothing, whatever the block size, and requests that end early cost nothing either: the chain
// runs to the end of the longest, and only loaders and writer know where the others end.
//
// All 64 lanes of the chain wave stay active, four per request. A wave of which 16 lanes are active issues its instructions at
// 20.7 to 28.5 clocks per step, depending on the place of its compute unit on the die; with all lanes active it is 20.7 everywhere
// (five instructions of 4 clocks, measured on all 256 units).
//
// Bound: issue slots of the chain wave. Of 25 clocks per step (64 x 16 384 tokens: 10.8 ns) 20.7 are the step, 2.5 the reads of
// 16 bytes per two steps, 0.8 the state write (26 clocks per 32 steps), 1 the barrier per tile and loop control.
// us, before / now: 4 x 512 9.6 / 8.1, 64 x 4096 tokens 51.6 / 46.5, 4096 x 4096 55.8 / 49.2, 160 ragged of 48 to 8192 4-byte
// tokens 102.4 / 89.4, 64 x 4096 of block size 8: 58.7 / 47.3, 24: 64.5 / 47.2, 7: 151 / 48.4, 1: 85.7 / 48.3; prefix chain, 1000
// sequences of 8 to 1024: 27.5 / 15.6.
// Tiles of 128 tokens (half as many barriers) take 46.8 and 8.8 where these take 46.5 and 8.2; without the idle loaders' help the
// writer sets the pace at block size 1 (75).
constexpr int kLeanRows = 16;    // requests per workgroup
constexpr int kLeanTok = 64;     // tokens per request and tile
constexpr int kLeanGroup = 32;   // steps whose terms are read ahead at a time
constexpr int kLeanStride = 16;  // steps between two states that are left for the writer
constexpr int kLeanStates = kLeanTok / kLeanStride;
constexpr int kLeanLoaders = 2;
constexpr uint32_t kLeanWriter = 1 + kLeanLoaders;
constexpr int kLeanThreads = 64 * (2 + kLeanLoaders);
// Offsets from kLeanOutside on lie outside every buffer: a load there fetches nothing.
constexpr uint32_t kLeanBufferMost = 0xFFFFFF00u, kLeanOutside = 0xFFFFFFF0u;

// One request as every wave of its workgroup sees it: lane i of a wave knows request i % 16.
struct LeanRow {
    int64_t start;  // first token
    int64_t ntok;   // tokens that make up keys
    int64_t key;    // index of its first key
};

__device__ __forceinline__ int64_t shfl_i64(int64_t v, int lane) {
    const int lo = __shfl(static_cast<int>(v), lane, 64), hi = __shfl(static_cast<int>(v >> 32), lane, 64);
    return static_cast<int64_t>((static_cast<uint64_t>(static_cast<uint32_t>(hi)) << 32) | static_cast<uint32_t>(lo));
}

// For values that are the same in all lanes where the compiler cannot see it: scalar registers, scalar branches.
__device__ __forceinline__ int64_t uniform_i64(int64_t v) {
    const uint32_t lo = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(v));
    const uint32_t hi = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(static_cast<uint64_t>(v) >> 32));
    return static_cast<int64_t>((static_cast<uint64_t>(hi) << 32) | lo);
}

// One tile in 16-byte buffer loads. A piece behind its request's last token is not fetched.
template <typename TokT>
struct LeanBufferLoader {
    static constexpr int kEPL = 16 / sizeof(TokT);
    static constexpr int kLPR = kLeanTok / kEPL;       // lanes per request row
    static constexpr int kRPW = 64 / kLPR;             // rows per load instruction
    static constexpr int kNL = kLeanRows / kRPW;       // loads per lane and tile
    typedef u32x4 Regs[kNL];
    __amdgpu_buffer_rsrc_t rsrc;
    uint32_t rel[kNL], lim[kNL];  // byte offset of this lane's piece of tile 0; bytes of the request from that piece on
    uint32_t sub, piece;

    __device__ __forceinline__ void setup(const TokT *tokens, int64_t first, int64_t total, const LeanRow &row, uint32_t lane) {
        sub = lane / kLPR;
        piece = lane % kLPR;
        const uint64_t bytes = static_cast<uint64_t>(total - first) * sizeof(TokT);
        rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<TokT *>(tokens + first), 0,
                                                 bytes > kLeanBufferMost ? kLeanBufferMost : static_cast<uint32_t>(bytes), 0x00020000);
        const int at = static_cast<int>((row.start - first) * static_cast<int64_t>(sizeof(TokT)));
        const int len = static_cast<int>(row.ntok * static_cast<int64_t>(sizeof(TokT)));
#pragma unroll
        for (int j = 0; j < kNL; ++j) {
            const int from = j * kRPW + static_cast<int>(sub);
            const uint32_t bytes_of_row = static_cast<uint32_t>(__shfl(len, from, 64));
            rel[j] = static_cast<uint32_t>(__shfl(at, from, 64)) + piece * 16u;
            lim[j] = bytes_of_row > piece * 16u ? bytes_of_row - piece * 16u : 0;
        }
    }
    __device__ __forceinline__ void issue(Regs &regs, int32_t t) const {
        const uint32_t off = static_cast<uint32_t>(t) * static_cast<uint32_t>(kLeanTok * sizeof(TokT));
#pragma unroll
        for (int j = 0; j < kNL; ++j) {
            regs[j] = __builtin_amdgcn_raw_buffer_load_b128(rsrc, off < lim[j] ? rel[j] + off : kLeanOutside, 0, 2);
        }
    }
    __device__ __forceinline__ void store(const Regs &regs, uint64_t (*tile)[kLeanTok + kPad]) const {
#pragma unroll
        for (int j = 0; j < kNL; ++j) {
            const u32x4 v = regs[j];
            ulonglong2 *dst = reinterpret_cast<ulonglong2 *>(&tile[j * kRPW + sub][piece * kEPL]);
            if (sizeof(TokT) == 8) {
                dst[0] = make_ulonglong2(((static_cast<uint64_t>(v.y) << 32) | v.x) + kGolden,
                                         ((static_cast<uint64_t>(v.w) << 32) | v.z) + kGolden);
            } else {
                dst[0] = make_ulonglong2(pre_add_i32(v.x), pre_add_i32(v.y));
                dst[1] = make_ulonglong2(pre_add_i32(v.z), pre_add_i32(v.w));
            }
        }
    }
};

// The same with an address per token, for workgroups with a request that a buffer offset does not reach.
template <typename TokT>
struct LeanGlobalLoader {
    static_assert(kLeanTok == 64, "a lane per token of a request's row");
    typedef TokT Regs[kLeanRows];
    const TokT *tokens;
    LeanRow row;
    uint32_t lane;
    __device__ __forceinline__ void setup(const TokT *tokens_, int64_t, int64_t, const LeanRow &row_, uint32_t lane_) {
        tokens = tokens_;
        row = row_;
        lane = lane_;
    }
    __device__ __forceinline__ void issue(Regs &regs, int32_t t) const {
        const int64_t at = static_cast<int64_t>(t) * kLeanTok + lane;
#pragma unroll
        for (int j = 0; j < kLeanRows; ++j) {
            const int64_t ntok = shfl_i64(row.ntok, j), start = shfl_i64(row.start, j);  // while all lanes are here
            regs[j] = at < ntok ? tokens[start + at] : 0;
        }
    }
    __device__ __forceinline__ void store(const Regs &regs, uint64_t (*tile)[kLeanTok + kPad]) const {
#pragma unroll
        for (int j = 0; j < kLeanRows; ++j) {
            tile[j][lane] = static_cast<uint64_t>(static_cast<int64_t>(regs[j])) + kGolden;
        }
    }
};

template <bool EVERY>
struct LeanShared {
    static constexpr int kRing = EVERY ? 8 : 2;
    uint64_t tile[kRing][kLeanRows][kLeanTok + kPad];  // terms; EVERY: then the states after every step
    uint64_t state[4][kLeanRows][kLeanStates + 2];     // states after every 16 steps, of four tiles
    KeyRow keyrow[kLeanRows];                          // the writer's own
};

// Who does what when. Barrier b ends interval b; there are nt + 2 of them, EVERY: nt + 3.
//   loader      stores tile t in interval t (its slot was read for the last time in interval t - 1 or before)
//   chain wave  reads the rest of tile t and goes through it in intervals t + 1 and t + 2: its barrier stands in front of the
//               tile's last 32 steps, when the last terms are in registers and those of the next tile are about to be asked for;
//               the tile's last states are written in interval t + 2
//   EVERY       loader t % 2 expands tile t in interval t + 3 (tile t + 3 is the other one's)
//   writer      stores the keys of tile t in interval t + 3, EVERY: t + 4 (tile t + 8 takes its slot, tile t + 4 its states)

// The states after every token of tile t, in place of the tile's terms: 64 lanes go through 16 steps each, from the states
// that the chain wave left.
__device__ __forceinline__ void lean_expand(LeanShared<true> &sh, int32_t t, uint64_t seed, uint32_t lane) {
    using SH = LeanShared<true>;
    static_assert(kLeanRows * kLeanStates == 64, "a lane per stretch of 16 steps");
    const uint32_t r = lane % kLeanRows, part = lane / kLeanRows;
    uint64_t h = part ? sh.state[t & 3][r][part - 1] : t ? sh.state[(t - 1) & 3][r][kLeanStates - 1] : seed;
    ulonglong2 *const terms = reinterpret_cast<ulonglong2 *>(&sh.tile[t & (SH::kRing - 1)][r][part * kLeanStride]);
    ulonglong2 a[kLeanStride / 2];
#pragma unroll
    for (int i = 0; i < kLeanStride / 2; ++i) {
        a[i] = terms[i];
    }
#pragma unroll
    for (int i = 0; i < kLeanStride / 2; ++i) {
        const uint64_t h1 = chain_step(h, a[i].x);
        h = chain_step(h1, a[i].y);
        terms[i] = make_ulonglong2(h1, h);
    }
}

// A loader wave's whole life: tiles me, me + 2, ..., in two register sets taking turns.
template <typename Loader, bool EVERY>
__device__ __forceinline__ void lean_load(LeanShared<EVERY> &sh, const Loader &ld, int32_t me, int32_t nt, uint64_t seed,
                                          uint32_t lane) {
    constexpr int32_t kAhead = 2 * kLeanLoaders;
    typename Loader::Regs even, odd;
    int32_t barriers = nt + (EVERY ? 3 : 2);
    const auto barrier = [&] {
        if (barriers > 0) {
            lds_barrier();
            --barriers;
        }
    };
    const auto turn = [&](typename Loader::Regs &regs, int32_t t) {
        if (t < nt) {
            ld.store(regs, sh.tile[t & (LeanShared<EVERY>::kRing - 1)]);
        }
        // also beyond the last tile, where nothing is fetched: how many loads are under way is then known when the code is
        // written, and a tile is waited for without the one behind it
        ld.issue(regs, t + kAhead);
        barrier();
        if constexpr (EVERY) {  // the other loader's turn: its tile is t + 1
            if (t >= 2 && t - 2 < nt) {
                lean_expand(sh, t - 2, seed, lane);
            }
        }
        barrier();
    };
    ld.issue(even, me);
    ld.issue(odd, me + kLeanLoaders);
    if (me) {
        barrier();
    }
    for (int32_t t = me; barriers > 0; t += kAhead) {
        turn(even, t);
        turn(odd, t + kLeanLoaders);
    }
}

// The writer's whole life. Keys lie `per` states apart (of those that are kept: every 16th step's, EVERY: every step's).
template <bool EVERY>
__device__ __forceinline__ void lean_write(LeanShared<EVERY> &sh, int32_t nt, const LeanRow &row, int64_t count, int32_t block_size,
                                           int64_t *__restrict__ keys, uint32_t lane) {
    constexpr uint32_t kUnit = EVERY ? 1 : kLeanStride, kUnits = kLeanTok / kUnit;  // states per tile
    const uint32_t per = static_cast<uint32_t>(block_size) / kUnit;
    const uint32_t q = kUnits / per;
    const uint32_t most = q * per == kUnits ? q : q + 1;              // keys per tile
    const uint32_t lg = most > 1 ? 32 - __builtin_clz(most - 1) : 0;  // log2 of the lanes that a request's keys take
    int64_t before = 0;                                               // keys of the tiles so far
    uint32_t off = per;                                               // states to the next key
    if (lane < kLeanRows) {
        sh.keyrow[lane] = KeyRow{row.key, count};
    }
    lds_barrier();
    lds_barrier();
    if (EVERY) {
        lds_barrier();
    }
    for (int32_t t = 0; t < nt; ++t) {
        lds_barrier();
        uint64_t(*const tile)[kLeanTok + kPad] = sh.tile[t & (LeanShared<EVERY>::kRing - 1)];
        const uint32_t nk = off > kUnits ? 0 : off + q * per <= kUnits ? q + 1 : q;
        for (uint32_t e = lane; e < static_cast<uint32_t>(kLeanRows) << lg; e += 64) {
            const uint32_t r = e >> lg, j = e & ((1u << lg) - 1);
            const KeyRow to = sh.keyrow[r];
            if (j < nk && before + j < to.count) {
                const uint32_t at = off - 1 + j * per;
                keys[to.first + before + j] = static_cast<int64_t>(EVERY ? tile[r][at] : sh.state[t & 3][r][at]);
            }
        }
        before += nk;
        off += nk * per - kUnits;
    }
}

// Keys of the requests [base, base + kAhead * 128) in front of r_first, a pair of requests per lane and load.
template <int kAhead>
__device__ __forceinline__ int64_t lean_keys_of(const int64_t *__restrict__ token_offsets, int64_t base, int64_t r_first,
                                                int32_t block_size, const Extent &have, const FastDiv by_block, uint32_t lane,
                                                bool &bad) {
    typedef uint64_t u64x2 __attribute__((ext_vector_type(2)));
    typedef u64x2 u64x2_a8 __attribute__((aligned(8)));
    static_assert(kLeanRows % 2 == 0, "lanes take requests in pairs");
    u64x2 from[kAhead];
    uint64_t to[kAhead];
#pragma unroll
    for (int j = 0; j < kAhead; ++j) {
        const int64_t i = base + j * 128 + lane * 2;
        from[j] = u64x2{0, 0};
        to[j] = 0;
        if (i < r_first) {
            from[j] = *reinterpret_cast<const u64x2_a8 *>(token_offsets + i);
            to[j] = static_cast<uint64_t>(token_offsets[i + 2]);
        }
    }
    bool odd = false;  // beyond the tokens or longer than the short division takes: looked at again, one by one
    int64_t sum = 0;
#pragma unroll
    for (int j = 0; j < kAhead; ++j) {
        const uint64_t len0 = from[j].y - from[j].x, len1 = to[j] - from[j].y;
        odd |= to[j] > static_cast<uint64_t>(have.tokens) || from[j].y > to[j] || from[j].x > from[j].y || (len0 | len1) >> 31 != 0;
        sum += fast_div(static_cast<uint32_t>(len0), by_block) + fast_div(static_cast<uint32_t>(len1), by_block);
    }
    if (__ballot(odd) != 0) {
        sum = 0;
        for (int j = 0; j < kAhead; ++j) {
            const int64_t i = base + j * 128 + lane * 2;
            for (int64_t k = i; k < i + 2 && k < r_first; ++k) {
                sum += keys_of_request(token_offsets[k], token_offsets[k + 1], block_size, have.tokens, bad);
            }
        }
    }
    return sum;
}

// Keys of all requests in front of a workgroup, added up by its writer wave while the loaders wait for their first tokens, so that
// no launch has to make the offsets first and nobody waits for another workgroup. Bound by trips to the caches, for the offsets and,
// with few requests, for the instructions: 2048 requests unrolled, whatever their number, cost 1 us more at 30 to 1000 of them.
// us a call that waits for the total, a launch for the offsets in front / here: 160 requests of 48 to 8192 4-byte tokens 94.2 / 90.9,
// 4 of 162 to 1296 20.7 / 17.6, 1500 of 700 to 1400 23.2 / 19.8, 4096 of 500 to 4096 in blocks of 24 55.1 / 51.2.
__device__ __forceinline__ int64_t lean_keys_before(const int64_t *__restrict__ token_offsets, int64_t r_first, int32_t block_size,
                                                    const Extent &have, const FastDiv by_block, uint32_t lane, bool &bad) {
    constexpr int kMany = 8, kFew = 2;
    int64_t before = 0, base = 0;
    for (; r_first - base > kMany * 64; base += kMany * 128) {
        before += lean_keys_of<kMany>(token_offsets, base, r_first, block_size, have, by_block, lane, bad);
    }
    for (; base < r_first; base += kFew * 128) {
        before += lean_keys_of<kFew>(token_offsets, base, r_first, block_size, have, by_block, lane, bad);
    }
    return before;
}

// The key offsets of a workgroup's requests, and of the last one the total. before: this lane's share of the keys in front. (4096
// requests of kMostKeys at most: no sum needs bringing down before the end.)
__device__ __forceinline__ void lean_key_offsets(int64_t r_first, int32_t R, int64_t before, int64_t own, bool bad_before, bool bad,
                                                 const Extent &have, const CountOut &out, uint32_t lane, LeanRow &row, int64_t &count) {
    const int64_t r = r_first + lane;
    const bool mine = lane < kLeanRows && r < R;
    own = mine ? own : 0;
    int64_t incl = own;
    for (int d = 1; d < 64; d <<= 1) {
        const int64_t up = __shfl_up(incl, d, 64);
        incl += static_cast<int>(lane) >= d ? up : 0;
        before += __shfl_xor(before, d, 64);
    }
    const int64_t key = before + incl - own, total = at_most_all_keys(key + own);
    const bool any = __ballot(bad_before || (mine && bad)) != 0;
    // without its tokens, or beyond the room the caller has: marked, and left out
    const bool fits = !bad && keys_fit(key, own, have.keys);
    if (mine) {
        out.key_offsets[r] = fits ? key : -1;
        if (r == R - 1) {
            out.key_offsets[R] = total;
            // relaxed: whoever waits for it reads nothing else by it (a release writes the whole L2 back first)
            __hip_atomic_store(out.h_total, any ? -1 : total, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        }
    }
    // every lane knows request lane % 16
    row.key = shfl_i64(key, lane % kLeanRows);
    const int64_t n = shfl_i64(fits ? own : 0, lane % kLeanRows);
    count = row.ntok > 0 ? n : 0;
}

// The same for block size 1, where every state is a key: 512 bytes of a request at a time, 16 per lane.
__device__ __forceinline__ void lean_write_all(LeanShared<true> &sh, int32_t nt, const LeanRow &row, int64_t count,
                                               int64_t *__restrict__ keys, uint32_t lane) {
    typedef uint64_t u64x2 __attribute__((ext_vector_type(2)));
    typedef u64x2 u64x2_a8 __attribute__((aligned(8)));
    constexpr int kN = kLeanRows / 2;  // two requests' rows per store instruction
    const uint32_t half = lane / 32, piece = lane % 32;
    int64_t *dst[kN];
    int32_t pairs[kN], singles[kN];  // tiles in which both of this lane's keys, or the first, belong to the request
#pragma unroll
    for (int i = 0; i < kN; ++i) {
        const int64_t left = shfl_i64(count, i * 2 + half) - piece * 2;
        dst[i] = keys + shfl_i64(row.key, i * 2 + half) + piece * 2;
        pairs[i] = left >= 2 ? static_cast<int32_t>((left - 2) / kLeanTok + 1) : 0;
        singles[i] = left >= 1 ? static_cast<int32_t>((left - 1) / kLeanTok + 1) : 0;
    }
    // tiles that all 16 requests fill
    const int32_t full = static_cast<int32_t>(wave_min_u32(static_cast<uint32_t>(count / kLeanTok)));
    lds_barrier();
    lds_barrier();
    lds_barrier();
    for (int32_t t = 0; t < nt; ++t) {
        lds_barrier();
        const uint64_t(*const tile)[kLeanTok + kPad] = sh.tile[t & (LeanShared<true>::kRing - 1)];
        u64x2 v[kN];
#pragma unroll
        for (int i = 0; i < kN; ++i) {
            v[i] = *reinterpret_cast<const u64x2 *>(&tile[i * 2 + half][piece * 2]);
        }
        if (t < full) {
#pragma unroll
            for (int i = 0; i < kN; ++i) {
                *reinterpret_cast<u64x2_a8 *>(dst[i]) = v[i];
            }
        } else {
#pragma unroll
            for (int i = 0; i < kN; ++i) {
                if (t < pairs[i]) {
                    *reinterpret_cast<u64x2_a8 *>(dst[i]) = v[i];
                } else if (t < singles[i]) {
                    *dst[i] = static_cast<int64_t>(v[i].x);
                }
            }
        }
#pragma unroll
        for (int i = 0; i < kN; ++i) {
            dst[i] += kLeanTok;
        }
    }
}

template <typename TokT, bool EVERY>
__global__ __launch_bounds__(kLeanThreads) void hash_lean_kernel(const TokT *__restrict__ tokens,
                                                                 const int64_t *__restrict__ token_offsets, int32_t R,
                                                                 int32_t block_size, uint64_t seed, int64_t *__restrict__ keys,
                                                                 const int64_t *__restrict__ key_offsets, const Uniform uni,
                                                                 const Extent have, const CountOut out, int32_t force_global_loads) {
    using SH = LeanShared<EVERY>;
    __shared__ __attribute__((aligned(16))) SH sh;
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int64_t r_first = static_cast<int64_t>(blockIdx.x) * kLeanRows;
    const int64_t r = r_first + lane % kLeanRows;
    LeanRow row{0, 0, 0};
    int64_t count = 0, first = 0, total;
    int32_t nt;  // tiles of the longest request
    if (token_offsets) {
        const bool known = have.tokens != kUnknown;
        total = known ? have.tokens : token_offsets[R];
        if (!within_reach<TokT>(total)) {
            first = token_offsets[r_first];
            if (known && (first < 0 || first > total)) {
                first = first < 0 ? 0 : total;
            }
        }
        const int64_t at = token_offsets[r < R ? r : R], next = token_offsets[r < R ? r + 1 : R];
        const bool counts = out.key_offsets && wave == kLeanWriter;
        int64_t before = 0;
        bool bad_before = false;
        if (counts) {
            before = lean_keys_before(token_offsets, r_first, block_size, have, out.by_block, lane, bad_before);
        }
        const int64_t nkeys = keys_of(distance(at, next), block_size);
        const bool there = !known || inside(at, nkeys * block_size, total);
        // where the keys go is the writer's business alone if this launch counts them
        row.key = out.key_offsets ? 0 : key_offsets ? key_offsets[r < R ? r : 0]
                                                    : r * keys_of(distance(token_offsets[0], token_offsets[1]), block_size);
        if (r < R && (out.key_offsets || inside(row.key, nkeys, have.keys)) && there) {
            row.start = at;
            row.ntok = nkeys * block_size;
            count = nkeys;
        }
        nt = static_cast<int32_t>(wave_max_u32(static_cast<uint32_t>((row.ntok + kLeanTok - 1) / kLeanTok)));
        if (counts) {
            lean_key_offsets(r_first, R, before, nkeys, bad_before, nkeys > 0 && !there, have, out, lane, row, count);
        }
    } else {
        total = R * uni.tokens;
        first = within_reach<TokT>(total) ? 0 : r_first * uni.tokens;
        if (r < R) {
            row.start = r * uni.tokens;
            row.key = key_offsets ? key_offsets[r] : r * uni.keys;
            count = row.key < 0 ? 0 : uni.keys;
            row.ntok = count * block_size;
        }
        nt = static_cast<int32_t>((uni.keys * block_size + kLeanTok - 1) / kLeanTok);
        if (key_offsets && __ballot(count > 0) == 0) {
            nt = 0;  // the caller wants no keys of any of them
        }
        if (uni.key_offsets_out && wave == kLeanWriter) {
            if (lane < kLeanRows && r < R) {
                uni.key_offsets_out[r] = r * uni.keys;
            }
            if (r_first + kLeanRows >= R && lane == 0) {
                uni.key_offsets_out[R] = R * uni.keys;
            }
        }
    }
    nt = __builtin_amdgcn_readfirstlane(nt);
    if (nt == 0) {
        return;
    }
    first = uniform_i64(first);
    total = uniform_i64(total);
    if (wave == kLeanWriter) {
        if constexpr (EVERY) {
            if (block_size == 1) {
                lean_write_all(sh, nt, row, count, keys, lane);
                return;
            }
        }
        lean_write<EVERY>(sh, nt, row, count, block_size, keys, lane);
        return;
    }
    if (wave != 0) {
        const bool buffer_loads = within_reach<TokT>(total) || __ballot(out_of_reach<TokT>(row.start, row.ntok, first)) == 0;
        if (buffer_loads && !force_global_loads) {
            LeanBufferLoader<TokT> ld;
            ld.setup(tokens, first, total, row, lane);
            lean_load<LeanBufferLoader<TokT>, EVERY>(sh, ld, wave - 1, nt, seed, lane);
        } else {
            LeanGlobalLoader<TokT> ld;
            ld.setup(tokens, first, total, row, lane);
            lean_load<LeanGlobalLoader<TokT>, EVERY>(sh, ld, wave - 1, nt, seed, lane);
        }
        return;
    }
    constexpr int kPieces = kLeanGroup / 2, NG = kLeanTok / kLeanGroup;
    static_assert(NG % 2 == 0 && kLeanGroup == 2 * kLeanStride, "register sets take turns; two states per group, one write");
    const uint32_t mine = lane % kLeanRows;
    uint64_t h = seed, held = 0;
    ulonglong2 a[2][kPieces];
    const auto read_group = [&](ulonglong2 (&to)[kPieces], const uint64_t *from) {
#pragma unroll
        for (int i = 0; i < kPieces; ++i) {
            to[i] = reinterpret_cast<const ulonglong2 *>(from)[i];
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    lds_barrier();
    read_group(a[0], &sh.tile[0][mine][0]);
    // A step is 32 bytes of code, and where the loop begins within 32 bytes decides up to 1 % (64 x 4096 8-byte tokens 47.1 us at byte
    // 8 or 12, 47.6 at 28). This, in front of the first tile, which the compiler takes out of the loop, puts it at 8, and at 16 where
    // EVERY state is kept (48.9 to 49.2), whatever the code above takes.
    asm volatile(".p2align 6\n\ts_nop 0\n\ts_nop 0\n\ts_nop 0");
    uint64_t *at = nullptr;  // where the states of the group before go
    for (int32_t k = 0; k < nt; ++k) {
        const uint64_t *const row_now = &sh.tile[k & (SH::kRing - 1)][mine][0], *const row_next = &sh.tile[(k + 1) & (SH::kRing - 1)][mine][0];
        uint64_t *const states = &sh.state[k & 3][mine][0];
#pragma unroll
        for (int g = 0; g < NG; ++g) {
            // This group's terms, asked for 32 steps ago. Waited for before the next are asked for: the counter of LDS operations
            // ends at 15, so behind 16 newer reads the wait would be for the first of those.
            __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
            if (g + 1 == NG) {
                lds_barrier();
            }
            if (g > 0 || k > 0) {
                *reinterpret_cast<ulonglong2 *>(at) = make_ulonglong2(held, h);
            }
            at = states + 2 * g;
            read_group(a[(g + 1) & 1], g + 1 < NG ? row_now + (g + 1) * kLeanGroup : row_next);  // behind the last tile: not used
#pragma unroll
            for (int s = 0; s < kLeanGroup; ++s) {
                const ulonglong2 v = a[g & 1][s / 2];
                h = chain_step(h, (s & 1) ? v.y : v.x);
                if (s == kLeanStride - 1) {
                    held = h;
                }
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    *reinterpret_cast<ulonglong2 *>(at) = make_ulonglong2(held, h);
    lds_barrier();
    if (EVERY) {
        lds_barrier();
    }
}

// sums[g] = keys of the requests of workgroup g of key_offsets_kernel, as its complement if one of them is bad
__global__ __launch_bounds__(kOffsetsThreads) void key_sums_kernel(const int64_t *__restrict__ token_offsets, int32_t R,
                                                                   int32_t block_size, int64_t n_tokens,
                                                                   int64_t *__restrict__ sums) {
    __shared__ int64_t s_sum[kOffsetsThreads / 64];
    __shared__ int32_t s_bad[kOffsetsThreads / 64];
    const int64_t base = blockIdx.x * kOffsetsPerWg;
    const int64_t end = base + kOffsetsPerWg < R ? base + kOffsetsPerWg : R;
    int64_t sum = 0;
    bool bad = false;
#pragma unroll 8
    for (int64_t i = base + threadIdx.x; i < end; i += kOffsetsThreads) {
        sum += keys_of_request(token_offsets[i], token_offsets[i + 1], block_size, n_tokens, bad);
    }
    for (int d = 1; d < 64; d <<= 1) {
        sum += __shfl_xor(sum, d, 64);
    }
    const bool any = __ballot(bad) != 0;
    if ((threadIdx.x & 63) == 0) {
        s_sum[threadIdx.x >> 6] = sum;
        s_bad[threadIdx.x >> 6] = any;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        int64_t all = 0;
        bool some = false;
        for (int w = 0; w < kOffsetsThreads / 64; ++w) {
            all += s_sum[w];
            some |= s_bad[w] != 0;
        }
        all = at_most_all_keys(all);
        sums[blockIdx.x] = some ? ~all : all;
    }
}

__global__ __launch_bounds__(kOffsetsThreads) void key_offsets_kernel(const int64_t *__restrict__ token_offsets, int32_t R,
                                                                      int32_t block_size, int64_t n_tokens, int64_t limit,
                                                                      const int64_t *__restrict__ sums,
                                                                      int64_t *__restrict__ key_offsets, int64_t *h_total) {
    __shared__ int64_t s_wave[2][kOffsetsThreads / 64];
    __shared__ int32_t s_bad[kOffsetsThreads / 64];
    const int32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6, waves = blockDim.x >> 6;
    const int64_t base = blockIdx.x * kOffsetsPerWg;
    int64_t before = 0;
    bool bad = false;
    if (sums) {
        for (int64_t g = threadIdx.x; g < static_cast<int64_t>(blockIdx.x); g += blockDim.x) {
            const int64_t v = sums[g];
            bad |= v < 0;
            before += v < 0 ? ~v : v;
        }
    } else {
        for (int64_t i = threadIdx.x; i < base; i += blockDim.x) {
            before += keys_of_request(token_offsets[i], token_offsets[i + 1], block_size, n_tokens, bad);
        }
    }
    before = at_most_all_keys(before);
    const int64_t first = base + static_cast<int64_t>(threadIdx.x) * kOffsetsPerThread;
    int64_t off[kOffsetsPerThread + 1];
#pragma unroll
    for (int j = 0; j <= kOffsetsPerThread; ++j) {
        off[j] = token_offsets[first + j < R ? first + j : R];
    }
    int64_t count[kOffsetsPerThread], sum = 0;
    uint32_t left_out = 0;
#pragma unroll
    for (int j = 0; j < kOffsetsPerThread; ++j) {
        bool mine = false;
        count[j] = keys_of_request(off[j], off[j + 1], block_size, n_tokens, mine);
        left_out |= mine ? 1u << j : 0u;
        sum += count[j];
    }
    bad |= left_out != 0;
    int64_t incl = sum;
    for (int d = 1; d < 64; d <<= 1) {
        const int64_t up = __shfl_up(incl, d, 64);
        incl += lane >= d ? up : 0;
        before += __shfl_xor(before, d, 64);
    }
    const bool any = __ballot(bad) != 0;
    if (lane == 63) {
        s_wave[0][wave] = incl;
        s_wave[1][wave] = before;
        s_bad[wave] = any;
    }
    __syncthreads();
    int64_t pos = incl - sum;
    bool some = false;
    for (int w = 0; w < waves; ++w) {
        pos += (w < wave ? s_wave[0][w] : 0) + s_wave[1][w];
        some |= s_bad[w] != 0;
    }
#pragma unroll
    for (int j = 0; j < kOffsetsPerThread; ++j) {
        if (first + j < R) {
            // without its tokens, or beyond the room the caller has: marked, and the hash kernel leaves the request out
            key_offsets[first + j] = keys_fit(pos, count[j], limit) && !(left_out >> j & 1) ? pos : -1;
            pos += count[j];
            if (first + j == R - 1) {
                pos = at_most_all_keys(pos);
                key_offsets[R] = pos;
                if (h_total) {  // the last workgroup has seen every request
                    __hip_atomic_store(h_total, some ? -1 : pos, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
                }
            }
        }
    }
}

// ------------------------------------------------------------------------------------------- SHA-256

__constant__ uint32_t kShaK[64] = {
    0x428a2f98, 0x71374491, 0xb5c0fbcf, 0xe9b5dba5, 0x3956c25b, 0x59f111f1, 0x923f82a4, 0xab1c5ed5,
    0xd807aa98, 0x12835b01, 0x243185be, 0x550c7dc3, 0x72be5d74, 0x80deb1fe, 0x9bdc06a7, 0xc19bf174,
    0xe49b69c1, 0xefbe4786, 0x0fc19dc6, 0x240ca1cc, 0x2de92c6f, 0x4a7484aa, 0x5cb0a9dc, 0x76f988da,
    0x983e5152, 0xa831c66d, 0xb00327c8, 0xbf597fc7, 0xc6e00bf3, 0xd5a79147, 0x06ca6351, 0x14292967,
    0x27b70a85, 0x2e1b2138, 0x4d2c6dfc, 0x53380d13, 0x650a7354, 0x766a0abb, 0x81c2c92e, 0x92722c85,
    0xa2bfe8a1, 0xa81a664b, 0xc24b8b70, 0xc76c51a3, 0xd192e819, 0xd6990624, 0xf40e3585, 0x106aa070,
    0x19a4c116, 0x1e376c08, 0x2748774c, 0x34b0bcb5, 0x391c0cb3, 0x4ed8aa4a, 0x5b9cca4f, 0x682e6ff3,
    0x748f82ee, 0x78a5636f, 0x84c87814, 0x8cc70208, 0x90befffa, 0xa4506ceb, 0xbef9a3f7, 0xc67178f2};

__device__ __forceinline__ uint32_t rotr(uint32_t x, int n) { return __builtin_amdgcn_alignbit(x, x, n); }
__device__ __forceinline__ uint32_t xor3(uint32_t x, uint32_t y, uint32_t z) { return __builtin_amdgcn_bitop3_b32(x, y, z, 0x96); }

// One FIPS 180-4 compression; w holds the 16 big-endian message words and is used as the rolling schedule.
__device__ void sha256_compress(uint32_t (&st)[8], uint32_t (&w)[16]) {
    uint32_t a = st[0], b = st[1], c = st[2], d = st[3], e = st[4], f = st[5], g = st[6], h = st[7];
#pragma unroll
    for (int i = 0; i < 64; ++i) {
        if (i >= 16) {
            const uint32_t w15 = w[(i + 1) & 15], w2 = w[(i + 14) & 15];
            const uint32_t s0 = xor3(rotr(w15, 7), rotr(w15, 18), w15 >> 3);
            const uint32_t s1 = xor3(rotr(w2, 17), rotr(w2, 19), w2 >> 10);
            w[i & 15] = w[i & 15] + s0 + w[(i + 9) & 15] + s1;
        }
        const uint32_t S1 = xor3(rotr(e, 6), rotr(e, 11), rotr(e, 25));
        const uint32_t ch = (e & f) ^ (~e & g);
        const uint32_t t1 = h + S1 + ch + kShaK[i] + w[i & 15];
        const uint32_t S0 = xor3(rotr(a, 2), rotr(a, 13), rotr(a, 22));
        const uint32_t mj = (a & b) ^ (a & c) ^ (b & c);
        const uint32_t t2 = S0 + mj;
        h = g;
        g = f;
        f = e;
        e = d + t1;
        d = c;
        c = b;
        b = a;
        a = t1 + t2;
    }
    st[0] += a;
    st[1] += b;
    st[2] += c;
    st[3] += d;
    st[4] += e;
    st[5] += f;
    st[6] += g;
    st[7] += h;
}

// One lane per string: key = big-endian signed int64 of SHA-256(bytes)[0:8]
// (kv_cache_manager/py_connector/sglang/connector.py:397-401).
// Bound: a compression is 1400 instructions of 4 clocks, one after the other, 2.6 us with what surrounds it, and a string of 64
// characters takes two. What lies in a block is read as words, only the word that holds the message's end byte by byte, and three
// operands are xored at a time. us a launch, before / now: 1024 or 16 384 strings of 64 characters 10.4 / 8.0, of 16: 8.0 / 5.4, 1024 of
// 1 to 200: 32.9 / 20.5. The bytes may lie in pinned host memory: 1024 strings of 64 characters 11.1.
__global__ __launch_bounds__(64) void sha256_first8_kernel(const uint8_t *__restrict__ bytes,
                                                           const int64_t *__restrict__ offsets, int32_t N,
                                                           int64_t *__restrict__ out) {
    // lanes beyond the last string go through it as well: a wave with few active lanes issues more slowly
    const int64_t lane = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x, i = lane < N ? lane : N - 1;
    const uint8_t *msg = bytes + offsets[i];
    const int64_t len = offsets[i + 1] - offsets[i];
    uint32_t st[8] = {0x6a09e667, 0xbb67ae85, 0x3c6ef372, 0xa54ff53a, 0x510e527f, 0x9b05688c, 0x1f83d9ab, 0x5be0cd19};
    const int64_t blocks = (len + 8) / 64 + 1;
    for (int64_t k = 0; k < blocks; ++k) {
        uint32_t w[16];
        const uint8_t *const at = msg + k * 64;
        if (k * 64 + 64 <= len) {
            __builtin_memcpy(w, at, 64);
#pragma unroll
            for (int j = 0; j < 16; ++j) {
                w[j] = __builtin_bswap32(w[j]);
            }
        } else {
            const int32_t left = static_cast<int32_t>(len - k * 64);  // message bytes in this block; below 0 in a block behind its end
            uint32_t end = 0;  // the word behind the whole ones: up to three bytes and the terminating bit
            if (left >= 0) {
                const int32_t n = left & 3;
                const uint8_t *const rest = at + (left - n);
                end = n > 0 ? static_cast<uint32_t>(rest[0]) << 24 : 0;
                end |= n > 1 ? static_cast<uint32_t>(rest[1]) << 16 : 0;
                end |= n > 2 ? static_cast<uint32_t>(rest[2]) << 8 : 0;
                end |= 0x80000000u >> 8 * n;
            }
#pragma unroll
            for (int j = 0; j < 16; ++j) {
                uint32_t v = 0;
                if (4 * j + 4 <= left) {
                    __builtin_memcpy(&v, at + 4 * j, 4);
                }
                w[j] = left >= 0 && left >> 2 == j ? end : __builtin_bswap32(v);
            }
            if (k + 1 == blocks) {
                w[14] = static_cast<uint32_t>(static_cast<uint64_t>(len) >> 29);
                w[15] = static_cast<uint32_t>(len) << 3;
            }
        }
        sha256_compress(st, w);
    }
    if (lane < N) {
        out[i] = static_cast<int64_t>((static_cast<uint64_t>(st[0]) << 32) | st[1]);
    }
}

// ------------------------------------------------------------------------------------------- iov CRC-32

// kv_cache_manager/client/src/internal/sdk/sdk_buffer_check_util.cu:10-19.
__device__ __forceinline__ uint32_t crc32_byte(uint32_t crc, uint8_t data) {
    crc ^= data;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const uint32_t mask = 0u - (crc & 1u);
        crc = (crc >> 1) ^ (0xEDB88320u & mask);
    }
    return crc;
}

// One lane per iov, head bytes then tail bytes through one running CRC (sdk_buffer_check_util.cu:21-44).
__global__ __launch_bounds__(256) void iov_crc32_kernel(const kvcm_iov_device *__restrict__ iovs, int32_t n,
                                                        uint32_t *__restrict__ out, size_t cal_bytes) {
    const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= n) {
        return;
    }
    const uint8_t *p = static_cast<const uint8_t *>(iovs[i].base);
    const size_t size = iovs[i].size;
    if (!p || size < cal_bytes) {
        // cal_bytes comes from the first iov only: an iov without an address, or shorter than that, is not read at
        // all and gets the value 0 (the reference reads out of bounds here). 0 is also a possible CRC, so callers
        // that cannot rule such iovs out check them on the host first, as the C++ and Python layers above do.
        out[i] = 0;
        return;
    }
    uint32_t crc = 0xFFFFFFFFu;
    for (size_t k = 0; k < cal_bytes; ++k) {
        crc = crc32_byte(crc, p[k]);
    }
    for (size_t k = size - cal_bytes; k < size; ++k) {
        crc = crc32_byte(crc, p[k]);
    }
    out[i] = ~crc;
}

// Non-zero makes every launch take the loader path that a workgroup spanning >= 4 GiB of tokens would take. A
// compile-time matter: the shipped library is built with 0 and has no switch; the parity tests build this file a second
// time, with KVCM_TEST_FORCE_GENERAL_LOADER=1, into a library of their own.
#ifndef KVCM_TEST_FORCE_GENERAL_LOADER
#define KVCM_TEST_FORCE_GENERAL_LOADER 0
#endif
constexpr int32_t kForceGeneralLoader = KVCM_TEST_FORCE_GENERAL_LOADER;

// Requests up to which a launch takes workgroups of 16 (hash_lean_kernel): as many as give each of the 256 compute units one. A
// second one on a unit shares its SIMDs, and one of 16 reads 512 bytes of each of 16 requests at a time where the other kernel
// reads 64. us, 16 per workgroup / 64: 4096 requests of 4096 tokens 49.2 / 55.8, 5120: 59.0 / 56.8, 8192: 71.4 / 59.9. The line
// holds for either token width, every block size and short requests too, though a launch of those is few tiles long. us on changing
// tokens, 64 per workgroup (in the form that launch took) / 16:
//                     4096 x 64   x 256      x 1024      x 4096         0..128     0..512      0..2048     512 x 1024
//   bs 1,   8 bytes   6.5/4.9     11.2/8.7   29.0/19.0   99.3/58.2      8.9/6.6    19.9/12.2   58.1/30.7   26.6/15.7
//   bs 16,  8 bytes   5.3/4.3     8.7/7.1    18.6/15.7   56.0/49.3      6.9/5.5    13.8/10.2   37.6/27.1   17.7/14.5
//   bs 128, 8 bytes   -           8.6/7.1    18.3/15.4   51.9/48.8      -          12.6/9.8    30.8/26.0   17.5/14.5
//   bs 1,   4 bytes   5.8/4.7     9.8/7.9    24.9/18.3   85.0/52.9      8.1/6.3    17.1/11.7   51.2/30.3   23.8/15.4
//   bs 16,  4 bytes   4.7/4.0     7.3/6.4    16.2/15.1   50.6/48.7      6.0/5.2    11.2/9.6    30.0/26.4   15.6/14.1
//   bs 128, 4 bytes   -           7.3/6.4    16.1/14.9   50.6/48.1      -          10.4/9.3    27.9/25.5   15.7/14.1
constexpr int32_t kLeanUpTo = 256 * kLeanRows;
static_assert(KVCM_COUNT_KEYS_UP_TO == kLeanUpTo, "only hash_lean_kernel counts keys");

// How keys reach memory in larger launches, by block size, token width and number of requests (hash_tokens_kernel<.., KS>).
// Chosen from timings on tokens that are not in the memory-side cache, us, requests of 4096 tokens each / of 500 to 4096
// (a request that has run out makes the direct form compare per key; the staged forms leave that to the loaders).
//   16-token blocks, 8-byte tokens: direct 4096: 61 / 69  8192: 73 / 77  10 240: 79 / 86
//                                   spread 4096: 60 / 60  8192: 65 / 70
//                                   burst  4096: 60 / 61  8192: 64 / 67  10 240: 68 / 72
//   (up to 8191 spread, whose short workgroups store directly: kSpreadFromTiles)
//   16-token blocks, 4-byte tokens: direct 4096: 55 / -   8192: 58 / 60  12 288: 70 / -
//                                   burst  4096: 58 / -   8192: 58 / 61  12 288: 60 / -      (raw tiles, see below)
// Other block sizes, direct / burst:
//   block size 1, 8-byte tokens   8192: 246 / 115   (a workgroup may still store directly: chain_stays_direct)
//                 4-byte tokens   8192: 174 / 96   16 384 of 128 tokens: 10.8 / 7.1
//   block size 8, 8-byte tokens   4160: 70 / 62   8192: 89 / 69   12 288: 104 / 88
//                 4-byte tokens   8192: 66 / 61 (of 1024 tokens: 20.6 / 23.2)  12 288: 80 / 62
//   block size 32, 8-byte tokens  4096: 59 / 58 (of 1024 tokens: 21.6 / 22.0)  8192: 66 / 61   12 288: 87 / 76
//                  4-byte tokens  8192: 56 / 58   12 288: 67 / 60
//   block size 64, 8-byte tokens  4096: 58 / 57 (of 1024 tokens: 21.6 / 22.0)  8192: 65 / 59   12 288: 79 / 73
//                  4-byte tokens  8192: 55 / 58   12 288: 67 / 60
//   block size 128, 8-byte tokens 4160: 54 / 52 (of 1024 tokens: 18.3 / 18.5)  8192: 64 / 58
//                   4-byte tokens 8192: 55 / 58   12 288: 65 / 59
// Requests from which a launch takes the burst form: all, where it is the better one right behind kLeanUpTo; INT32_MAX = never.
constexpr int32_t burst_from(int32_t block_size, bool tokens_8_byte) {
    switch (block_size) {
        case 1: return 0;
        case 8: return tokens_8_byte ? 0 : 12288;
        case 16: return tokens_8_byte ? 8192 : 12288;
        case 32: return tokens_8_byte ? 8192 : 12288;
        case 64: return tokens_8_byte ? 8192 : 12288;
        case 128: return tokens_8_byte ? 0 : 12288;
        default: return INT32_MAX;
    }
}
// Tokens per request from which such a launch does: the last group leaves after the last token, so staging costs about 1 us
// more than direct stores and has to earn that first. Lengths are known for [R, L] batches, their mean where the caller has
// said how many tokens there are; otherwise requests are taken for long. us, staged / direct, at 8192 requests (4-byte tokens 12 288):
//   equally long        64       256        512        768        1024       1536       2048       4096
//   bs 8,   8 bytes  6.4/5.4  10.1/9.2   13.9/14.2  17.7/19.5  21.0/23.3  29.9/36.9  35.4/43.1  64.5/80.4
//   bs 16,  8 bytes  5.4/4.4   9.5/8.6   13.5/13.1  16.5/17.1  19.2/20.2  27.9/30.8  32.4/35.9  60.0/69.3
//   bs 32,  8 bytes  5.6/4.6   9.5/8.6   13.6/13.0  16.3/16.2  19.4/19.8  26.3/28.3  31.3/34.2  57.9/64.8
//   bs 64,  8 bytes  6.1/5.0   9.5/8.4   13.5/12.8  16.3/16.1  19.2/19.6  26.3/28.0  31.2/33.7  55.8/61.5
//   bs 128, 8 bytes  -         9.8/8.9   13.5/13.0  16.4/16.3  19.2/19.5  26.6/28.2  30.9/33.7  54.0/59.6
//   bs 8,   4 bytes  6.1/4.2   9.1/7.7   12.8/11.4  17.1/15.4  20.9/19.8  27.1/27.1  34.1/35.6  59.3/73.5
//   bs 16,  4 bytes  6.2/4.3   9.0/7.5   12.8/10.9  16.8/14.0  20.1/18.4  26.2/24.6  33.1/33.3  56.8/65.7
//   bs 32,  4 bytes  6.4/4.4   8.9/7.4   12.8/10.8  16.8/13.8  20.4/17.7  26.0/22.9  32.8/32.1  56.4/65.3
//   bs 64,  4 bytes  6.5/4.4   8.9/7.3   12.7/10.6  16.8/13.6  20.4/17.0  26.1/22.5  32.9/31.3  56.0/63.2
//   bs 128, 4 bytes  3.3/3.3   8.9/7.4   12.7/10.5  16.8/13.5  20.2/16.9  25.8/22.3  32.7/30.7  56.1/61.1
//   ragged            16..64   64..512   64..768    64..1024   256..1024  64..2048   512..1536  64..4096   1024..2048 500..4096
//   (mean)              35       215       283        346        554        573        932        969        1477       1710
//   bs 16,  8 bytes  7.9/4.5  14.3/13.0  17.5/17.2  20.6/21.0  20.8/22.7  33.8/36.7  29.2/32.3  61.2/68.1  36.0/42.3  64.9/76.3
//   bs 32,  8 bytes  5.6/4.4  14.5/12.8  17.4/16.4  20.3/19.9  20.6/21.0  31.8/34.2  27.4/29.3  58.6/63.4  34.5/37.7  62.4/68.3
//   bs 64,  8 bytes  5.4/4.3  14.7/12.2  17.9/15.8  20.2/19.1  20.3/19.8  32.0/33.1  26.8/27.5  57.4/61.8  33.8/35.7  60.6/64.8
//   bs 8,   4 bytes  8.6/4.2  14.1/11.8  16.8/15.6  20.6/19.3  21.7/20.2  34.0/33.5  28.3/28.7  59.3/62.0  35.4/37.9  60.2/67.6
//   bs 16,  4 bytes  9.1/4.2  13.9/11.3  17.4/14.6  20.8/17.7  21.5/18.1  33.0/30.6  27.4/25.7  57.2/56.0  33.3/33.7  58.6/60.3
//   bs 32,  4 bytes  6.3/4.4  14.1/11.0  17.7/14.2  20.9/17.3  21.2/17.6  32.3/29.8  27.8/24.3  57.7/54.1  34.0/31.7  58.4/56.7
//   bs 64,  4 bytes  6.1/4.1  15.0/10.6  18.3/13.4  21.0/16.4  21.5/16.8  32.3/28.0  27.5/22.9  55.6/51.6  33.5/29.0  56.5/52.8
//   bs 128, 4 bytes  3.3/3.3  14.2/10.3  17.6/13.0  20.2/16.2  20.7/16.8  32.0/27.5  26.5/22.7  54.7/50.5  32.2/28.6  55.2/51.6
//   ragged            0..128   0..512     0..640     0..768     0..1024    0..1280    0..1792    0..2048    0..4096
//   (mean)              64       256        320        384        512        640        896        1024       2048
//   bs 8,   8 bytes  9.1/7.1  15.5/15.1  17.0/17.9  18.9/20.7  22.9/26.2  26.9/31.7  34.7/42.7  38.7/49.2  71.4/95.8
//   bs 128, 8 bytes  -        15.7/13.1  16.8/14.9  17.4/16.4  20.3/20.1  23.3/23.7  30.0/31.0  33.3/34.6  60.2/63.5
//   Four times as many requests move the lines little (4-byte tokens, 32 768 requests of 2000 to 8192: bs 64 215/248, 128 208/222).
constexpr int64_t burst_from_tokens(int32_t block_size, bool tokens_8_byte, bool equally_long) {
    switch (block_size) {
        case 8: return tokens_8_byte ? (equally_long ? 512 : 320) : equally_long ? 1280 : 640;
        case 16: return tokens_8_byte ? (equally_long ? 640 : 320) : equally_long ? 1792 : 1024;
        case 32: return tokens_8_byte ? (equally_long ? 896 : 560) : equally_long ? 1792 : 1600;
        case 64: return tokens_8_byte ? 896 : 2304;
        case 128: return tokens_8_byte ? 960 : 2560;
        default: return 0;
    }
}

template <typename TokT>
int32_t launch_hash(const TokT *d_tokens, const int64_t *d_token_offsets, int32_t R, int32_t block_size, int64_t seed,
                    int64_t *d_keys, const int64_t *d_key_offsets, hipStream_t stream,
                    const Uniform &uni = Uniform{0, 0, nullptr}, const Extent &have = Extent{kUnknown, kUnknown},
                    const CountOut &out = CountOut{nullptr, nullptr, {0, 0}}) {
    if (R < 0 || block_size <= 0) {
        return KVCM_ERR_INVALID_ARG;
    }
    if (R == 0) {
        return KVCM_OK;
    }
    if (!d_tokens || (!d_token_offsets && uni.keys <= 0) || !d_keys) {
        return KVCM_ERR_INVALID_ARG;
    }
    const dim3 grid(static_cast<uint32_t>((static_cast<int64_t>(R) + kReqs - 1) / kReqs));
    const int32_t force_global = kForceGeneralLoader;
    if (R <= kLeanUpTo) {
        const dim3 lean_grid(static_cast<uint32_t>((static_cast<int64_t>(R) + kLeanRows - 1) / kLeanRows));
        if (block_size % kLeanStride == 0) {
            hipLaunchKernelGGL((hash_lean_kernel<TokT, false>), lean_grid, dim3(kLeanThreads), 0, stream, d_tokens, d_token_offsets, R,
                               block_size, static_cast<uint64_t>(seed), d_keys, d_key_offsets, uni, have, out, force_global);
        } else {
            hipLaunchKernelGGL((hash_lean_kernel<TokT, true>), lean_grid, dim3(kLeanThreads), 0, stream, d_tokens, d_token_offsets, R,
                               block_size, static_cast<uint64_t>(seed), d_keys, d_key_offsets, uni, have, out, force_global);
        }
        return launch_status();
    }
#define KVCM_LAUNCH_HASH(CHUNK, BS)                                                                                  \
    hipLaunchKernelGGL((hash_tokens_kernel<TokT, CHUNK, BS>), grid, dim3(kThreads), 0, stream, d_tokens,            \
                       d_token_offsets, R, block_size, static_cast<uint64_t>(seed), d_keys, d_key_offsets, uni, have, \
                       force_global)
    constexpr bool k8 = sizeof(TokT) == 8;
    const bool many = R >= burst_from(block_size, k8);
    const int64_t tokens_per_request = !d_token_offsets ? uni.tokens : have.tokens == kUnknown ? kUnknown : have.tokens / R;
    const bool burst = many && tokens_per_request >= burst_from_tokens(block_size, k8, !d_token_offsets);
    const bool spread = block_size == 16 && k8 && !many;
#define KVCM_LAUNCH_HASH_STAGED(CHUNK, BS, KS)                                                                       \
    hipLaunchKernelGGL((hash_tokens_kernel<TokT, CHUNK, BS, KS>), grid, dim3(kThreads), 0, stream, d_tokens,        \
                       d_token_offsets, R, block_size, static_cast<uint64_t>(seed), d_keys, d_key_offsets, uni, have, \
                       force_global)
    // 4-byte tokens from as many requests as take the burst form: tiles of 128 raw tokens (512-byte pieces of the
    // token stream per request and load instruction instead of 256-byte ones). Cold timings, 16-token blocks, requests
    // of 4096 tokens, 64-token tiles of pre-added terms / raw tiles: 8192 requests 58.1 / 60.2 us,
    // 12 288 66.6 / 62.2, 16 384 77.3 / 66.4, 32 768 149 / 127.
    const bool raw = !k8 && burst && (block_size == 8 || block_size == 16 || block_size == 32 || block_size == 64 ||
                                      block_size == 128);
#define KVCM_LAUNCH_HASH_RAW(BS)                                                                                      \
    hipLaunchKernelGGL((hash_tokens_kernel<TokT, 8, BS, kKeysBurst, true>), grid, dim3(kThreads), 0, stream, d_tokens, \
                       d_token_offsets, R, block_size, static_cast<uint64_t>(seed), d_keys, d_key_offsets, uni, have, \
                       force_global)
    if (raw) {
        if constexpr (!k8) {
            switch (block_size) {
                case 8: KVCM_LAUNCH_HASH_RAW(8); break;
                case 16: KVCM_LAUNCH_HASH_RAW(16); break;
                case 32: KVCM_LAUNCH_HASH_RAW(32); break;
                case 64: KVCM_LAUNCH_HASH_RAW(64); break;
                default: KVCM_LAUNCH_HASH_RAW(128); break;
            }
        }
    } else if (spread) {
        if constexpr (k8) {
            KVCM_LAUNCH_HASH_STAGED(8, 16, kKeysSpread);
        }
    } else if (block_size == 16) {  // the engines' usual block sizes get kernels of their own
        if (k8 && burst) {  // 4-byte tokens take the burst form with raw tiles, above
            if constexpr (k8) {
                KVCM_LAUNCH_HASH_STAGED(8, 16, kKeysBurst);
            }
        } else {
            KVCM_LAUNCH_HASH(8, 16);
        }
    } else if (block_size == 8) {
        if (k8 && burst) {  // 4-byte tokens take the burst form with raw tiles, above
            if constexpr (k8) {
                KVCM_LAUNCH_HASH_STAGED(8, 8, kKeysBurst);
            }
        } else {
            KVCM_LAUNCH_HASH(8, 8);
        }
    } else if (block_size == 32) {
        if (k8 && burst) {  // 4-byte tokens take the burst form with raw tiles, above
            if constexpr (k8) {
                KVCM_LAUNCH_HASH_STAGED(8, 32, kKeysBurst);
            }
        } else {
            KVCM_LAUNCH_HASH(8, 32);
        }
    } else if (block_size == 64) {
        if (k8 && burst) {  // 4-byte tokens take the burst form with raw tiles, above
            if constexpr (k8) {
                KVCM_LAUNCH_HASH_STAGED(8, 64, kKeysBurst);
            }
        } else {
            KVCM_LAUNCH_HASH(8, 64);
        }
    } else if (block_size == 128) {
        if (k8 && burst) {  // 4-byte tokens take the burst form with raw tiles, above
            if constexpr (k8) {
                KVCM_LAUNCH_HASH_STAGED(8, 128, kKeysBurst);
            }
        } else {
            KVCM_LAUNCH_HASH(8, 128);
        }
    } else if (block_size == 1) {  // the prefix chain over digests: a key after every step
        KVCM_LAUNCH_HASH_STAGED(1, 1, kKeysBurst);
    } else if (block_size % 8 == 0) {
        KVCM_LAUNCH_HASH(8, 0);
    } else {
        KVCM_LAUNCH_HASH(1, 0);
    }
#undef KVCM_LAUNCH_HASH_RAW
#undef KVCM_LAUNCH_HASH_STAGED
#undef KVCM_LAUNCH_HASH
    return launch_status();
}

}  // namespace
}  // namespace kvcm

extern "C" {

int32_t kvcm_hip_hash_tokens(const int64_t *d_tokens, const int64_t *d_token_offsets, int32_t R, int32_t block_size,
                             int64_t seed, int64_t *d_keys, const int64_t *d_key_offsets, kvcm_stream_t stream) {
    return kvcm::launch_hash<int64_t>(d_tokens, d_token_offsets, R, block_size, seed, d_keys, d_key_offsets,
                                      static_cast<hipStream_t>(stream));
}

int32_t kvcm_hip_hash_tokens_i32(const int32_t *d_tokens, const int64_t *d_token_offsets, int32_t R,
                                 int32_t block_size, int64_t seed, int64_t *d_keys, const int64_t *d_key_offsets,
                                 kvcm_stream_t stream) {
    return kvcm::launch_hash<int32_t>(d_tokens, d_token_offsets, R, block_size, seed, d_keys, d_key_offsets,
                                      static_cast<hipStream_t>(stream));
}

int32_t kvcm_hip_hash_tokens_2d(const void *d_tokens, int32_t token_bytes, int32_t R, int64_t tokens_per_request,
                                int32_t block_size, int64_t seed, int64_t *d_keys, const int64_t *d_key_offsets,
                                int64_t *d_key_offsets_out, kvcm_stream_t stream) {
    if ((token_bytes != 4 && token_bytes != 8) || R < 0 || block_size <= 0 || tokens_per_request < block_size) {
        return KVCM_ERR_INVALID_ARG;
    }
    const kvcm::Uniform uni{tokens_per_request, tokens_per_request / block_size, d_key_offsets_out};
    if (token_bytes == 8) {
        return kvcm::launch_hash<int64_t>(static_cast<const int64_t *>(d_tokens), nullptr, R, block_size, seed, d_keys,
                                          d_key_offsets, static_cast<hipStream_t>(stream), uni);
    }
    return kvcm::launch_hash<int32_t>(static_cast<const int32_t *>(d_tokens), nullptr, R, block_size, seed, d_keys,
                                      d_key_offsets, static_cast<hipStream_t>(stream), uni);
}

int32_t kvcm_hip_hash_tokens_checked(const void *d_tokens, int32_t token_bytes, int64_t n_tokens,
                                     const int64_t *d_token_offsets, int32_t R, int32_t block_size, int64_t seed,
                                     int64_t *d_keys, int64_t n_keys, const int64_t *d_key_offsets, kvcm_stream_t stream) {
    if ((token_bytes != 4 && token_bytes != 8) || n_tokens < 0 || n_keys < 0) {
        return KVCM_ERR_INVALID_ARG;
    }
    const kvcm::Uniform no{0, 0, nullptr};
    const kvcm::Extent have{n_tokens, n_keys};
    if (token_bytes == 8) {
        return kvcm::launch_hash<int64_t>(static_cast<const int64_t *>(d_tokens), d_token_offsets, R, block_size, seed, d_keys,
                                          d_key_offsets, static_cast<hipStream_t>(stream), no, have);
    }
    return kvcm::launch_hash<int32_t>(static_cast<const int32_t *>(d_tokens), d_token_offsets, R, block_size, seed, d_keys,
                                      d_key_offsets, static_cast<hipStream_t>(stream), no, have);
}

int32_t kvcm_hip_hash_tokens_counted(const void *d_tokens, int32_t token_bytes, int64_t n_tokens,
                                     const int64_t *d_token_offsets, int32_t R, int32_t block_size, int64_t seed,
                                     int64_t *d_keys, int64_t n_keys, int64_t *d_key_offsets, int64_t *h_total,
                                     kvcm_stream_t stream) {
    if ((token_bytes != 4 && token_bytes != 8) || n_tokens < 0 || n_keys < 0 || R <= 0 || block_size <= 0 || !d_tokens ||
        !d_token_offsets || !d_keys || !d_key_offsets || !h_total) {
        return KVCM_ERR_INVALID_ARG;
    }
    if (R > KVCM_COUNT_KEYS_UP_TO) {
        return KVCM_ERR_TOO_LARGE;
    }
    // recorded into a graph the launch would write h_total at every replay, long after the caller has given it back
    if (kvcm::is_capturing(static_cast<hipStream_t>(stream))) {
        return static_cast<int32_t>(hipErrorStreamCaptureUnsupported);
    }
    *h_total = KVCM_PENDING;
    const kvcm::Uniform no{0, 0, nullptr};
    const kvcm::Extent have{n_tokens, kvcm::room_for_keys(n_keys)};
    const kvcm::CountOut out{d_key_offsets, h_total, kvcm::make_fastdiv(static_cast<uint32_t>(block_size))};
    if (token_bytes == 8) {
        return kvcm::launch_hash<int64_t>(static_cast<const int64_t *>(d_tokens), d_token_offsets, R, block_size, seed, d_keys,
                                          nullptr, static_cast<hipStream_t>(stream), no, have, out);
    }
    return kvcm::launch_hash<int32_t>(static_cast<const int32_t *>(d_tokens), d_token_offsets, R, block_size, seed, d_keys,
                                      nullptr, static_cast<hipStream_t>(stream), no, have, out);
}

int64_t kvcm_hip_key_offsets_workspace_bytes(int32_t R) {
    return R <= kvcm::kOffsetsRereadUpTo ? 0 : kvcm::offsets_groups(R) * 8;
}

int32_t kvcm_hip_key_offsets_checked(const int64_t *d_token_offsets, int32_t R, int32_t block_size, int64_t n_tokens,
                                     int64_t n_keys, void *d_workspace, int64_t workspace_bytes, int64_t *d_key_offsets,
                                     int64_t *h_total, kvcm_stream_t stream) {
    if (R <= 0 || block_size <= 0 || n_tokens < 0 || !d_token_offsets || !d_key_offsets) {
        return KVCM_ERR_INVALID_ARG;
    }
    const int64_t groups = kvcm::offsets_groups(R);
    if (d_workspace && workspace_bytes < kvcm_hip_key_offsets_workspace_bytes(R)) {
        return KVCM_ERR_INVALID_ARG;
    }
    if (reinterpret_cast<uintptr_t>(d_workspace) % 8 != 0) {
        return KVCM_ERR_ALIGNMENT;
    }
    const hipStream_t s = static_cast<hipStream_t>(stream);
    if (h_total) {
        // recorded into a graph the launch would write h_total at every replay, long after the caller has given it back
        if (kvcm::is_capturing(s)) {
            return static_cast<int32_t>(hipErrorStreamCaptureUnsupported);
        }
        *h_total = KVCM_PENDING;
    }
    int64_t *sums = R > kvcm::kOffsetsRereadUpTo ? static_cast<int64_t *>(d_workspace) : nullptr;
    if (sums) {
        hipLaunchKernelGGL(kvcm::key_sums_kernel, dim3(static_cast<uint32_t>(groups)), dim3(kvcm::kOffsetsThreads), 0, s,
                           d_token_offsets, R, block_size, n_tokens, sums);
    }
    const int64_t threads = groups > 1 ? kvcm::kOffsetsThreads : ((R + kvcm::kOffsetsPerThread - 1) / kvcm::kOffsetsPerThread + 63) / 64 * 64;
    hipLaunchKernelGGL(kvcm::key_offsets_kernel, dim3(static_cast<uint32_t>(groups)), dim3(static_cast<uint32_t>(threads)), 0, s,
                       d_token_offsets, R, block_size, n_tokens, kvcm::room_for_keys(n_keys), sums, d_key_offsets, h_total);
    return kvcm::launch_status();
}

int32_t kvcm_hip_key_offsets(const int64_t *d_token_offsets, int32_t R, int32_t block_size, int64_t limit,
                             int64_t *d_key_offsets, int64_t *h_total, kvcm_stream_t stream) {
    return kvcm_hip_key_offsets_checked(d_token_offsets, R, block_size, kvcm::kUnknown, limit, nullptr, 0, d_key_offsets, h_total,
                                        stream);
}

int32_t kvcm_hip_prefix_chain(const int64_t *d_digests, const int64_t *d_offsets, int32_t R, int64_t *d_keys,
                              kvcm_stream_t stream) {
    // ApplyPrefixHash (trace_util.cc:47-56) is the token fold with one element per key: block_size 1,
    // seed 0, keys laid out like the digests.
    return kvcm::launch_hash<int64_t>(d_digests, d_offsets, R, 1, 0, d_keys, d_offsets,
                                      static_cast<hipStream_t>(stream));
}

int32_t kvcm_hip_sha256_first8_be(const uint8_t *d_bytes, const int64_t *d_offsets, int32_t N, int64_t *d_out,
                                  kvcm_stream_t stream) {
    if (N < 0) {
        return KVCM_ERR_INVALID_ARG;
    }
    if (N == 0) {
        return KVCM_OK;
    }
    if (!d_bytes || !d_offsets || !d_out) {
        return KVCM_ERR_INVALID_ARG;
    }
    hipLaunchKernelGGL(kvcm::sha256_first8_kernel, dim3((N + 63) / 64), dim3(64), 0, static_cast<hipStream_t>(stream),
                       d_bytes, d_offsets, N, d_out);
    return kvcm::launch_status();
}

int32_t kvcm_hip_iov_crc32(const kvcm_iov_device *d_iovs, int32_t n, uint32_t *d_crc, size_t cal_bytes,
                           kvcm_stream_t stream) {
    if (n < 0) {
        return KVCM_ERR_INVALID_ARG;
    }
    if (n == 0) {
        return KVCM_OK;
    }
    if (!d_iovs || !d_crc) {
        return KVCM_ERR_INVALID_ARG;
    }
    hipLaunchKernelGGL(kvcm::iov_crc32_kernel, dim3((n + 255) / 256), dim3(256), 0, static_cast<hipStream_t>(stream),
                       d_iovs, n, d_crc, cal_bytes);
    return kvcm::launch_status();
}

}  // extern "C"
