// si_index.hip -- device build of the superset index.
//
// Replaces superintervals.hpp:112-130 (build) + :1415-1439 (sort_intervals) and
// c_superintervals.h:462-521 (sortIntervals / indexSuperIntervals):
//   1. unless the add() flags promise canonical order, a stable LSD radix sort by start with
//      the input position as payload, whose last pass writes the sorted starts, ends, values
//      and permutation; then short runs of equal starts are put into end order (long ones:
//      the whole sort again by (start asc, end desc)).  Arrays are padded to a multiple of
//      64 entries: ends with the minimum coordinate, starts with the maximum, branch and
//      exits with NONE, so aligned 64-byte line loads never leave the allocation;
//   2. the ends in ascending order;
//   3. branch[i] = previous-greater-or-equal of ends[i] and the line exits, one lane per 16
//      positions, through a 16-ary max tree.  The previous-greater-or-equal is unique, so
//      this equals the reference's stack;
//   4. a 64-ary max tree over ends, the search trees, the long list.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <chrono>
#include <cstring>
#include <mutex>
#include <new>
#include <type_traits>
#include <vector>

#include "si_internal.h"
#include "si_prims.h"

// ============================================================================
// Error state
// ============================================================================
namespace {
thread_local char g_err[1024] = {0};
}

int si_set_error(int code, const char* fmt, ...) {
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(g_err, sizeof(g_err), fmt, ap);
    va_end(ap);
    return code;
}

// ============================================================================
// Kept blocks (si_internal.h)
// ============================================================================
namespace {
struct KeptBlock {
    void* p;
    size_t bytes;
    int device;
};
constexpr size_t KEPT_BLOCKS = 64;
struct Kept {
    std::mutex mu;
    std::vector<KeptBlock> blocks;   // oldest first, at most KEPT_BLOCKS (room for all of them from the start)
    Kept() { blocks.reserve(KEPT_BLOCKS); }
    size_t bytes = 0;
    int users = 0;
    HostStage* stages[STAGE_KEEP] = {};
};
// (never destroyed: an index may outlive the library's own static objects)
Kept& kept() {
    static Kept* const k = new Kept;
    return *k;
}

// Frees the kept blocks of one device (of all: -1).  The caller holds k.mu.
void drop_kept(Kept& k, int device) {
    size_t left = 0;
    for (const KeptBlock& b : k.blocks) {
        if (device >= 0 && b.device != device) {
            k.blocks[left++] = b;
        } else {
            (void)hipFree(b.p);
            k.bytes -= b.bytes;
        }
    }
    k.blocks.resize(left);
}
}  // namespace

void* si_block_take(size_t bytes, size_t* got, bool lasting) {
    bytes = (std::max<size_t>(bytes, 256) + 255) & ~(size_t)255;
    int dev = 0;
    (void)hipGetDevice(&dev);
    const size_t most = lasting ? bytes + bytes / 8 + (64u << 10) : 2 * bytes + (1u << 20);
    Kept& k = kept();
    {
        std::lock_guard<std::mutex> lock(k.mu);
        size_t best = k.blocks.size();
        for (size_t i = 0; i < k.blocks.size(); ++i) {
            const KeptBlock& b = k.blocks[i];
            // (a larger block is left for a request that needs it)
            if (b.device == dev && b.bytes >= bytes && b.bytes <= most &&
                (best == k.blocks.size() || b.bytes < k.blocks[best].bytes))
                best = i;
        }
        if (best < k.blocks.size()) {
            const KeptBlock b = k.blocks[best];
            k.blocks.erase(k.blocks.begin() + (ptrdiff_t)best);
            k.bytes -= b.bytes;
            *got = b.bytes;
            return b.p;
        }
    }
    void* p = nullptr;
    if (si_malloc(&p, bytes) != hipSuccess) return nullptr;
    *got = bytes;
    return p;
}

namespace {
template <class Alloc>
hipError_t malloc_or_drop(void** p, bool may_drop, Alloc alloc) {
    hipError_t e = alloc();
    if (e == hipSuccess) return e;
    (void)hipGetLastError();
    int dev = 0;
    (void)hipGetDevice(&dev);
    if (may_drop) {
        Kept& k = kept();
        std::lock_guard<std::mutex> lock(k.mu);
        drop_kept(k, dev);
    }
    if (may_drop && (e = alloc()) == hipSuccess) return e;
    (void)hipGetLastError();
    *p = nullptr;
    return e;
}
}  // namespace

hipError_t si_malloc(void** p, size_t bytes) {
    return malloc_or_drop(p, true, [&] { return hipMalloc(p, bytes); });
}

hipError_t si_malloc_async(void** p, size_t bytes, hipStream_t st) {
    hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
    const bool free_stream = hipStreamIsCapturing(st, &capture) == hipSuccess && capture == hipStreamCaptureStatusNone;
    return malloc_or_drop(p, free_stream, [&] { return hipMallocAsync(p, bytes, st); });
}

void si_block_give(void* p, size_t bytes, int device, bool quiet) {
    Kept& k = kept();
    std::lock_guard<std::mutex> lock(k.mu);
    if (!quiet || bytes > BLOCK_KEEP || k.users == 0) {
        (void)hipFree(p);
        return;
    }
    while (k.bytes + bytes > BLOCK_KEEP || k.blocks.size() >= KEPT_BLOCKS) {   // the oldest go first
        (void)hipFree(k.blocks.front().p);
        k.bytes -= k.blocks.front().bytes;
        k.blocks.erase(k.blocks.begin());
    }
    k.blocks.push_back(KeptBlock{p, bytes, device});
    k.bytes += bytes;
}

bool si_device_quiet(int device) {
    int cur = 0;
    if (hipGetDevice(&cur) != hipSuccess) return false;
    if (cur != device && hipSetDevice(device) != hipSuccess) return false;
    const hipError_t e = hipDeviceSynchronize();
    if (cur != device) (void)hipSetDevice(cur);
    if (e != hipSuccess) (void)hipGetLastError();
    return e == hipSuccess;
}

namespace {
void drop_stage(HostStage* s) {
    for (hipEvent_t e : s->ev)
        if (e) (void)hipEventDestroy(e);
    if (s->p) (void)hipHostFree(s->p);
    delete s;
}
}  // namespace

void si_block_users(int change) {
    Kept& k = kept();
    std::lock_guard<std::mutex> lock(k.mu);
    k.users += change;
    if (k.users == 0) {
        drop_kept(k, -1);
        for (HostStage*& s : k.stages) {
            if (s) drop_stage(s);
            s = nullptr;
        }
    }
}

HostStage* si_stage_take() {
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) return nullptr;
    Kept& k = kept();
    {
        std::lock_guard<std::mutex> lock(k.mu);
        for (HostStage*& s : k.stages) {
            if (s && s->device == dev) {   // (its events are the device's)
                HostStage* const got = s;
                s = nullptr;
                return got;
            }
        }
    }
    HostStage* const s = new (std::nothrow) HostStage;
    if (!s) return nullptr;
    s->device = dev;
    bool ok = hipHostMalloc((void**)&s->p, STAGE_SLOTS * STAGE_CHUNK + 256, hipHostMallocDefault) == hipSuccess;
    for (hipEvent_t& e : s->ev) ok = ok && hipEventCreateWithFlags(&e, hipEventDisableTiming) == hipSuccess;
    if (!ok) {
        (void)hipGetLastError();
        drop_stage(s);
        return nullptr;
    }
    return s;
}

void si_stage_give(HostStage* s) {
    Kept& k = kept();
    {
        std::lock_guard<std::mutex> lock(k.mu);
        if (k.users > 0) {
            for (HostStage*& slot : k.stages) {
                if (!slot) {
                    slot = s;
                    return;
                }
            }
        }
    }
    drop_stage(s);
}

SI_EXPORT const char* siGetLastError(void) { return g_err; }
SI_EXPORT const char* siVersion(void) { return "superintervals-mi355x 0.2.0 (reference API 1.0.0)"; }

namespace {
// ============================================================================
// Build kernels
// ============================================================================
__global__ void k_iota(uint32_t* __restrict__ v, size_t n) {
    size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) v[i] = (uint32_t)i;
}

// The add() flags of n intervals (superintervals.hpp:95-105): out[0] = the first i with
// starts[i + 1] < starts[i], out[1] = the first i with equal starts and ends[i + 1] > ends[i]
// (n when there is none).  start_sorted = no out[0]; end_sorted = no out[1] before out[0].
// One pass over both arrays at most (copying 10M int32 intervals to the host and scanning them
// there took 55 ms): blocks past the first break found so far read nothing.
constexpr int FLAG_ITEMS = 8;   // intervals per thread
template <typename S>
__global__ __launch_bounds__(256) void k_add_flags(const S* __restrict__ s, const S* __restrict__ e, size_t n,
                                                   unsigned long long* __restrict__ out) {
    const size_t base = (size_t)blockIdx.x * (256 * FLAG_ITEMS);
    // (one thread reads out[0], which other workgroups lower meanwhile: all waves leave, or none)
    __shared__ unsigned long long s_m[3];
    if (threadIdx.x < 2) s_m[threadIdx.x] = ~0ull;
    else if (threadIdx.x == 2) s_m[2] = __hip_atomic_load(&out[0], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __syncthreads();
    if (s_m[2] < base) return;
    unsigned long long bad = ~0ull, tie = ~0ull;
#pragma unroll
    for (int k = FLAG_ITEMS - 1; k >= 0; --k) {
        const size_t i = base + (size_t)k * 256 + threadIdx.x;
        if (i + 1 < n) {
            const S a = s[i], b = s[i + 1];
            if (b < a) bad = i;
            else if (b == a && e[i + 1] > e[i]) tie = i;
        }
    }
    // one pair of atomics a block, and only when it has found something earlier
    if (bad != ~0ull) atomicMin(&s_m[0], bad);
    if (tie != ~0ull) atomicMin(&s_m[1], tie);
    __syncthreads();
    if (threadIdx.x < 2 && s_m[threadIdx.x] < __hip_atomic_load(&out[threadIdx.x], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
        atomicMin(&out[threadIdx.x], s_m[threadIdx.x]);
}

// Padding beyond n: ends = minimum (never a hit), starts = maximum (branch and exits: NONE, by
// k_branch_exit).
template <typename S>
__global__ void k_pad(S* __restrict__ st, S* __restrict__ en, int32_t* __restrict__ vals, size_t n, size_t npad) {
    size_t i = n + threadIdx.x;
    if (i < npad) {
        st[i] = (sizeof(S) == 4) ? (S)INT32_MAX : (S)INT64_MAX;
        en[i] = (sizeof(S) == 4) ? (S)INT32_MIN : (S)INT64_MIN;
        if (vals) vals[i] = 0;
    }
}

// Sort keys and payload (the input position).  int32: (start asc, end desc) in one 64-bit
// unsigned order, so the sorted keys hold both coordinates; int64: the start.
__global__ __launch_bounds__(RS_THREADS) void k_keys_i32(const int32_t* __restrict__ s, const int32_t* __restrict__ e,
                                                         uint64_t* __restrict__ key, uint32_t* __restrict__ val, size_t n,
                                                         uint64_t* __restrict__ bits) {
    rs_each_key(n, bits, [&](size_t i) {
        const uint32_t hs = (uint32_t)s[i] ^ 0x80000000u;
        const uint32_t le = ~((uint32_t)e[i] ^ 0x80000000u);
        const uint64_t k = ((uint64_t)hs << 32) | le;
        key[i] = k;
        val[i] = (uint32_t)i;
        return k;
    });
}
__global__ __launch_bounds__(RS_THREADS) void k_keys_i64(const int64_t* __restrict__ s, uint64_t* __restrict__ key,
                                                         uint32_t* __restrict__ val, size_t n, uint64_t* __restrict__ bits) {
    rs_each_key(n, bits, [&](size_t i) {
        const uint64_t k = (uint64_t)s[i] ^ 0x8000000000000000ull;
        key[i] = k;
        val[i] = (uint32_t)i;
        return k;
    });
}

// int64 by end descending, the first of two stable sorts when runs of equal starts are long.
__global__ __launch_bounds__(RS_THREADS) void k_key_end_desc_i64(const int64_t* __restrict__ e, uint64_t* __restrict__ key,
                                                                 uint32_t* __restrict__ val, size_t n,
                                                                 uint64_t* __restrict__ bits) {
    rs_each_key(n, bits, [&](size_t i) {
        const uint64_t k = ~((uint64_t)e[i] ^ 0x8000000000000000ull);
        key[i] = k;
        val[i] = (uint32_t)i;
        return k;
    });
}

// int64 second pass key: start ascending, gathered through the first pass's order.
__global__ __launch_bounds__(RS_THREADS) void k_key_start_i64(const int64_t* __restrict__ s,
                                                              const uint32_t* __restrict__ order,
                                                              uint64_t* __restrict__ key, size_t n,
                                                              uint64_t* __restrict__ bits) {
    rs_each_key(n, bits, [&](size_t i) {
        const uint64_t k = (uint64_t)s[order[i]] ^ 0x8000000000000000ull;
        key[i] = k;
        return k;
    });
}

// The sort's last pass writes the index's arrays: the coordinates from the key where it holds
// them, the rest gathered by input position: 0.23 ms for 10M int32 intervals with payload, where
// the sort's own last pass and a gather of all three took 0.07 and 0.58 ms.
struct BuildOutI32 {
    int32_t* __restrict__ s;
    int32_t* __restrict__ e;
    uint32_t* __restrict__ perm;
    int32_t* __restrict__ v;             // null without payload
    const int32_t* __restrict__ v_in;
    __device__ __forceinline__ void put(size_t dst, uint64_t key, uint32_t val) const {
        s[dst] = (int32_t)((uint32_t)(key >> 32) ^ 0x80000000u);
        e[dst] = (int32_t)(~(uint32_t)key ^ 0x80000000u);
        perm[dst] = val;
        if (v) v[dst] = v_in[val];
    }
};
struct BuildOutI64 {
    int64_t* __restrict__ s;
    int64_t* __restrict__ e;
    uint32_t* __restrict__ perm;
    int32_t* __restrict__ v;
    const int32_t* __restrict__ v_in;
    const int64_t* __restrict__ e_in;
    __device__ __forceinline__ void put(size_t dst, uint64_t key, uint32_t val) const {
        s[dst] = (int64_t)(key ^ 0x8000000000000000ull);
        e[dst] = e_in[val];
        perm[dst] = val;
        if (v) v[dst] = v_in[val];
    }
};

// The items of a sort that ran no pass (all digits equal).
template <class Out>
__global__ __launch_bounds__(256) void k_write_items(const uint64_t* __restrict__ key, const uint32_t* __restrict__ val,
                                                     size_t n, Out out) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) out.put(i, key[i], val[i]);
}

// What the build reads back in one copy.
struct BuildInfo {
    unsigned long long inverted;   // intervals with start > end
    long long end_lo, end_hi;      // smallest and largest end
    uint32_t long_run;             // 1: a run of equal starts longer than TIE_RUN was left as it was
    uint32_t crowded[2][3];        // sampled keys in crowded buckets (CROWD) of the starts' and the sorted ends' tables
    uint32_t gaps[2];              // long gaps of the two tables (BucketGap)
    uint32_t unsorted;             // 1: a start is below the one before it
    uint32_t pad;
    long long start_lo, start_hi;  // smallest and largest start
};

// Intervals sorted by start only, in input order within equal starts: puts every run of equal
// starts into (end desc, input order), by insertion, from the lane at its head.  Runs longer
// than TIE_RUN are left and reported.  Sorting by the start alone and mending the ties takes
// half the radix passes of a sort by (start, end): 0.06 ms against four passes of 0.10 ms for 10M
// int32 intervals on 2.5e8 positions, whose runs are of one or two.
constexpr uint32_t TIE_RUN = 32;
template <typename S>
__global__ __launch_bounds__(256) void k_fix_ties(const S* __restrict__ st, S* __restrict__ en, uint32_t* __restrict__ perm,
                                                  int32_t* __restrict__ vals, size_t n, BuildInfo* __restrict__ info) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i + 1 >= n) return;
    // (everything a run of two needs to be judged is loaded at once)
    const S s = st[i], s1 = st[i + 1], s0 = i > 0 ? st[i - 1] : s, s2 = i + 2 < n ? st[i + 2] : s, e0 = en[i], e1 = en[i + 1];
    if (s1 != s || (i > 0 && s0 == s)) return;   // not the head of a run
    if (i + 2 >= n || s2 != s) {
        if (e0 >= e1) return;
        const uint32_t p0 = perm[i], p1 = perm[i + 1];
        const int32_t v0 = vals ? vals[i] : 0, v1 = vals ? vals[i + 1] : 0;
        en[i] = e1;
        en[i + 1] = e0;
        perm[i] = p1;
        perm[i + 1] = p0;
        if (vals) {
            vals[i] = v1;
            vals[i + 1] = v0;
        }
        return;
    }
    uint32_t len = 2;
    while (len <= TIE_RUN && i + len < n && st[i + len] == s) ++len;
    if (len > TIE_RUN) {
        info->long_run = 1u;
        return;
    }
    for (uint32_t k = 1; k < len; ++k) {
        const S e = en[i + k];
        const uint32_t p = perm[i + k];
        const int32_t v = vals ? vals[i + k] : 0;
        uint32_t j = k;
        for (; j > 0 && en[i + j - 1] < e; --j) {
            en[i + j] = en[i + j - 1];
            perm[i + j] = perm[i + j - 1];
            if (vals) vals[i + j] = vals[i + j - 1];
        }
        if (j != k) {
            en[i + j] = e;
            perm[i + j] = p;
            if (vals) vals[i + j] = v;
        }
    }
}

// The 16-ary max tree over the ends that the branch search climbs: level 0 = ends, level l + 1
// = the maxima of 16 entries of level l, every level padded to whole groups of 16 with the
// minimum, the last one a single group.
template <typename S>
struct Max16 {
    const S* lv[MAX_LEVELS];
    int n;   // levels
};

template <typename S>
__device__ __forceinline__ void load16(const S* __restrict__ p, S (&v)[16]) {
    constexpr int N = (int)sizeof(S);   // 16-byte words of a group
    uint4 w[N];
#pragma unroll
    for (int k = 0; k < N; ++k) w[k] = reinterpret_cast<const uint4*>(p)[k];
    memcpy(v, w, sizeof(w));
}

template <typename S>
__global__ __launch_bounds__(256) void k_max16(const S* __restrict__ in, uint32_t n_out, uint32_t n_pad,
                                               S* __restrict__ out) {
    const uint32_t j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= n_pad) return;
    S m = (sizeof(S) == 4) ? (S)INT32_MIN : (S)INT64_MIN;
    if (j < n_out) {
        S v[16];
        load16(in + (size_t)j * 16, v);
#pragma unroll
        for (int k = 0; k < 16; ++k) m = v[k] > m ? v[k] : m;
    }
    out[j] = m;
}

// Entries >= x of the group at p, as a bit mask.
template <typename S>
__device__ __forceinline__ uint32_t ge_mask16(const S* __restrict__ p, S x) {
    S v[16];
    load16(p, v);
    uint32_t m = 0;
#pragma unroll
    for (int k = 15; k >= 0; --k) m = m + m + (v[k] >= x ? 1u : 0u);
    return m;
}

// Last position <= u whose end is >= x, or NONE: the group of u, then groups further left level
// by level, then down to the last child >= x at each level.
template <typename S>
__device__ __forceinline__ uint32_t last_ge(const Max16<S>& t, uint32_t u, S x) {
    uint32_t pos = u;
    for (int l = 0; l < t.n; ++l) {
        const uint32_t g = pos & ~15u;
        const uint32_t m = ge_mask16(t.lv[l] + g, x) & ((2u << (pos & 15u)) - 1u);
        if (m) {
            uint32_t node = g + 31u - (uint32_t)__builtin_clz(m);
            for (int d = l - 1; d >= 0; --d)
                node = node * 16u + 31u - (uint32_t)__builtin_clz(ge_mask16(t.lv[d] + (size_t)node * 16u, x));
            return node;
        }
        if (g == 0u) return NONE;
        pos = g / 16u - 1u;
    }
    return NONE;
}

// branch[i] = nearest j < i with ends[j] >= ends[i], or NONE (unique, so it equals the
// reference's stack), and exitp[i]: where the line walk leaves position i's line [b0, b0 + W)
// (W = 64 bytes of ends) when every position of [b0, i] is a miss.  The reference walk entering
// that run of misses at i follows branch[] until it drops below b0; the first such element is
// the nearest j < b0 with ends[j] >= max(ends[b0..i]), i.e. branch[a] for the leftmost maximum a
// of ends[b0..i] (all of [b0, a) is below ends[a]).  It depends on i only, not on the query.
//
// One lane per 16 positions, held in registers: 120 compares give every branch inside the
// group; the others are the group's prefix maxima (3.4 of 16 for random ends), whose branches
// lie further left the larger they are, so the lane finds them in one sweep leftwards through
// the max tree, 16 entries a step.  10M int32 intervals: 0.095 ms, where a lane per position
// scanning its 64-group and climbing entry by entry took 0.36 ms (and exitp another 0.08).
// Also counts the intervals with start > end, and says whether the starts are in order (a caller's
// promise that they are may be wrong).
template <typename S>
__global__ __launch_bounds__(256) void k_branch_exit(Max16<S> t, const S* __restrict__ starts, uint32_t n, uint32_t ngroups,
                                                     uint32_t* __restrict__ branch, uint32_t* __restrict__ ex,
                                                     BuildInfo* __restrict__ info) {
    constexpr int W = 64 / (int)sizeof(S);
    __shared__ uint32_t s_b[256][17];
    const uint32_t g = blockIdx.x * 256u + threadIdx.x;
    if (g >= ngroups) return;
    uint32_t* const b = s_b[threadIdx.x];
    const uint32_t i0 = g * 16u;
    S v[16];
    load16(t.lv[0] + i0, v);
    uint32_t open = 0;   // positions whose branch lies left of the group
#pragma unroll
    for (int k = 0; k < 16; ++k) {
        uint32_t r = NONE;
#pragma unroll
        for (int j = 0; j < k; ++j) r = v[j] >= v[k] ? i0 + (uint32_t)j : r;
        const bool in = i0 + (uint32_t)k < n;
        open |= (r == NONE && in) ? 1u << k : 0u;
        b[k] = in ? r : NONE;
    }
    for (uint32_t u = i0; open && u != 0u;) {   // the branches of what is open lie below u
        const uint32_t k = (uint32_t)__builtin_ctz(open);
        open &= open - 1u;
        const uint32_t r = last_ge(t, u - 1u, t.lv[0][i0 + k]);
        if (r == NONE) break;   // the larger ones have none either
        b[k] = r;
        u = r + 1u;
    }
    uint32_t br[16], xo[16];
#pragma unroll
    for (int k = 0; k < 16; ++k) br[k] = b[k];
#pragma unroll
    for (int l = 0; l < 16; l += W) {
        S best = v[l];
        uint32_t cur = br[l];
#pragma unroll
        for (int k = 0; k < W; ++k) {
            const bool more = v[l + k] > best;
            best = more ? v[l + k] : best;
            cur = more ? br[l + k] : cur;
            xo[l + k] = i0 + (uint32_t)(l + k) < n ? cur : NONE;
        }
    }
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        reinterpret_cast<uint4*>(branch + i0)[k] = make_uint4(br[4 * k], br[4 * k + 1], br[4 * k + 2], br[4 * k + 3]);
        reinterpret_cast<uint4*>(ex + i0)[k] = make_uint4(xo[4 * k], xo[4 * k + 1], xo[4 * k + 2], xo[4 * k + 3]);
    }
    S st[16];
    load16(starts + i0, st);
    uint32_t inv = 0;
#pragma unroll
    for (int k = 0; k < 16; ++k) inv += (st[k] > v[k] && i0 + (uint32_t)k < n) ? 1u : 0u;
    if (inv) atomicAdd(&info->inverted, (unsigned long long)inv);
    bool falls = g + 1u < ngroups && starts[i0 + 16u] < st[15];   // (padded with the maximum)
#pragma unroll
    for (int k = 1; k < 16; ++k) falls |= st[k] < st[k - 1];
    if (falls) info->unsorted = 1u;
}

// Sums of 16 consecutive entries of a and of b (lines of n / 16 + 1 each, the last one partial;
// a is padded to whole lines, b is not), modulo 2^32, into out and out + lines.
__global__ __launch_bounds__(256) void k_line_sums(const int32_t* __restrict__ a, const int32_t* __restrict__ b, uint32_t n,
                                                   uint32_t lines, uint32_t* __restrict__ out) {
    const uint32_t k = blockIdx.x * 256u + threadIdx.x;
    if (k >= 2u * lines) return;
    const uint32_t l = k < lines ? k : k - lines;
    const int32_t* const p = (k < lines ? a : b) + (size_t)l * 16;
    uint32_t sum = 0;
    if (l + 1 < lines) {
        int32_t v[16];
        load16(p, v);
#pragma unroll
        for (int j = 0; j < 16; ++j) sum += (uint32_t)v[j];
    } else {
        for (uint32_t j = 0; j < (n & 15u); ++j) sum += (uint32_t)p[j];
    }
    out[k] = sum;
}

// ---- bucket tables (BucketView) ----------------------------------------------------------
// Entries of a table between the buckets of two neighbouring keys that are too many for one
// wave; filled by k_bucket_gaps.
struct BucketGap {
    uint32_t from, to, value;   // tab[from .. to) = value
};
constexpr uint32_t GAP_WAVE = 4096;       // most entries a wave fills by itself

// At most max(n / 4, 1) buckets of a power of two of values over a span: its exponent.
__host__ __device__ inline uint32_t bucket_shift(uint64_t span, uint64_t n) {
    const uint64_t most = n / 4 ? n / 4 : 1;
    uint32_t shift = 0;
    while ((span >> shift) >= most && shift < 63) ++shift;
    return shift;
}

// The ranges of the sorted starts and ends, and how crowded their buckets will be: of CROWD_SAMPLE keys
// those that share one with the CROWD-th key after them, three degrees (in a bucket of m keys m - CROWD do,
// half from twice as many on).  One workgroup, before the tables: counted by the kernel that fills them, an
// atomic a sample, 10M intervals in 20 clusters took 5.5 ms to build, so 2.6.
__device__ constexpr uint32_t CROWD[3] = {32, 256, 4096};
constexpr uint32_t CROWD_SAMPLE = 512;   // (4096: 40 us, the misses of one CU)
template <typename S>
__global__ __launch_bounds__(CROWD_SAMPLE) void k_ranges(const S* __restrict__ starts, const S* __restrict__ sorted, size_t n,
                                                 BuildInfo* __restrict__ info) {
    __shared__ uint32_t s_c[2][3];
    if (threadIdx.x < 6) s_c[threadIdx.x / 3][threadIdx.x % 3] = 0;
    __syncthreads();
    for (int which = 0; which < 2; ++which) {
        const S* const v = which ? sorted : starts;
        const S lo = v[0], hi = v[n - 1];
        const BucketView<S> t{nullptr, lo, hi, bucket_shift((uint64_t)hi - (uint64_t)lo, n)};
        if (threadIdx.x == 0) {
            (which ? info->end_lo : info->start_lo) = (long long)lo;
            (which ? info->end_hi : info->start_hi) = (long long)hi;
        }
        const size_t i = (uint64_t)threadIdx.x * n / CROWD_SAMPLE;
        const uint64_t b = bucket_of(t, v[i]);
        bool with[3];
#pragma unroll
        for (int d = 0; d < 3; ++d) with[d] = n - i > CROWD[d] && bucket_of(t, v[i + (n - i > CROWD[d] ? CROWD[d] : 0u)]) == b;
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            const uint64_t m = __ballot(with[d]);
            if (lane_id() == 0 && m) atomicAdd(&s_c[which][d], (uint32_t)__popcll(m));
        }
    }
    __syncthreads();
    if (threadIdx.x < 6) info->crowded[threadIdx.x / 3][threadIdx.x % 3] = s_c[threadIdx.x / 3][threadIdx.x % 3];
}

// tab[b] = i for the buckets b above key i - 1's up to key i's, and n above the last key's.
template <typename S>
__global__ __launch_bounds__(256) void k_bucket_table(const S* __restrict__ v, uint32_t n, BucketView<S> t, uint32_t nb,
                                                      uint32_t* __restrict__ tab, BucketGap* __restrict__ gaps,
                                                      uint32_t* __restrict__ ngaps, const uint32_t* __restrict__ unsorted) {
    if (*unsorted) return;   // a key may lie in no bucket: the searches go through the trees
    const uint32_t i = blockIdx.x * 256u + threadIdx.x;   // n included: the entries past the last key
    const int lane = lane_id();
    uint32_t lo = 0, hi = 0;   // entries [lo, hi) are i
    if (i < n) {
        hi = (uint32_t)bucket_of(t, v[i]) + 1u;
        lo = i ? (uint32_t)bucket_of(t, v[i - 1]) + 1u : 0u;
    } else if (i == n) {
        lo = (uint32_t)bucket_of(t, v[n - 1]) + 1u;
        hi = nb + 1u;
    }
    const uint32_t len = hi - lo;
    if (len == 1u) tab[lo] = i;
    if (len > GAP_WAVE) gaps[atomicAdd(ngaps, 1u)] = BucketGap{lo, hi, i};
    for (uint64_t m = __ballot(len > 1u && len <= GAP_WAVE); m; m &= m - 1ull) {
        const int L = __builtin_ctzll(m);
        const uint32_t a = __shfl(lo, L, WAVE), b = __shfl(hi, L, WAVE), x = __shfl(i, L, WAVE);
        for (uint32_t k = a + (uint32_t)lane; k < b; k += WAVE) tab[k] = x;
    }
}

__global__ __launch_bounds__(256) void k_bucket_gaps(const BucketGap* __restrict__ gaps, const uint32_t* __restrict__ ngaps,
                                                     uint32_t* __restrict__ tab) {
    const uint32_t m = *ngaps;
    for (uint32_t g = 0; g < m; ++g) {
        const BucketGap p = gaps[g];
        for (uint64_t k = (uint64_t)p.from + blockIdx.x * 256u + threadIdx.x; k < p.to; k += (uint64_t)gridDim.x * 256u)
            tab[k] = p.value;
    }
}

// One wave per output node: out[b] = max(in[64b .. 64b+63]).
template <typename S>
__global__ __launch_bounds__(256) void k_tree_level(const S* __restrict__ in, size_t n_in,
                                                    S* __restrict__ out, size_t n_out) {
    size_t b = ((size_t)blockIdx.x * blockDim.x + threadIdx.x) >> 6;
    if (b >= n_out) return;
    size_t i = b * FAN + lane_id();
    S v = (i < n_in) ? in[i] : (sizeof(S) == 4 ? (S)INT32_MIN : (S)INT64_MIN);
    v = wave_max(v);
    if (lane_id() == 0) out[b] = v;
}

// Search tree for upper_bound.  Level l + 1 holds every 64th key of level l (out[j] =
// in[64 j]), so the 64 keys of level l below entry j of level l + 1 are one 256-byte
// (int32) node whose first key is that entry.
template <typename S>
__global__ __launch_bounds__(256) void k_every64(const S* __restrict__ in, uint32_t n_out, S* __restrict__ out) {
    const uint32_t j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j < n_out) out[j] = in[(size_t)j * 64];
}

// The top level in Eytzinger order: node k (1-based, k < 2^h) at depth d holds in-order
// element i = ((2 (k - 2^d) + 1) << (h - 1 - d)) - 1 of the level, or max(S) past its end.
template <typename S>
__global__ __launch_bounds__(256) void k_eytz(const S* __restrict__ lvl, uint32_t m, uint32_t h, S* __restrict__ top) {
    const uint32_t k = 1 + blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= (1u << h)) return;
    const uint32_t d = 31u - (uint32_t)__builtin_clz(k);
    const uint32_t i = ((2u * (k - (1u << d)) + 1u) << (h - 1u - d)) - 1u;
    top[k - 1] = (i < m) ? lvl[i] : ((sizeof(S) == 4) ? (S)INT32_MAX : (S)INT64_MAX);
}

// ends[i] - base as uint32 (the caller checked that every end fits), 0 in the padding.
__global__ __launch_bounds__(256) void k_ends32(const int64_t* __restrict__ ends, size_t n, size_t npad, int64_t base,
                                                uint32_t* __restrict__ out) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < npad) out[i] = (i < n) ? (uint32_t)((uint64_t)ends[i] - (uint64_t)base) : 0u;
}

// ---- the long list (LongView) ---------------------------------------------------------
// end - start + 1 > len, in 64-bit arithmetic that cannot overflow (start > end: not long).
template <typename S>
__device__ __forceinline__ bool longer_than(S st, S en, int64_t len) {
    if (en < st) return false;
    return (uint64_t)en - (uint64_t)st >= (uint64_t)len;   // (end - start + 1) > len
}

// Lengths of m evenly spaced intervals (for the threshold).
template <typename S>
__global__ __launch_bounds__(256) void k_len_sample(const S* __restrict__ st, const S* __restrict__ en, uint32_t n,
                                                    uint32_t m, int64_t* __restrict__ out) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= m) return;
    const uint32_t p = (uint32_t)((uint64_t)i * n / m);
    const uint64_t d = (uint64_t)en[p] - (uint64_t)st[p];
    out[i] = (en[p] < st[p]) ? 0 : (d >= (uint64_t)INT64_MAX ? INT64_MAX : (int64_t)d + 1);
}

template <typename S>
__global__ __launch_bounds__(256) void k_long_flags(const S* __restrict__ st, const S* __restrict__ en, uint32_t n,
                                                    int64_t len, uint32_t* __restrict__ flags) {
    const uint32_t p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p < n) flags[p] = longer_than(st[p], en[p], len) ? 1u : 0u;
}

// Entry j = lrank[p] of every long position p; the padding past nlong never hits.
template <typename S>
__global__ __launch_bounds__(256) void k_long_fill(const S* __restrict__ en, const uint32_t* __restrict__ en32,
                                                   const uint32_t* __restrict__ flags, const uint32_t* __restrict__ lrank,
                                                   uint32_t n, uint32_t nlong, uint32_t npad, uint32_t* __restrict__ pos,
                                                   S* __restrict__ lends, uint32_t* __restrict__ lends32) {
    const uint32_t p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p < n && flags[p]) {
        const uint32_t j = lrank[p];
        pos[j] = p;
        lends[j] = en[p];
        if (lends32) lends32[j] = en32[p];
    }
    if (p >= nlong && p < npad) {
        pos[p] = NONE;
        lends[p] = (sizeof(S) == 4) ? (S)INT32_MIN : (S)INT64_MIN;
        if (lends32) lends32[p] = 0u;
    }
}

// Device memory handed out from one allocation, in 256-byte steps.
struct Carver {
    char* base = nullptr;
    size_t used = 0;
    template <typename T>
    T* take(size_t count) {
        T* const p = base ? (T*)(base + used) : nullptr;
        used += align256(count * sizeof(T));
        return p;
    }
};

// Sizes of a search tree over n sorted keys: 64-ary levels of first keys up to a top level of
// at most 4095 keys, which is also stored in Eytzinger order (k_every64, k_eytz).
struct KeyTreeShape {
    uint32_t size[MAX_LEVELS + 1];   // level 0 = the keys
    int nlv = 0;
    size_t entries = 0;              // of levels 1 .. nlv
    uint32_t top_h = 0;
    explicit KeyTreeShape(size_t n) {
        size[0] = (uint32_t)n;
        while (size[nlv] > 4095 && nlv < MAX_LEVELS - 1) {
            size[nlv + 1] = (uint32_t)(((size_t)size[nlv] + 63) / 64);
            ++nlv;
            entries += size[nlv];
        }
        while (((1u << top_h) - 1u) < size[nlv]) ++top_h;
    }
};

template <typename S>
void carve_key_tree(const KeyTreeShape& h, KeyTree& t, Carver& c) {
    t.d_lv = c.take<S>(h.entries);
    t.d_top = c.take<S>((1u << h.top_h) - 1u);
}

template <typename S>
int build_key_tree(const S* keys, const KeyTreeShape& h, KeyTree& t, hipStream_t st) {
    t.nlv = h.nlv;
    size_t tot = 0;
    for (int l = 1; l <= h.nlv; ++l) {
        t.lv_off[l] = tot;
        t.lv_size[l] = h.size[l];
        const S* in = (l == 1) ? keys : (const S*)t.d_lv + t.lv_off[l - 1];
        k_every64<S><<<grid_for(h.size[l], 256), 256, 0, st>>>(in, h.size[l], (S*)t.d_lv + tot);
        LAUNCH_CHECK();
        tot += h.size[l];
    }
    t.top_size = h.size[h.nlv];
    t.top_h = h.top_h;
    const S* topl = (h.nlv == 0) ? keys : (const S*)t.d_lv + t.lv_off[h.nlv];
    k_eytz<S><<<grid_for((1u << h.top_h) - 1u, 256), 256, 0, st>>>(topl, t.top_size, h.top_h, (S*)t.d_top);
    LAUNCH_CHECK();
    return SI_OK;
}

// Entries a bucket table over n keys may take, and its longest list of gaps.
constexpr size_t bucket_entries(size_t n) { return n / 4 + 2; }
constexpr size_t bucket_gaps(size_t n) { return bucket_entries(n) / GAP_WAVE + 2; }

// Bucket table over n sorted keys in [lo, hi]: at most n / 4 buckets of a power of two of values.
// scratch holds bucket_gaps(n) entries.  Whether the table is used (t.ok) is left to the caller,
// who has read the crowded samples back (k_ranges).
template <typename S>
int build_bucket_table(const S* keys, size_t n, int64_t lo, int64_t hi, BucketTable& t, BuildInfo* info, int which,
                       Carver scratch, hipStream_t st) {
    t.lo = lo;
    t.hi = hi;
    const uint64_t span = (uint64_t)hi - (uint64_t)lo;
    t.shift = bucket_shift(span, n);
    const uint32_t nb = (uint32_t)(span >> t.shift) + 1u;
    BucketGap* const gaps = scratch.take<BucketGap>(bucket_gaps(n));
    const BucketView<S> v{t.d_tab, (S)lo, (S)hi, t.shift};
    k_bucket_table<S><<<grid_for(n + 1, 256), 256, 0, st>>>(keys, (uint32_t)n, v, nb, t.d_tab, gaps, &info->gaps[which],
                                                            &info->unsorted);
    LAUNCH_CHECK();
    if (nb > GAP_WAVE) {
        k_bucket_gaps<<<64, 256, 0, st>>>(gaps, &info->gaps[which], t.d_tab);
        LAUNCH_CHECK();
    }
    return SI_OK;
}

// Level sizes and offsets of a 64-ary max tree over n entries (level 0); returns the entries of
// the levels above.
size_t tree_shape(uint32_t n, int* nlev, size_t* off, uint32_t* size) {
    size[0] = n;
    int l = 1;
    size_t tot = 0;
    while (size[l - 1] > (uint32_t)FAN && l < MAX_LEVELS) {
        off[l] = tot;
        size[l] = (uint32_t)(((size_t)size[l - 1] + FAN - 1) / FAN);
        tot += size[l];
        ++l;
    }
    *nlev = l;
    return tot;
}

template <typename S>
int build_max_tree(const S* ends, int nlev, const size_t* off, const uint32_t* size, S* tree, hipStream_t st) {
    for (int l = 1; l < nlev; ++l) {
        const S* in = (l == 1) ? ends : tree + off[l - 1];
        k_tree_level<S><<<grid_for((size_t)size[l] * FAN, 256), 256, 0, st>>>(in, size[l - 1], tree + off[l], size[l]);
        LAUNCH_CHECK();
    }
    return SI_OK;
}

constexpr uint32_t LEN_SAMPLE = 4096;        // lengths the long list's threshold is chosen from
constexpr size_t LONG_FROM = 1u << 16;        // smallest index that gets one by itself

// The long list of a built index: the threshold (the tuning's, or 64 x the median of the sampled
// lengths rounded up to a power of two), the positions and ends of the longer intervals and the
// max tree over those ends.  Left out (len = 0) for indexes under 2^16 intervals, and when the
// chosen threshold leaves more than half of the intervals long.  scratch holds 4 n bytes and a
// scan workspace.
template <typename S>
int build_long_list(siIndex* ix, std::vector<int64_t>& lens, Carver scratch, hipStream_t st) {
    const uint32_t n = (uint32_t)ix->n;
    int64_t len = si_tune_long_len();
    const bool automatic = len == 0;
    if (len < 0 || (automatic && n < LONG_FROM)) return SI_OK;   // (scratch untouched)
    const S* d_st = (const S*)ix->d_starts;
    const S* d_en = (const S*)ix->d_ends;
    if (automatic) {
        std::nth_element(lens.begin(), lens.begin() + LEN_SAMPLE / 2, lens.end());
        const int64_t med = std::max<int64_t>(lens[LEN_SAMPLE / 2], 1);
        len = 1;
        while (len < 64 * med && len < ((int64_t)1 << 62)) len <<= 1;
    }
    LongList& L = ix->lng;
    uint32_t* const flags = scratch.take<uint32_t>(n);
    uint32_t* const ws = scratch.take<uint32_t>(scan_ws_items(n));
    if (!(L.d_lrank = (uint32_t*)si_block_take(((size_t)n + 1) * 4, &L.lrank_bytes, true)))
        return si_set_error(SI_ERR_NOMEM, "long list: %zu bytes", ((size_t)n + 1) * 4);
    k_long_flags<S><<<grid_for(n, 256), 256, 0, st>>>(d_st, d_en, n, len, flags);
    LAUNCH_CHECK();
    const int rc = device_excl_scan<uint32_t, uint32_t>(flags, n, L.d_lrank, L.d_lrank + n, ws, st);
    if (rc != SI_OK) return rc;
    uint32_t nlong = 0;
    HIP_TRY(hipMemcpyAsync(&nlong, L.d_lrank + n, 4, hipMemcpyDeviceToHost, st));
    HIP_TRY(hipStreamSynchronize(st));
    if (nlong == 0 || (automatic && nlong > n / 2)) {
        L.release(ix->device, true);
        return SI_OK;
    }
    const uint32_t npad = (nlong + 63u) & ~63u;
    const size_t tot = tree_shape(nlong, &L.nlev, L.lvl_off, L.lvl_size);
    Carver c;
    for (int pass = 0; pass < 2; ++pass) {   // sizes, then pointers
        c.used = 0;
        L.d_pos = c.take<uint32_t>(npad);
        L.d_ends = c.take<S>(npad);
        L.d_ends32 = ix->d_ends32 ? c.take<uint32_t>(npad) : nullptr;
        L.d_tree = c.take<S>(tot);
        if (pass == 0) {
            if (!(L.d_block = si_block_take(c.used, &L.block_bytes, true)))
                return si_set_error(SI_ERR_NOMEM, "long list: %zu bytes", c.used);
            c.base = (char*)L.d_block;
        }
    }
    k_long_fill<S><<<grid_for(std::max(n, npad), 256), 256, 0, st>>>(d_en, ix->d_ends32, flags, L.d_lrank, n, nlong,
                                                                     npad, L.d_pos, (S*)L.d_ends, L.d_ends32);
    LAUNCH_CHECK();
    const int rt = build_max_tree<S>((const S*)L.d_ends, L.nlev, L.lvl_off, L.lvl_size, (S*)L.d_tree, st);
    if (rt != SI_OK) return rt;
    L.len = len;
    L.n = nlong;
    return SI_OK;
}

// The build's scratch: one block, given back when the build ends either way.
struct BuildScratch {
    void* p = nullptr;
    size_t bytes = 0;
    int device = 0;
    hipStream_t st = nullptr;
    ~BuildScratch() {
        if (!p) return;
        // (an early return may leave kernels that use it)
        si_block_give(p, bytes, device, hipStreamSynchronize(st) == hipSuccess);
    }
};

// Sorts the n > 0 intervals into ix's arrays, canonically: by start, in one radix sort, then the
// runs of equal starts by end (k_fix_ties); full = true sorts by (start, end) instead.
template <typename S>
int sort_intervals(siIndex* ix, const S* in_s, const S* in_e, const int32_t* in_v, size_t n, bool full, uint64_t* k0,
                   uint64_t* k1, uint32_t* v0, uint32_t* v1, const RsTemp& rt, BuildInfo* info, uint64_t* varying,
                   hipStream_t st) {
    const unsigned g = grid_for(n, 256), gk = rs_bits_grid(n);
    uint64_t* ks;
    uint32_t* vs;
    bool written = false;
    int rc;
    if constexpr (sizeof(S) == 4) {
        const BuildOutI32 out{(int32_t*)ix->d_starts, (int32_t*)ix->d_ends, ix->d_perm, ix->d_values, in_v};
        k_keys_i32<<<gk, RS_THREADS, 0, st>>>(in_s, in_e, k0, v0, n, rt.bits);
        LAUNCH_CHECK();
        if ((rc = rs_varying_bits(n, rt, varying, st)) != SI_OK) return rc;
        rc = radix_sort_pairs(k0, v0, k1, v1, n, full ? 0 : 4, 8, rt, &ks, &vs, st, *varying, &out, &written);
        if (rc != SI_OK) return rc;
        *varying &= 0xFFFFFFFFull;   // the ends', for their sort
        if (!written) k_write_items<BuildOutI32><<<g, 256, 0, st>>>(ks, vs, n, out);
    } else {
        const BuildOutI64 out{(int64_t*)ix->d_starts, (int64_t*)ix->d_ends, ix->d_perm, ix->d_values, in_v,
                              (const int64_t*)in_e};
        uint64_t *ka = k0, *kb = k1, vary = 0;
        uint32_t *va = v0, *vb = v1;
        if (full) {   // two stable sorts: end descending, then start ascending
            k_key_end_desc_i64<<<gk, RS_THREADS, 0, st>>>((const int64_t*)in_e, k0, v0, n, rt.bits);
            LAUNCH_CHECK();
            if ((rc = rs_varying_bits(n, rt, &vary, st)) != SI_OK) return rc;
            if ((rc = radix_sort_pairs(k0, v0, k1, v1, n, 0, 8, rt, &ks, &vs, st, vary)) != SI_OK) return rc;
            ka = (ks == k0) ? k1 : k0;   // the free key buffer
            kb = ks;
            va = vs;
            vb = (vs == v0) ? v1 : v0;
            k_key_start_i64<<<gk, RS_THREADS, 0, st>>>((const int64_t*)in_s, va, ka, n, rt.bits);
        } else {
            k_keys_i64<<<gk, RS_THREADS, 0, st>>>((const int64_t*)in_s, ka, va, n, rt.bits);
        }
        LAUNCH_CHECK();
        if ((rc = rs_varying_bits(n, rt, &vary, st)) != SI_OK) return rc;
        rc = radix_sort_pairs(ka, va, kb, vb, n, 0, 8, rt, &ks, &vs, st, vary, &out, &written);
        if (rc != SI_OK) return rc;
        if (!written) k_write_items<BuildOutI64><<<g, 256, 0, st>>>(ks, vs, n, out);
    }
    LAUNCH_CHECK();
    if (!full) {
        k_fix_ties<S><<<g, 256, 0, st>>>((const S*)ix->d_starts, (S*)ix->d_ends, ix->d_perm, ix->d_values, n, info);
        LAUNCH_CHECK();
    }
    return SI_OK;
}

template <typename S>
int build_impl(siIndex* ix, const void* starts, const void* ends, const int32_t* values, size_t n,
               int start_sorted, int end_sorted, int on_device, hipStream_t st) {
    auto t0 = std::chrono::steady_clock::now();
    ix->release();
    (void)hipGetDevice(&ix->device);   // the arrays lie on the device that is current now
    if (n == 0) {
        ix->built = true;
        ix->last_build_ms = 0;
        return SI_OK;
    }
    if (n >= (size_t)NONE) return si_set_error(SI_ERR_ARG, "index size %zu exceeds 2^32-2", n);
    const size_t nb = n * sizeof(S);
    const size_t npad = (n + 63) & ~(size_t)63;   // sorted arrays: a multiple of 64 entries (see the file comment)

    // ---- the index's block: sizes, then pointers
    const KeyTreeShape shape(n);
    const size_t tree_n = tree_shape((uint32_t)n, &ix->nlev, ix->lvl_off, ix->lvl_size);
    Carver c;
    for (int pass = 0; pass < 2; ++pass) {
        c.used = 0;
        ix->d_starts = c.take<S>(npad + 64);   // (bucket searches read a little past the last key)
        ix->d_ends = c.take<S>(npad);
        ix->d_branch = c.take<uint32_t>(npad);
        ix->d_exit = c.take<uint32_t>(npad);
        ix->d_perm = c.take<uint32_t>(n);
        ix->d_values = values ? c.take<int32_t>(npad) : nullptr;
        ix->d_ends_sorted = c.take<S>(npad + 64);   // (bucket searches read a little past the last key)
        ix->ubt.d_tab = c.take<uint32_t>(bucket_entries(n));
        ix->ebt.d_tab = c.take<uint32_t>(bucket_entries(n));
        ix->d_tree = c.take<S>(tree_n);
        ix->d_line_sums = sizeof(S) == 4 ? c.take<uint32_t>(2 * (n / 16 + 1)) : nullptr;
        carve_key_tree<S>(shape, ix->ub, c);
        carve_key_tree<S>(shape, ix->eb, c);
        if (pass == 0) {
            if (!(ix->d_block = si_block_take(c.used, &ix->block_bytes, true)))
                return si_set_error(SI_ERR_NOMEM, "index of %zu intervals: %zu bytes", n, c.used);
            c.base = (char*)ix->d_block;
        }
    }

    // ---- the scratch: read-backs, device copies of host inputs, then what the stages share one
    // after another (sort buffers, the 16-ary max tree, the long list's flags)
    BuildScratch scratch;
    scratch.device = ix->device;
    scratch.st = st;
    Carver w;
    BuildInfo* info = nullptr;
    int64_t* d_lens = nullptr;
    unsigned long long* d_flags = nullptr;
    S *in_s = nullptr, *in_e = nullptr;
    int32_t* in_v = nullptr;
    uint64_t *k0 = nullptr, *k1 = nullptr;
    uint32_t *v0 = nullptr, *v1 = nullptr;
    char* rt_base = nullptr;
    size_t shared_from = 0;
    for (int pass = 0; pass < 2; ++pass) {
        w.used = 0;
        info = w.take<BuildInfo>(1);
        d_lens = w.take<int64_t>(LEN_SAMPLE);   // (right behind info: read back together)
        d_flags = w.take<unsigned long long>(2);
        in_s = on_device ? (S*)starts : w.take<S>(n);
        in_e = on_device ? (S*)ends : w.take<S>(n);
        in_v = !values ? nullptr : on_device ? (int32_t*)values : w.take<int32_t>(n);
        shared_from = w.used;
        rt_base = w.take<char>(rs_temp_bytes(n));
        k0 = w.take<uint64_t>(npad);
        k1 = w.take<uint64_t>(npad);
        v0 = w.take<uint32_t>(npad);
        v1 = w.take<uint32_t>(npad);
        if (pass == 0) {
            if (!(scratch.p = si_block_take(w.used, &scratch.bytes)))
                return si_set_error(SI_ERR_NOMEM, "build scratch: %zu bytes", w.used);
            w.base = (char*)scratch.p;
        }
    }
    const RsTemp rt = rs_temp_carve(rt_base, n);
    if (!on_device) {
        HIP_TRY(hipMemcpyAsync(in_s, starts, nb, hipMemcpyHostToDevice, st));
        HIP_TRY(hipMemcpyAsync(in_e, ends, nb, hipMemcpyHostToDevice, st));
        if (values) HIP_TRY(hipMemcpyAsync(in_v, values, n * sizeof(int32_t), hipMemcpyHostToDevice, st));
    }
    k_zero_u32<<<1, 64, 0, st>>>((uint32_t*)info, sizeof(BuildInfo) / 4);
    LAUNCH_CHECK();
    if (start_sorted < 0 || end_sorted < 0) {
        unsigned long long f[2] = {~0ull, ~0ull};
        HIP_TRY(hipMemcpyAsync(d_flags, f, sizeof(f), hipMemcpyHostToDevice, st));
        k_add_flags<S><<<grid_for(n, 256 * FLAG_ITEMS), 256, 0, st>>>(in_s, in_e, n, d_flags);
        LAUNCH_CHECK();
        HIP_TRY(hipMemcpyAsync(f, d_flags, sizeof(f), hipMemcpyDeviceToHost, st));
        HIP_TRY(hipStreamSynchronize(st));
        if (start_sorted < 0) start_sorted = f[0] == ~0ull;
        if (end_sorted < 0) end_sorted = !(f[1] < f[0]);
    }
    if (npad > n) {
        k_pad<S><<<1, 64, 0, st>>>((S*)ix->d_starts, (S*)ix->d_ends, ix->d_values, n, npad);
        LAUNCH_CHECK();
    }
    ix->n = n;
    const bool presorted = start_sorted && end_sorted;
    struct { BuildInfo info; char gap[align256(sizeof(BuildInfo)) - sizeof(BuildInfo)]; int64_t lens[LEN_SAMPLE]; } back;
    for (bool full = false;; full = true) {
        // ---- the sorted arrays
        uint64_t varying = 0;   // the ends' bits that vary
        bool known = false;
        if (presorted) {
            k_iota<<<grid_for(n, 256), 256, 0, st>>>(ix->d_perm, n);
            LAUNCH_CHECK();
            HIP_TRY(hipMemcpyAsync(ix->d_starts, in_s, nb, hipMemcpyDeviceToDevice, st));
            HIP_TRY(hipMemcpyAsync(ix->d_ends, in_e, nb, hipMemcpyDeviceToDevice, st));
            if (values) HIP_TRY(hipMemcpyAsync(ix->d_values, in_v, n * 4, hipMemcpyDeviceToDevice, st));
        } else {
            const int rc = sort_intervals<S>(ix, in_s, in_e, in_v, n, full, k0, k1, v0, v1, rt, info, &varying, st);
            if (rc != SI_OK) return rc;
            known = sizeof(S) == 4;
        }
        // ---- ends in ascending order, for the rank form of count (whatever the order within equal starts)
        if (!full) {
            using K = typename std::conditional<sizeof(S) == 4, uint32_t, uint64_t>::type;
            const K* raw = (const K*)ix->d_ends;
            if (!known) {
                k_rs_bits<K><<<rs_bits_grid(n), RS_THREADS, 0, st>>>(raw, n, rt.bits);
                LAUNCH_CHECK();
                const int rc = rs_varying_bits(n, rt, &varying, st);
                if (rc != SI_OK) return rc;
            }
            if (varying) {
                const int rc = radix_sort_signed<K>(raw, (K*)k0, (K*)k1, (K*)ix->d_ends_sorted, n, varying, rt, st);
                if (rc != SI_OK) return rc;
            } else {   // all ends equal
                HIP_TRY(hipMemcpyAsync(ix->d_ends_sorted, ix->d_ends, nb, hipMemcpyDeviceToDevice, st));
            }
            k_ranges<S><<<1, CROWD_SAMPLE, 0, st>>>((const S*)ix->d_starts, (const S*)ix->d_ends_sorted, n, info);
            LAUNCH_CHECK();
        }
        // ---- the lengths the long list's threshold is chosen from, and the one read-back (before the
        // stages that another sort would have to repeat: 10M int32 intervals with one run of 50 equal
        // starts 2.9 ms with them in between, so 2.5, without such a run 1.4)
        const bool sample = n >= LONG_FROM && si_tune_long_len() == 0;
        if (sample) {
            k_len_sample<S><<<grid_for(LEN_SAMPLE, 256), 256, 0, st>>>((const S*)ix->d_starts, (const S*)ix->d_ends,
                                                                       (uint32_t)n, LEN_SAMPLE, d_lens);
            LAUNCH_CHECK();
        }
        HIP_TRY(hipMemcpyAsync(&back, info, sample ? sizeof(back) : sizeof(BuildInfo), hipMemcpyDeviceToHost, st));
        HIP_TRY(hipStreamSynchronize(st));
        if (presorted || full || !back.info.long_run) break;
        // runs of equal starts too long to mend: sort by (start, end)
    }
    // ---- branch and exits, through the 16-ary max tree
    {
        Carver m;
        m.base = (char*)scratch.p;
        m.used = shared_from;
        Max16<S> t;
        t.lv[0] = (const S*)ix->d_ends;
        t.n = 1;
        size_t sz = npad;
        while (sz > 16 && t.n < MAX_LEVELS) {
            const size_t up = (sz + 15) / 16, pad = (up + 15) & ~(size_t)15;
            S* const lv = m.take<S>(pad);
            k_max16<S><<<grid_for(pad, 256), 256, 0, st>>>(t.lv[t.n - 1], (uint32_t)up, (uint32_t)pad, lv);
            LAUNCH_CHECK();
            t.lv[t.n++] = lv;
            sz = up;
        }
        for (int l = t.n; l < MAX_LEVELS; ++l) t.lv[l] = nullptr;
        k_branch_exit<S><<<grid_for(npad / 16, 256), 256, 0, st>>>(t, (const S*)ix->d_starts, (uint32_t)n,
                                                                   (uint32_t)(npad / 16), ix->d_branch, ix->d_exit,
                                                                   info);
        LAUNCH_CHECK();
    }
    int rc = build_max_tree<S>((const S*)ix->d_ends, ix->nlev, ix->lvl_off, ix->lvl_size, (S*)ix->d_tree, st);
    if (rc == SI_OK) rc = build_key_tree<S>((const S*)ix->d_starts, shape, ix->ub, st);        // upper_bound
    if (rc == SI_OK) rc = build_key_tree<S>((const S*)ix->d_ends_sorted, shape, ix->eb, st);   // rank count
    if (rc != SI_OK) return rc;
    {
        Carver m;
        m.base = (char*)scratch.p;
        m.used = shared_from;
        rc = build_bucket_table<S>((const S*)ix->d_starts, n, back.info.start_lo, back.info.start_hi, ix->ubt, info, 0, m, st);
        m.take<BucketGap>(bucket_gaps(n));
        if (rc == SI_OK)
            rc = build_bucket_table<S>((const S*)ix->d_ends_sorted, n, back.info.end_lo, back.info.end_hi, ix->ebt, info, 1,
                                       m, st);
        if (rc != SI_OK) return rc;
    }
    if constexpr (sizeof(S) == 4) {
        const size_t lines = ix->sum_lines();
        Carver m;
        m.base = (char*)scratch.p;
        m.used = shared_from;
        m.take<BucketGap>(2 * bucket_gaps(n) + 64);   // (behind the tables' gaps)
        uint32_t* const sums = m.take<uint32_t>(2 * lines);
        uint32_t* const ws = m.take<uint32_t>(scan_ws_items(2 * lines));
        k_line_sums<<<grid_for(2 * lines, 256), 256, 0, st>>>((const int32_t*)ix->d_starts, (const int32_t*)ix->d_ends_sorted,
                                                              (uint32_t)n, (uint32_t)lines, sums);
        LAUNCH_CHECK();
        rc = device_excl_scan<uint32_t, uint32_t>(sums, 2 * lines, ix->d_line_sums, nullptr, ws, st);
        if (rc != SI_OK) return rc;
    }
    // 32-bit ends for the wave-cooperative walk of int64 indexes whose ends span < 2^32:
    // a third fewer bytes per position than ends + exitp at 8 + 4
    if constexpr (sizeof(S) == 8) {
        if ((uint64_t)back.info.end_hi - (uint64_t)back.info.end_lo < 0xFFFFFFFFull) {
            if (!(ix->d_ends32 = (uint32_t*)si_block_take(npad * sizeof(uint32_t), &ix->ends32_bytes, true)))
                return si_set_error(SI_ERR_NOMEM, "32-bit ends: %zu bytes", npad * sizeof(uint32_t));
            ix->ends32_base = back.info.end_lo;
            k_ends32<<<grid_for(npad, 256), 256, 0, st>>>((const int64_t*)ix->d_ends, n, npad, ix->ends32_base,
                                                           ix->d_ends32);
            LAUNCH_CHECK();
        }
    }
    {
        std::vector<int64_t> lens(back.lens, back.lens + LEN_SAMPLE);
        Carver m;
        m.base = (char*)scratch.p;
        m.used = shared_from;
        rc = build_long_list<S>(ix, lens, m, st);
        if (rc != SI_OK) return rc;
    }
    HIP_TRY(hipMemcpyAsync(&back.info, info, sizeof(BuildInfo), hipMemcpyDeviceToHost, st));
    HIP_TRY(hipStreamSynchronize(st));
    // intervals with start > end (queries on such an index take the walk, see siIndex)
    ix->n_inverted = (size_t)back.info.inverted;
    // A search in a bucket of m keys takes about log2(m) - 2 reads after the table's, one through the
    // 64-ary tree 14 (n > 4095 x 64): the tables are used unless half of the keys share a bucket
    // with more than 4096 others (what large batches do from 64 on: count_by_plan, bound_by_tree).
    const auto half = [&](int d) { return std::max(back.info.crowded[0][d], back.info.crowded[1][d]) > CROWD_SAMPLE / 2; };
    ix->ubt.ok = ix->ebt.ok = !back.info.unsorted && !half(2);
    ix->ubt.busy = ix->ebt.busy = half(1) ? 2 : half(0) ? 1 : 0;
    ix->built = true;
    ix->last_build_ms =
        std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count();
    return SI_OK;
}

}  // namespace

// ============================================================================
// C entry points
// ============================================================================
SI_EXPORT siIndex* siIndexCreate(int coord_bytes) {
    if (coord_bytes != 4 && coord_bytes != 8) {
        si_set_error(SI_ERR_ARG, "coord_bytes must be 4 or 8");
        return nullptr;
    }
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || ndev == 0) {
        si_set_error(SI_ERR_HIP, "no HIP device available");
        return nullptr;
    }
    siIndex* ix = new siIndex();
    ix->cb = coord_bytes;
    hipGetDevice(&ix->device);
    si_block_users(1);
    return ix;
}

SI_EXPORT void siIndexDestroy(siIndex* ix) {
    if (!ix) return;
    for (siLearned* m : ix->models) si_learned_forget_index(m);
    ix->release();
    ix->one.release();
    delete ix;
    si_block_users(-1);
}

static int index_build(siIndex* ix, const void* starts, const void* ends, const int32_t* values, size_t n,
                       int start_sorted, int end_sorted, int on_device, void* stream) {
    if (!ix) return si_set_error(SI_ERR_ARG, "null index");
    if (n && (!starts || !ends)) return si_set_error(SI_ERR_ARG, "null starts/ends");
    hipStream_t st = (hipStream_t)stream;
    int rc = ix->cb == 4 ? build_impl<int32_t>(ix, starts, ends, values, n, start_sorted, end_sorted, on_device, st)
                         : build_impl<int64_t>(ix, starts, ends, values, n, start_sorted, end_sorted, on_device, st);
    if (rc != SI_OK) ix->release();
    return rc;
}

SI_EXPORT int siIndexBuild(siIndex* ix, const void* starts, const void* ends, const int32_t* values,
                           size_t n, int start_sorted, int end_sorted, int on_device, void* stream) {
    return index_build(ix, starts, ends, values, n, start_sorted != 0, end_sorted != 0, on_device, stream);
}

SI_EXPORT int siIndexBuildDetect(siIndex* ix, const void* starts, const void* ends, const int32_t* values,
                                 size_t n, int start_sorted, int end_sorted, int on_device, void* stream) {
    return index_build(ix, starts, ends, values, n, start_sorted, end_sorted, on_device, stream);
}

SI_EXPORT size_t siIndexSize(const siIndex* ix) { return ix ? ix->n : 0; }
SI_EXPORT int siIndexCoordBytes(const siIndex* ix) { return ix ? ix->cb : 0; }
SI_EXPORT double siIndexLastBuildMs(const siIndex* ix) { return ix ? ix->last_build_ms : 0.0; }
SI_EXPORT const void* siIndexDeviceStarts(const siIndex* ix) { return ix ? ix->d_starts : nullptr; }
SI_EXPORT const void* siIndexDeviceEnds(const siIndex* ix) { return ix ? ix->d_ends : nullptr; }
SI_EXPORT const uint32_t* siIndexDeviceBranch(const siIndex* ix) { return ix ? ix->d_branch : nullptr; }
SI_EXPORT const uint32_t* siIndexDevicePerm(const siIndex* ix) { return ix ? ix->d_perm : nullptr; }

SI_EXPORT int siIndexDownload(const siIndex* ix, void* starts, void* ends, int32_t* values,
                              uint32_t* perm, uint64_t* branch) {
    int rc = check_ix(ix);
    if (rc) return rc;
    const size_t n = ix->n;
    if (n == 0) return SI_OK;
    if (values && !ix->d_values) return si_set_error(SI_ERR_ARG, "index was built without values");
    if (starts) HIP_TRY(hipMemcpy(starts, ix->d_starts, n * ix->cb, hipMemcpyDeviceToHost));
    if (ends) HIP_TRY(hipMemcpy(ends, ix->d_ends, n * ix->cb, hipMemcpyDeviceToHost));
    if (values) HIP_TRY(hipMemcpy(values, ix->d_values, n * 4, hipMemcpyDeviceToHost));
    if (perm) HIP_TRY(hipMemcpy(perm, ix->d_perm, n * 4, hipMemcpyDeviceToHost));
    if (branch) {
        std::vector<uint32_t> b(n);
        HIP_TRY(hipMemcpy(b.data(), ix->d_branch, n * 4, hipMemcpyDeviceToHost));
        for (size_t i = 0; i < n; ++i) branch[i] = (b[i] == NONE) ? UINT64_MAX : (uint64_t)b[i];
    }
    return SI_OK;
}

