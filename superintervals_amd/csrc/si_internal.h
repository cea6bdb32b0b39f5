// si_internal.h -- the device index object shared by the library's translation units.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <mutex>
#include <vector>

#include "si_common.h"
#include "si_kernels.h"

using namespace sik;

// ---- device blocks kept between uses ---------------------------------------------------------
// The driver clears freed device memory before it hands it out again, at about 40 GB/s: an
// index built over and over (600 MB of arrays and scratch for 10M intervals) ran at 15 ms a
// build once the card's cleared memory was used up, against 2.2 ms with the blocks kept.  Blocks
// the library is done with are therefore kept for its next one, at most BLOCK_KEEP bytes in all
// and only while an index exists; a block is handed out to one owner at a time, from any thread.
constexpr size_t BLOCK_KEEP = (size_t)2 << 30;
// A block of at least `bytes` bytes on the current device (null when there is no memory);
// *got receives its size, to be given back with it: at most an eighth more for memory that stays
// with an index (lasting), at most twice as much for what a call gives back at its end.
void* si_block_take(size_t bytes, size_t* got, bool lasting = false);
// hipMalloc and hipMallocAsync; when there is no memory the current device's kept blocks are freed
// and it is tried again (not while the stream is captured, where freeing would end the capture).
hipError_t si_malloc(void** p, size_t bytes);
hipError_t si_malloc_async(void** p, size_t bytes, hipStream_t st);
// Gives a block back: with quiet, nothing on its device uses it any more; otherwise it is freed
// (which waits).
void si_block_give(void* p, size_t bytes, int device, bool quiet);
// Waits for a device; false when that was not possible (a stream is being captured).
bool si_device_quiet(int device);
// An index of the library was created (+1) or destroyed (-1); the last one takes the kept
// blocks with it.
void si_block_users(int change);

// Search tree over a sorted key array: level l + 1 holds every 64th key of level l
// (level 0 = the keys themselves) up to a top level of at most 4095 keys, which is also
// kept in Eytzinger (breadth-first) order with max(S) padding to 2^top_h - 1 keys.  Both lie
// in the index's block.
struct KeyTree {
    void* d_lv = nullptr;            // levels 1 .. nlv, contiguous
    void* d_top = nullptr;
    int nlv = 0;                     // levels above the keys
    size_t lv_off[MAX_LEVELS] = {0}; // element offsets of levels 1 .. nlv in d_lv
    uint32_t lv_size[MAX_LEVELS] = {0};
    uint32_t top_size = 0, top_h = 0;

    void release() {
        d_lv = d_top = nullptr;
        nlv = 0;
        top_size = top_h = 0;
    }
};

// Bucket table over a sorted key array (BucketView), in the index's block.
struct BucketTable {
    uint32_t* d_tab = nullptr;
    bool ok = false;          // false: too many keys share a bucket, the search trees are used
    int busy = 0;             // 1, 2: half of the keys share a bucket with more than 64, 512 others or so
    int64_t lo = 0, hi = 0;
    uint32_t shift = 0;
    void release() {
        d_tab = nullptr;
        ok = false;
        busy = 0;
    }
    template <typename S>
    BucketView<S> view() const { return BucketView<S>{ok ? d_tab : nullptr, (S)lo, (S)hi, shift}; }
};

// Pinned host memory that the host-buffer calls copy through, STAGE_SLOTS chunks in turn with an
// event each.  4.9 MB of results (100K queries on 1M intervals) came to pageable memory in 265 us,
// now in about 170, bound by one core's copy out of the chunks (with streaming stores; 200 without).
// The whole call 700 us -> 415, for 195 MB of results 14.4 ms -> 6.9.  Chunks of 1 and 4 MB: within
// 10 %.  Taken by a call and given back, at most STAGE_KEEP kept until the last index is destroyed.
constexpr size_t STAGE_CHUNK = (size_t)2 << 20;
constexpr int STAGE_SLOTS = 4;
constexpr size_t STAGE_KEEP = 4;
struct HostStage {
    char* p = nullptr;                       // STAGE_SLOTS chunks, then 256 bytes for a flag
    hipEvent_t ev[STAGE_SLOTS] = {};
    bool busy[STAGE_SLOTS] = {};             // the slot's event is recorded and not waited for
    int device = 0;
};
HostStage* si_stage_take();                  // null: none to be had
void si_stage_give(HostStage* s);            // (no copy through it is under way)

// Scratch of the single-query calls (the host-buffer forms with one query): a pinned host
// buffer mapped into the device, which the one-wave kernel writes directly (header + up to
// cap results), and a stream.  Made on the first such call, kept until the index is
// destroyed; the last query's results stay in it, so a repeated identical call (a caller
// that sized its buffer from the first) is answered without a launch.
struct OneQuery {
    std::mutex mu;
    void* h = nullptr;          // pinned host memory: [0] total, [1] the last finished call's seq, then cap uint32 results
    uint64_t seq = 0;           // calls launched
    void* d = nullptr;          // its device address
    hipStream_t st = nullptr;
    uint64_t cap = 0;
    bool last_valid = false;
    int last_mode = -1;
    int64_t last_s = 0, last_e = 0;
    uint64_t last_total = 0;
    // Makes the scratch for `results` results when it is not there: all of it or, on an error, nothing
    // (the next call tries again).
    int make(uint64_t results) {
        if (cap) return SI_OK;
        const char* what = "hipHostMalloc";
        hipError_t e = hipHostMalloc(&h, 16 + results * 4, hipHostMallocMapped);
        if (e != hipSuccess) h = nullptr;
        if (e == hipSuccess) e = hipHostGetDevicePointer(&d, h, 0), what = "hipHostGetDevicePointer";
        if (e == hipSuccess) e = hipStreamCreateWithFlags(&st, hipStreamNonBlocking), what = "hipStreamCreateWithFlags";
        if (e != hipSuccess) {
            (void)hipGetLastError();
            release();
            return si_set_error(SI_ERR_HIP, "single-query scratch: %s: %s", what, hipGetErrorString(e));
        }
        ((uint64_t*)h)[1] = 0;   // (may hold what an earlier index left there)
        seq = 0;
        cap = results;
        return SI_OK;
    }
    void release() {
        if (st) (void)hipStreamSynchronize(st);   // (a call ends before its kernel does)
        if (h) (void)hipHostFree(h);
        if (st) (void)hipStreamDestroy(st);
        h = d = nullptr;
        st = nullptr;
        cap = 0;
        last_valid = false;
    }
};

// The long list of an index (LongView): device arrays and the max tree over its ends, in two
// blocks.
struct LongList {
    void* d_block = nullptr;
    size_t block_bytes = 0;
    size_t lrank_bytes = 0;       // d_lrank is a block of its own (it is there before the list's size is known)
    int64_t len = 0;              // threshold; 0 = no list
    uint32_t n = 0;
    uint32_t* d_pos = nullptr;    // n, padded to 64 entries
    void* d_ends = nullptr;       // n, padded with the minimum
    uint32_t* d_ends32 = nullptr; // int64 indexes with a 32-bit copy of the ends
    uint32_t* d_lrank = nullptr;  // index size + 1
    void* d_tree = nullptr;       // levels 1.. of the max tree over d_ends
    int nlev = 0;
    size_t lvl_off[MAX_LEVELS] = {0};
    uint32_t lvl_size[MAX_LEVELS] = {0};
    void release(int device, bool quiet) {
        if (d_block) si_block_give(d_block, block_bytes, device, quiet);
        if (d_lrank) si_block_give(d_lrank, lrank_bytes, device, quiet);
        d_block = nullptr;
        d_pos = d_ends32 = d_lrank = nullptr;
        d_ends = d_tree = nullptr;
        len = 0;
        n = 0;
        nlev = 0;
    }
};

// ============================================================================
// siIndex
// ============================================================================
struct siIndex {
    int cb = 4;
    size_t n = 0;
    bool built = false;
    int device = 0;
    void* d_block = nullptr;   // one block: the arrays below but for d_ends32 and the long list
    size_t block_bytes = 0;
    size_t ends32_bytes = 0;
    void* d_starts = nullptr;
    void* d_ends = nullptr;
    uint32_t* d_branch = nullptr;
    uint32_t* d_exit = nullptr;      // line exit targets (IndexView::exitp)
    uint32_t* d_perm = nullptr;
    int32_t* d_values = nullptr;
    void* d_tree = nullptr;   // levels 1.. of the max tree, contiguous
    void* d_ends_sorted = nullptr;   // ends in ascending order (rank count)
    uint32_t* d_ends32 = nullptr;    // int64 only, ends - ends32_base when they span < 2^32
    int64_t ends32_base = 0;
    // int32 only (coverage): d_line_sums[k] = sum of starts[0 .. 16 k), and from entry
    // sum_lines() on the same over the sorted ends plus a constant, modulo 2^32
    uint32_t* d_line_sums = nullptr;
    size_t sum_lines() const { return n / 16 + 1; }
    // intervals with start > end: the rank form of count and the guaranteed-hit run
    // [first start >= s, upper_bound] both assume start <= end, so queries on an index
    // holding any such interval take the walk
    size_t n_inverted = 0;
    // the learned position model trained on this build (siLearnedTrain attaches it,
    // siLearnedDestroy and the next build detach it); generation counts builds
    siLearned* learned = nullptr;
    uint64_t generation = 0;
    std::vector<siLearned*> models;   // every model created on this index (siIndexDestroy unlinks them)
    OneQuery one;                     // single-query scratch (see OneQuery)
    LongList lng;                     // intervals longer than a threshold (LongView)
    KeyTree ub;   // search tree over the starts (upper_bound)
    KeyTree eb;   // search tree over the sorted ends (rank count)
    BucketTable ubt, ebt;   // bucket tables over the same
    int nlev = 0;
    size_t lvl_off[MAX_LEVELS] = {0};   // element offsets into d_tree (level >= 1)
    uint32_t lvl_size[MAX_LEVELS] = {0};
    double last_build_ms = 0.0;

    void release() {
        const bool quiet = d_block && si_device_quiet(device);   // as freeing would: calls in flight end
        if (d_block) si_block_give(d_block, block_bytes, device, quiet);
        if (d_ends32) si_block_give(d_ends32, ends32_bytes, device, quiet);
        d_block = nullptr;
        d_starts = d_ends = d_tree = d_ends_sorted = nullptr;
        d_ends32 = nullptr;
        ends32_base = 0;
        n_inverted = 0;
        learned = nullptr;
        one.last_valid = false;   // the cached last query belongs to the old build
        lng.release(device, quiet);
        ++generation;
        ub.release();
        eb.release();
        ubt.release();
        ebt.release();
        d_branch = d_exit = d_perm = d_line_sums = nullptr;
        d_values = nullptr;
        n = 0;
        nlev = 0;
        built = false;
    }

    template <typename S>
    IndexView<S> view() const {
        IndexView<S> v;
        v.starts = (const S*)d_starts;
        v.ends = (const S*)d_ends;
        v.branch = d_branch;
        v.exitp = d_exit;
        v.ends32 = d_ends32;
        v.ends32_base = ends32_base;
        v.n = (uint32_t)n;
        v.npad = (uint32_t)((n + 63) & ~(size_t)63);
        return v;
    }

    template <typename S>
    LongView<S> long_view() const {
        LongView<S> v;
        v.pos = lng.d_pos;
        v.ends = (const S*)lng.d_ends;
        v.ends32 = lng.d_ends32;
        v.ends32_base = ends32_base;
        v.lrank = lng.d_lrank;
        v.len = lng.len;
        v.n = lng.n;
        v.td.nlev = lng.nlev;
        v.td.lvl[0] = (const S*)lng.d_ends;
        v.td.size[0] = lng.n;
        for (int l = 1; l < lng.nlev; ++l) {
            v.td.lvl[l] = (const S*)lng.d_tree + lng.lvl_off[l];
            v.td.size[l] = lng.lvl_size[l];
        }
        for (int l = (lng.nlev > 0 ? lng.nlev : 1); l < MAX_LEVELS; ++l) { v.td.lvl[l] = nullptr; v.td.size[l] = 0; }
        return v;
    }

    template <typename S>
    TreeDesc<S> tree() const {
        TreeDesc<S> t;
        t.nlev = nlev;
        t.lvl[0] = (const S*)d_ends;
        t.size[0] = (uint32_t)n;
        for (int l = 1; l < nlev; ++l) {
            t.lvl[l] = (const S*)d_tree + lvl_off[l];
            t.size[l] = lvl_size[l];
        }
        for (int l = nlev; l < MAX_LEVELS; ++l) { t.lvl[l] = nullptr; t.size[l] = 0; }
        return t;
    }
};

inline int check_ix(const siIndex* ix) {
    if (!ix) return si_set_error(SI_ERR_ARG, "null index");
    if (!ix->built) return si_set_error(SI_ERR_NOT_BUILT, "index has not been built");
    return SI_OK;
}
