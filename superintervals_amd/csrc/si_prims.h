// si_prims.h -- device primitives shared by the build and query translation units:
// wave/block scans and reductions, a three-kernel exclusive scan and a stable LSD
// radix sort of 64-bit keys with a 32-bit payload.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <vector>

#include "si_common.h"
#include "si_kernels.h"

#define HIP_TRY(expr)                                                                     \
    do {                                                                                  \
        hipError_t _e = (expr);                                                           \
        if (_e != hipSuccess)                                                             \
            return si_set_error(SI_ERR_HIP, "%s failed: %s (%s:%d)", #expr,               \
                                hipGetErrorString(_e), __FILE__, __LINE__);               \
    } while (0)

#define LAUNCH_CHECK() HIP_TRY(hipGetLastError())

namespace sik {
namespace {

inline unsigned grid_for(size_t n, unsigned per_block) {
    return (unsigned)((n + per_block - 1) / per_block);
}

// ============================================================================
// Wave / block primitives
// ============================================================================
template <typename T>
__device__ __forceinline__ T wave_incl_scan(T v) {
    const int lane = lane_id();
#pragma unroll
    for (int d = 1; d < WAVE; d <<= 1) {
        T t = __shfl_up(v, d, WAVE);
        if (lane >= d) v += t;
    }
    return v;
}

// Inclusive scan of a 32-bit value across the wave in six DPP adds: shifts by 1, 2, 4, 8
// within each row of 16 lanes (a lane with no source in its row adds 0, bound_ctrl), then
// row 0's total broadcast into rows 1 and 3 (row_bcast:15, rows 0 and 2 not written) and
// lane 31's into rows 2 and 3 (row_bcast:31).  A DPP source VGPR written by the previous
// VALU instruction needs two wait states, hence the s_nop 1 before each add.
__device__ __forceinline__ uint32_t wave_incl_scan_dpp(uint32_t v) {
    asm volatile(
        "s_nop 1\n\t"
        "v_add_u32_dpp %0, %0, %0 row_shr:1 row_mask:0xf bank_mask:0xf bound_ctrl:0\n\t"
        "s_nop 1\n\t"
        "v_add_u32_dpp %0, %0, %0 row_shr:2 row_mask:0xf bank_mask:0xf bound_ctrl:0\n\t"
        "s_nop 1\n\t"
        "v_add_u32_dpp %0, %0, %0 row_shr:4 row_mask:0xf bank_mask:0xf bound_ctrl:0\n\t"
        "s_nop 1\n\t"
        "v_add_u32_dpp %0, %0, %0 row_shr:8 row_mask:0xf bank_mask:0xf bound_ctrl:0\n\t"
        "s_nop 1\n\t"
        "v_add_u32_dpp %0, %0, %0 row_bcast:15 row_mask:0xa bank_mask:0xf\n\t"
        "s_nop 1\n\t"
        "v_add_u32_dpp %0, %0, %0 row_bcast:31 row_mask:0xc bank_mask:0xf\n\t"
        "s_nop 1"
        : "+v"(v));
    return v;
}

template <typename T>
__device__ __forceinline__ T wave_max(T v) {
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) {
        T t = __shfl_xor(v, d, WAVE);
        v = t > v ? t : v;
    }
    return v;
}

// Exclusive scan across a 256-thread block; *total receives the block sum.
template <typename T>
__device__ __forceinline__ T block_excl_scan256(T v, T* s_w /*[4]*/, T* total) {
    const int lane = lane_id(), w = threadIdx.x >> 6;
    T inc = wave_incl_scan(v);
    if (lane == WAVE - 1) s_w[w] = inc;
    __syncthreads();
    T pre = 0, tot = 0;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        T x = s_w[k];
        pre += (k < w) ? x : (T)0;
        tot += x;
    }
    __syncthreads();
    *total = tot;
    return pre + inc - v;
}

// ============================================================================
// Exclusive scan (reduce -> scan of tile sums -> downsweep), 4096 items per tile
// ============================================================================
constexpr int SCAN_THREADS = 256;
constexpr int SCAN_ITEMS = 16;
constexpr int SCAN_TILE = SCAN_THREADS * SCAN_ITEMS;

template <typename TI, typename TO>
__global__ __launch_bounds__(SCAN_THREADS) void k_scan_reduce(const TI* __restrict__ in, size_t n,
                                                              TO* __restrict__ tile_sums) {
    __shared__ TO s_w[4];
    size_t base = (size_t)blockIdx.x * SCAN_TILE;
    TO sum = 0;
#pragma unroll
    for (int k = 0; k < SCAN_ITEMS; ++k) {
        size_t i = base + (size_t)k * SCAN_THREADS + threadIdx.x;
        if (i < n) sum += (TO)in[i];
    }
    TO tot;
    block_excl_scan256<TO>(sum, s_w, &tot);
    if (threadIdx.x == 0) tile_sums[blockIdx.x] = tot;
}

// Single block: exclusive scan of nt tile sums in place; *grand receives the total.
template <typename TO>
__global__ __launch_bounds__(1024) void k_scan_tiles(TO* __restrict__ ts, size_t nt, TO* grand) {
    __shared__ TO s_part[1024];
    __shared__ TO s_carry;
    if (threadIdx.x == 0) s_carry = 0;
    __syncthreads();
    for (size_t base = 0; base < nt; base += 1024) {
        size_t i = base + threadIdx.x;
        TO v = (i < nt) ? ts[i] : (TO)0;
        // inclusive scan over 1024 threads: wave scan then wave totals
        TO inc = wave_incl_scan(v);
        const int lane = lane_id(), w = threadIdx.x >> 6;
        if (lane == WAVE - 1) s_part[w] = inc;
        __syncthreads();
        if (threadIdx.x < 16) {
            TO x = s_part[threadIdx.x];
            TO acc = 0;
            for (int k = 0; k < 16; ++k) {
                TO y = s_part[k];
                acc += (k < (int)threadIdx.x) ? y : (TO)0;
            }
            s_part[16 + threadIdx.x] = acc;
            (void)x;
        }
        __syncthreads();
        TO excl = s_carry + s_part[16 + w] + inc - v;
        __syncthreads();
        if (i < nt) ts[i] = excl;
        if (threadIdx.x == 1023) s_carry = excl + v;
        __syncthreads();
    }
    if (threadIdx.x == 0 && grand) *grand = s_carry;
}

// Downsweep: out[i] = tile prefix + exclusive scan within the tile.  Each thread owns
// SCAN_ITEMS consecutive items; the tile passes through LDS (one pad entry per 32 items)
// so that global loads and stores are coalesced across the wave.  A block reads and
// writes only its own tile, all reads before any write, so in and out may alias.
//
// SELF: tile_pre holds the tiles' sums, and every block adds up those before its own (a launch and
// 2.5 us less; one tile is scanned by this kernel alone).
constexpr size_t SCAN_SELF_TILES = 256;
template <typename TI, typename TO, bool SELF>
__global__ __launch_bounds__(SCAN_THREADS) void k_scan_down(const TI* in, size_t n,
                                                            const TO* __restrict__ tile_pre,
                                                            TO* out, TO* grand) {
    __shared__ TO s_w[4];
    __shared__ TO s_v[SCAN_TILE + SCAN_TILE / 32];
    const size_t tbase = (size_t)blockIdx.x * SCAN_TILE;
#pragma unroll
    for (int k = 0; k < SCAN_ITEMS; ++k) {
        const uint32_t li = (uint32_t)k * SCAN_THREADS + threadIdx.x;
        const size_t i = tbase + li;
        s_v[li + li / 32] = (i < n) ? (TO)in[i] : (TO)0;
    }
    __syncthreads();
    TO v[SCAN_ITEMS];
    TO sum = 0;
#pragma unroll
    for (int k = 0; k < SCAN_ITEMS; ++k) {
        const uint32_t li = threadIdx.x * SCAN_ITEMS + k;
        v[k] = s_v[li + li / 32];
        sum += v[k];
    }
    TO tot;
    TO run = block_excl_scan256<TO>(sum, s_w, &tot);
    if (SELF) {
        const TO mine = threadIdx.x < blockIdx.x ? tile_pre[threadIdx.x] : (TO)0;   // (blockIdx.x < SCAN_SELF_TILES)
        TO before;
        block_excl_scan256<TO>(mine, s_w, &before);
        run += before;
        if (grand && threadIdx.x == 0 && blockIdx.x == gridDim.x - 1) *grand = before + tot;
    } else {
        run += tile_pre[blockIdx.x];
    }
#pragma unroll
    for (int k = 0; k < SCAN_ITEMS; ++k) {
        const uint32_t li = threadIdx.x * SCAN_ITEMS + k;
        s_v[li + li / 32] = run;
        run += v[k];
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < SCAN_ITEMS; ++k) {
        const uint32_t li = (uint32_t)k * SCAN_THREADS + threadIdx.x;
        const size_t i = tbase + li;
        if (i < n) out[i] = s_v[li + li / 32];
    }
}

// Exclusive scan of n items (TI) into out (TO); out may alias in when TI == TO.
// If total != nullptr (device pointer) the grand total is stored there.
// ws must hold at least scan_ws_items(n) TO values.
constexpr size_t scan_ws_items(size_t n) { return (n + SCAN_TILE - 1) / SCAN_TILE + 1; }

template <typename TI, typename TO>
int device_excl_scan(const TI* in, size_t n, TO* out, TO* total, TO* ws, hipStream_t st) {
    if (n == 0) {
        if (total) HIP_TRY(hipMemsetAsync(total, 0, sizeof(TO), st));
        return SI_OK;
    }
    const size_t nt = (n + SCAN_TILE - 1) / SCAN_TILE;
    if (nt > 1) {
        k_scan_reduce<TI, TO><<<(unsigned)nt, SCAN_THREADS, 0, st>>>(in, n, ws);
        LAUNCH_CHECK();
    }
    if (nt <= SCAN_SELF_TILES) {
        k_scan_down<TI, TO, true><<<(unsigned)nt, SCAN_THREADS, 0, st>>>(in, n, ws, out, total);
        LAUNCH_CHECK();
        return SI_OK;
    }
    k_scan_tiles<TO><<<1, 1024, 0, st>>>(ws, nt, total);
    LAUNCH_CHECK();
    k_scan_down<TI, TO, false><<<(unsigned)nt, SCAN_THREADS, 0, st>>>(in, n, ws, out, nullptr);
    LAUNCH_CHECK();
    return SI_OK;
}

// ============================================================================
// Radix sort: stable LSD over 32- or 64-bit keys, with a 32-bit payload or none
// ============================================================================
constexpr int RS_THREADS = 256;
// 2048-item tiles: the scatter's LDS (keys, payloads, digit starts: 25 KB) lets six
// blocks share a CU; 4096-item tiles (two blocks) were 10 % slower per pass
#ifndef SI_RS_ROUNDS
#define SI_RS_ROUNDS 8
#endif
constexpr int RS_ROUNDS = SI_RS_ROUNDS;   // rounds of 256 items per tile
constexpr int RS_TILE = RS_THREADS * RS_ROUNDS;   // items per tile
constexpr int RS_BINS = 256;

// Which bits of a sort's keys vary: the kernel that writes (or reads) the keys leaves the AND and
// the OR of its block's in slots[2 * block], [2 * block + 1], and the host joins them.  A digit
// whose bits are all alike needs no pass.  (Histograms of every digit, in a pass of their own,
// said the same for 63 us of a 10M-key sort.)
constexpr unsigned RS_BITS_BLOCKS = 1024;   // most blocks of a kernel that leaves them
constexpr unsigned RS_BITS_ITEMS = 4;       // items a thread takes at a time in such a kernel
inline unsigned rs_bits_grid(size_t n) {
    return (unsigned)std::min<size_t>((n + RS_THREADS * RS_BITS_ITEMS - 1) / (RS_THREADS * RS_BITS_ITEMS), RS_BITS_BLOCKS);
}

__device__ __forceinline__ void rs_block_bits(uint64_t all_and, uint64_t all_or, uint64_t* __restrict__ slots) {
    __shared__ uint64_t s_and[RS_THREADS / WAVE], s_or[RS_THREADS / WAVE];
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) {
        all_and &= __shfl_xor(all_and, d, WAVE);
        all_or |= __shfl_xor(all_or, d, WAVE);
    }
    if (lane_id() == 0) {
        s_and[threadIdx.x >> 6] = all_and;
        s_or[threadIdx.x >> 6] = all_or;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < RS_THREADS / WAVE; ++w) {
            all_and &= s_and[w];
            all_or |= s_or[w];
        }
        slots[2 * blockIdx.x] = all_and;
        slots[2 * blockIdx.x + 1] = all_or;
    }
}

// Runs f(i) for the items i < n of this thread (a grid of rs_bits_grid(n) blocks), f returning
// item i's key, and leaves the block's bits in slots.
template <class F>
__device__ __forceinline__ void rs_each_key(size_t n, uint64_t* __restrict__ slots, F f) {
    uint64_t all_and = ~0ull, all_or = 0ull;
    const size_t step = (size_t)gridDim.x * (RS_THREADS * RS_BITS_ITEMS);
    for (size_t base = (size_t)blockIdx.x * (RS_THREADS * RS_BITS_ITEMS); base < n; base += step) {
#pragma unroll
        for (unsigned k = 0; k < RS_BITS_ITEMS; ++k) {
            const size_t i = base + k * RS_THREADS + threadIdx.x;
            if (i < n) {
                const uint64_t key = f(i);
                all_and &= key;
                all_or |= key;
            }
        }
    }
    rs_block_bits(all_and, all_or, slots);
}

// The bits of keys that are there already.
template <typename K>
__global__ __launch_bounds__(RS_THREADS) void k_rs_bits(const K* __restrict__ keys, size_t n, uint64_t* __restrict__ slots) {
    rs_each_key(n, slots, [&](size_t i) { return (uint64_t)keys[i]; });
}

// A pass's digit of a key.  flip = 0x80 on the top digit sorts the raw bits of signed numbers.
template <typename K>
__device__ __forceinline__ uint32_t rs_digit(K key, int shift, uint32_t flip) {
    return ((uint32_t)(key >> shift) & 255u) ^ flip;
}

// Sorts of at most this many tiles need no scan kernel: every scatter block adds up the tiles'
// counts itself (SELF), 256 coalesced counts a tile.  int32 plans, four passes: 30K queries (15 tiles)
// 53 us, with the scan kernel 62; 100K 62.6 and 64.1; 150K (73 tiles) 69 and 66; 250K 82 and 70.
constexpr uint32_t RS_SELF_TILES = 56;

// Per-tile digit counts, digit-major (th[d * ntiles + tile], for the scan), or tile-major (SELF:
// th[tile * 256 + d]).  A digit equal across a wave is added once, from one lane.
template <typename K, bool SELF>
__global__ __launch_bounds__(RS_THREADS) void k_rs_tile_hist(const K* __restrict__ keys,
                                                             size_t n, int shift, uint32_t flip,
                                                             uint32_t* __restrict__ th,
                                                             uint32_t ntiles) {
    __shared__ uint32_t h[RS_BINS];
    h[threadIdx.x] = 0;
    __syncthreads();
    size_t base = (size_t)blockIdx.x * RS_TILE;
#pragma unroll 4
    for (int r = 0; r < RS_ROUNDS; ++r) {
        const size_t i = base + (size_t)r * RS_THREADS + threadIdx.x;
        const bool valid = i < n;
        const uint64_t vm = __builtin_amdgcn_ballot_w64(valid);
        if (vm == 0ull) continue;   // wave-uniform
        const uint32_t digit = valid ? rs_digit(keys[i], shift, flip) : 0u;
        const uint32_t d0 = __builtin_amdgcn_readfirstlane(digit);   // lane 0's: valid whenever any is
        if (__builtin_amdgcn_ballot_w64(valid && digit == d0) == vm) {
            if (lane_id() == 0) atomicAdd(&h[d0], (uint32_t)__popcll(vm));
        } else if (valid) {
            atomicAdd(&h[digit], 1u);
        }
    }
    __syncthreads();
    th[SELF ? (size_t)blockIdx.x * RS_BINS + threadIdx.x : (size_t)threadIdx.x * ntiles + blockIdx.x] = h[threadIdx.x];
}

// Ranking of one tile of up to RS_TILE items held in registers (item r * 256 + tid in
// key[r]): off[r] receives the item's position among the tile's items of equal digit, in
// item order, and the return value is the tile's count of digit tid.  Each round of 256
// items finds, per wave, the lanes with equal digits by 8 ballots; the wave's leader of
// each digit records their number in s_c[round * 4 + wave][digit], and one column scan
// per digit over the 32 (round, wave) entries turns those numbers into each entry's start.
// s_c (RS_ROUNDS * 4 rows of RS_BINS 16-bit counts) must be free on entry; it is free
// again once every thread has passed a barrier after the call.
template <typename K>
__device__ __forceinline__ uint32_t rs_rank_tile(const K (&key)[RS_ROUNDS], uint32_t tile_n, int shift, uint32_t flip,
                                                 uint16_t (*s_c)[RS_BINS], uint32_t (&off)[RS_ROUNDS]) {
    const int tid = threadIdx.x, lane = lane_id(), w = tid >> 6;
    uint32_t* const s_c32 = reinterpret_cast<uint32_t*>(&s_c[0][0]);
#pragma unroll
    for (int k = 0; k < RS_ROUNDS * 4 * RS_BINS / 2 / RS_THREADS; ++k) s_c32[k * RS_THREADS + tid] = 0u;
    __syncthreads();
    const uint64_t lt_mask = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
#pragma unroll
    for (int r = 0; r < RS_ROUNDS; ++r) {
        const bool valid = (uint32_t)r * RS_THREADS + tid < tile_n;
        const uint32_t digit = rs_digit(key[r], shift, flip);
        uint64_t peers = __builtin_amdgcn_ballot_w64(valid);
#pragma unroll
        for (int b = 0; b < 8; ++b) {
            const uint64_t bal = __builtin_amdgcn_ballot_w64((digit >> b) & 1u);
            peers &= ((digit >> b) & 1u) ? bal : ~bal;
        }
        const uint32_t rank = (uint32_t)__popcll(peers & lt_mask);
        if (valid && rank == 0) s_c[r * 4 + w][digit] = (uint16_t)__popcll(peers);
        off[r] = rank;
    }
    __syncthreads();
    uint32_t run = 0;
#pragma unroll
    for (int k = 0; k < RS_ROUNDS * 4; ++k) {
        const uint32_t c = s_c[k][tid];
        s_c[k][tid] = (uint16_t)run;
        run += c;
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < RS_ROUNDS; ++r) off[r] += s_c[r * 4 + w][rs_digit(key[r], shift, flip)];
    return run;
}

// Where a scatter writes item (key, val) at position dst: the sort's buffers, or, in a
// sort's last pass, whatever arrays its caller wants the sorted items unpacked into.
struct ArrayOut {
    uint64_t* __restrict__ k;
    uint32_t* __restrict__ v;
    __device__ __forceinline__ void put(size_t dst, uint64_t key, uint32_t val) const {
        k[dst] = key;
        v[dst] = val;
    }
};

// The sort's buffer of a sort without payload.
template <typename K>
struct KeyOut {
    K* __restrict__ k;
    __device__ __forceinline__ void put(size_t dst, K key, uint32_t) const { k[dst] = key; }
};

// What a scatter moves beside the keys: a payload array, nothing, or the item's input position.
enum RsVals { RS_NONE = 0, RS_ARRAY = 1, RS_INDEX = 2 };

// Stable scatter of one tile (digit offsets from the scan of the per-tile digit counts, or, with
// SELF, from the counts themselves): the tile is ranked in registers, staged in LDS in digit order and written out so
// equal digits land contiguously.
template <class Out, typename K, RsVals VALS, bool SELF>
__global__ __launch_bounds__(RS_THREADS) void k_rs_scatter(
    const K* __restrict__ kin, const uint32_t* __restrict__ vin, Out out, size_t n, int shift, uint32_t flip,
    const uint32_t* __restrict__ th_base, const uint32_t* __restrict__ totals, uint32_t ntiles) {
    __shared__ union {
        uint16_t c[RS_ROUNDS * 4][RS_BINS];
        K key[RS_TILE];
    } s_u;
    __shared__ uint32_t s_val[VALS ? RS_TILE : 1];
    __shared__ uint32_t s_dstart[RS_BINS];
    __shared__ uint32_t s_gbase[RS_BINS];   // the tile's first output slot of each digit
    __shared__ uint32_t s_w[4];

    const int tid = threadIdx.x;
    const uint32_t tile = blockIdx.x;
    const size_t base = (size_t)tile * RS_TILE;
    const uint32_t tile_n = (uint32_t)min((size_t)RS_TILE, n - base);
    K key[RS_ROUNDS];
    uint32_t val[RS_ROUNDS], off[RS_ROUNDS];
#pragma unroll
    for (int r = 0; r < RS_ROUNDS; ++r) {
        const uint32_t li = (uint32_t)r * RS_THREADS + tid;
        key[r] = li < tile_n ? kin[base + li] : (K)0;
        val[r] = VALS == RS_INDEX ? (uint32_t)(base + li) : VALS == RS_ARRAY && li < tile_n ? vin[base + li] : 0u;
    }
    uint32_t tot;
    if (SELF) {   // this thread's digit: its items in the tiles before this one, and in all
        uint32_t before = 0, all = 0;
        for (uint32_t t = 0; t < ntiles; t += 8) {
            uint32_t c[8];
#pragma unroll
            for (uint32_t k = 0; k < 8; ++k) c[k] = t + k < ntiles ? th_base[(size_t)(t + k) * RS_BINS + tid] : 0u;
#pragma unroll
            for (uint32_t k = 0; k < 8; ++k) {
                all += c[k];
                before += t + k < tile ? c[k] : 0u;
            }
        }
        s_gbase[tid] = block_excl_scan256<uint32_t>(all, s_w, &tot) + before;
    } else {
        s_gbase[tid] = block_excl_scan256<uint32_t>(totals[tid], s_w, &tot) + th_base[(size_t)tid * ntiles + tile];
    }
    const uint32_t cnt = rs_rank_tile(key, tile_n, shift, flip, s_u.c, off);
    s_dstart[tid] = block_excl_scan256<uint32_t>(cnt, s_w, &tot);   // its barriers free s_u.c
    __syncthreads();
#pragma unroll
    for (int r = 0; r < RS_ROUNDS; ++r) {
        if ((uint32_t)r * RS_THREADS + tid < tile_n) {
            const uint32_t slot = s_dstart[rs_digit(key[r], shift, flip)] + off[r];
            s_u.key[slot] = key[r];
            if (VALS) s_val[slot] = val[r];
        }
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < RS_ROUNDS; ++r) {
        const uint32_t slot = (uint32_t)r * RS_THREADS + tid;
        if (slot < tile_n) {
            const K k = s_u.key[slot];
            const uint32_t digit = rs_digit(k, shift, flip);
            const size_t dst = (size_t)s_gbase[digit] + (slot - s_dstart[digit]);
            out.put(dst, k, VALS ? s_val[slot] : 0u);
        }
    }
}

// Exclusive scan of each digit's tile counts (digit-major, a block a digit) in place, and the digits'
// totals, which the scatter's blocks add up themselves.  (A scan over all the counts in three kernels:
// two launches and 35 us more for the passes of a 300K sort, 50 of 850 us for a 10M one.)
constexpr int DS_THREADS = 1024;
constexpr int DS_ITEMS = 4;
__global__ __launch_bounds__(DS_THREADS) void k_rs_digit_scan(uint32_t* __restrict__ th, uint32_t ntiles,
                                                              uint32_t* __restrict__ totals) {
    __shared__ uint32_t s_w[2][DS_THREADS / WAVE];
    uint32_t* const row = th + (size_t)blockIdx.x * ntiles;
    const uint32_t lane = (uint32_t)lane_id(), w = threadIdx.x >> 6;
    uint32_t carry = 0, par = 0;
    for (uint32_t base = 0; base < ntiles; base += DS_THREADS * DS_ITEMS, par ^= 1u) {
        uint32_t c[DS_ITEMS], sum = 0;
#pragma unroll
        for (int k = 0; k < DS_ITEMS; ++k) {
            const uint32_t i = base + threadIdx.x * DS_ITEMS + k;
            c[k] = i < ntiles ? row[i] : 0u;
            sum += c[k];
        }
        const uint32_t inc = wave_incl_scan(sum);
        if (lane == WAVE - 1) s_w[par][w] = inc;
        __syncthreads();
        uint32_t run = carry + inc - sum;
#pragma unroll
        for (uint32_t k = 0; k < DS_THREADS / WAVE; ++k) {
            const uint32_t x = s_w[par][k];
            run += k < w ? x : 0u;
            carry += x;
        }
#pragma unroll
        for (int k = 0; k < DS_ITEMS; ++k) {
            const uint32_t i = base + threadIdx.x * DS_ITEMS + k;
            if (i < ntiles) row[i] = run;
            run += c[k];
        }
    }
    if (threadIdx.x == 0) totals[blockIdx.x] = carry;
}

// Temporary device memory of a radix sort of n items (rs_temp_bytes).
struct RsTemp {
    uint64_t* bits;    // AND and OR of the keys, per block (rs_each_key)
    uint32_t* th;      // per-tile digit counts
    uint32_t* totals;  // of the digits
};

constexpr size_t rs_ntiles(size_t n) { return (n + RS_TILE - 1) / RS_TILE; }

constexpr size_t align256(size_t b) { return (b + 255) & ~(size_t)255; }

constexpr size_t rs_temp_bytes(size_t n) {
    const size_t nth = rs_ntiles(n) * RS_BINS;
    return RS_BITS_BLOCKS * 16 + align256(nth * 4) + RS_BINS * 4;
}

inline RsTemp rs_temp_carve(void* base, size_t n) {
    const size_t nth = rs_ntiles(n) * RS_BINS;
    char* p = (char*)base;
    RsTemp t;
    t.bits = (uint64_t*)p; p += RS_BITS_BLOCKS * 16;
    t.th = (uint32_t*)p; p += align256(nth * 4);
    t.totals = (uint32_t*)p;
    return t;
}

__global__ void k_zero_u32(uint32_t* __restrict__ p, size_t n) {
    size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0;
}

__global__ void k_zero_u64(uint64_t* __restrict__ p, size_t n) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0;
}

// The bits that vary over n > 0 keys, from what a grid of rs_bits_grid(n) blocks has left in
// tmp.bits (one read-back; synchronises the stream).
inline int rs_varying_bits(size_t n, const RsTemp& tmp, uint64_t* varying, hipStream_t st) {
    uint64_t slots[2 * RS_BITS_BLOCKS];
    const unsigned nb = rs_bits_grid(n);
    HIP_TRY(hipMemcpyAsync(slots, tmp.bits, (size_t)nb * 16, hipMemcpyDeviceToHost, st));
    HIP_TRY(hipStreamSynchronize(st));
    uint64_t all_and = ~0ull, all_or = 0ull;
    for (unsigned b = 0; b < nb; ++b) {
        all_and &= slots[2 * b];
        all_or |= slots[2 * b + 1];
    }
    *varying = all_and ^ all_or;
    return SI_OK;
}

// ---- sorts of one workgroup
// Batches of a few thousand keys are sorted by one workgroup in LDS, with the digits to sort by
// found on the way: the passes of the kernels above are two launches each, and a read-back of the
// varying bits stands before them.  A wave holds ITEMS consecutive lines of 64 items in registers;
// a pass ranks them by ballots, a line at a time, against its own counts of each digit, a column
// scan over the waves' counts and a scan over the digits make the positions, and the items move
// through LDS.  Bound by one CU's chain of passes, four for int32 (4 us each at 4096 items): plan of 500
// int32 queries 12 us (78 before), 4096 23 (78), 8192 36 (82; by the passes above without a
// read-back 49); of 16384 by this sort 67, by the passes 50.  int64: 4096 26 us, 8192 42.
constexpr int RS1_THREADS = 1024;
constexpr int RS1_WAVES = RS1_THREADS / WAVE;
constexpr size_t RS1_MAX = 8 * RS1_THREADS;

// in.key(i): the key of input item i (ordered as an unsigned number); out.put(position, key, i).
template <typename K, int ITEMS, class In, class Out>
__global__ __launch_bounds__(RS1_THREADS) void k_rs_one(In in, Out out, uint32_t n, int digit_lo, int digit_hi) {
    __shared__ K s_key[RS1_THREADS * ITEMS];
    __shared__ uint16_t s_item[RS1_THREADS * ITEMS];
    __shared__ uint16_t s_h[RS1_WAVES][RS_BINS];   // a wave's items of each digit, then those of the waves before
    __shared__ uint32_t s_base[RS_BINS];           // items of the smaller digits
    __shared__ K s_and[RS1_WAVES], s_or[RS1_WAVES];
    const uint32_t lane = (uint32_t)lane_id(), w = threadIdx.x >> 6, x0 = w * (WAVE * ITEMS) + lane;
    K key[ITEMS];
    uint32_t item[ITEMS], rank[ITEMS];
    K all_and = (K)~(K)0, all_or = 0;
#pragma unroll
    for (int r = 0; r < ITEMS; ++r) {
        const uint32_t x = x0 + (uint32_t)r * WAVE;
        item[r] = x;
        key[r] = x < n ? in.key(x) : (K)0;
        all_and &= x < n ? key[r] : (K)~(K)0;
        all_or |= key[r];
    }
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) {
        all_and &= __shfl_xor(all_and, d, WAVE);
        all_or |= __shfl_xor(all_or, d, WAVE);
    }
    if (lane == 0) {
        s_and[w] = all_and;
        s_or[w] = all_or;
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < RS1_WAVES; ++k) {
        all_and &= s_and[k];
        all_or |= s_or[k];
    }
    const K varying = all_and ^ all_or;   // the same in every thread
    for (int d = digit_lo; d < digit_hi; ++d) {
        if (((uint32_t)(varying >> (8 * d)) & 255u) == 0u) continue;
        // ranks within the wave
        uint32_t* const h32 = reinterpret_cast<uint32_t*>(s_h[w]);
        h32[lane] = 0u;
        h32[lane + WAVE] = 0u;
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
#pragma unroll
        for (int r = 0; r < ITEMS; ++r) {
            const bool valid = x0 + (uint32_t)r * WAVE < n;
            const uint32_t digit = (uint32_t)(key[r] >> (8 * d)) & 255u;
            uint64_t peers = __builtin_amdgcn_ballot_w64(valid);
#pragma unroll
            for (int b = 0; b < 8; ++b) {
                const uint64_t bal = __builtin_amdgcn_ballot_w64((digit >> b) & 1u);
                peers &= ((digit >> b) & 1u) ? bal : ~bal;
            }
            const uint32_t below = __builtin_amdgcn_mbcnt_hi((uint32_t)(peers >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)peers, 0u));
            const uint32_t before = s_h[w][digit];
            rank[r] = before + below;
            __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
            if (valid && below == 0u) s_h[w][digit] = (uint16_t)(before + (uint32_t)__popcll(peers));
            __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
        }
        __syncthreads();
        if (threadIdx.x < RS_BINS) {   // over the waves, a digit a thread
            uint32_t c[RS1_WAVES], run = 0;
#pragma unroll
            for (int k = 0; k < RS1_WAVES; ++k) c[k] = s_h[k][threadIdx.x];
#pragma unroll
            for (int k = 0; k < RS1_WAVES; ++k) {
                s_h[k][threadIdx.x] = (uint16_t)run;
                run += c[k];
            }
            s_base[threadIdx.x] = run;
        }
        __syncthreads();
        if (w == 0) {   // over the digits, four a lane
            uint32_t c[4], sum = 0;
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                c[k] = s_base[4u * lane + k];
                sum += c[k];
            }
            uint32_t run = sum;
#pragma unroll
            for (int o = 1; o < WAVE; o <<= 1) {
                const uint32_t y = __shfl_up(run, o, WAVE);
                run += lane >= (uint32_t)o ? y : 0u;
            }
            run -= sum;
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                s_base[4u * lane + k] = run;
                run += c[k];
            }
        }
        __syncthreads();
#pragma unroll
        for (int r = 0; r < ITEMS; ++r) {
            const uint32_t digit = (uint32_t)(key[r] >> (8 * d)) & 255u;
            const uint32_t to = s_base[digit] + s_h[w][digit] + rank[r];
            if (x0 + (uint32_t)r * WAVE < n) {
                s_key[to] = key[r];
                s_item[to] = (uint16_t)item[r];
            }
        }
        __syncthreads();
#pragma unroll
        for (int r = 0; r < ITEMS; ++r) {
            const uint32_t x = x0 + (uint32_t)r * WAVE;
            if (x < n) {
                key[r] = s_key[x];
                item[r] = s_item[x];
            }
        }
    }
#pragma unroll
    for (int r = 0; r < ITEMS; ++r) {
        const uint32_t x = x0 + (uint32_t)r * WAVE;
        if (x < n) out.put(x, key[r], item[r]);
    }
}

// Stable sort of n <= RS1_MAX items by the key digits [digit_lo, digit_hi), through out.
template <typename K, class In, class Out>
int rs_sort_one(const In& in, const Out& out, size_t n, int digit_lo, int digit_hi, hipStream_t st) {
    const uint32_t m = (uint32_t)n;
    if (n <= 1 * RS1_THREADS) k_rs_one<K, 1><<<1, RS1_THREADS, 0, st>>>(in, out, m, digit_lo, digit_hi);
    else if (n <= 2 * RS1_THREADS) k_rs_one<K, 2><<<1, RS1_THREADS, 0, st>>>(in, out, m, digit_lo, digit_hi);
    else if (n <= 4 * RS1_THREADS) k_rs_one<K, 4><<<1, RS1_THREADS, 0, st>>>(in, out, m, digit_lo, digit_hi);
    else k_rs_one<K, 8><<<1, RS1_THREADS, 0, st>>>(in, out, m, digit_lo, digit_hi);
    LAUNCH_CHECK();
    return SI_OK;
}

// True when digit d holds a bit that varies.
inline bool rs_digit_varies(uint64_t varying, int d) { return ((varying >> (8 * d)) & 255u) != 0; }

// One pass by the digit at `shift`: counts per tile, their scan, the scatter through out.
template <typename K, RsVals VALS, class Out>
int rs_pass(const K* kin, const uint32_t* vin, const Out& out, size_t n, int shift, uint32_t flip, const RsTemp& tmp,
            hipStream_t st) {
    const uint32_t ntiles = (uint32_t)rs_ntiles(n);
    if (ntiles <= RS_SELF_TILES) {
        k_rs_tile_hist<K, true><<<ntiles, RS_THREADS, 0, st>>>(kin, n, shift, flip, tmp.th, ntiles);
        LAUNCH_CHECK();
        k_rs_scatter<Out, K, VALS, true><<<ntiles, RS_THREADS, 0, st>>>(kin, vin, out, n, shift, flip, tmp.th, tmp.totals, ntiles);
        LAUNCH_CHECK();
        return SI_OK;
    }
    k_rs_tile_hist<K, false><<<ntiles, RS_THREADS, 0, st>>>(kin, n, shift, flip, tmp.th, ntiles);
    LAUNCH_CHECK();
    k_rs_digit_scan<<<RS_BINS, DS_THREADS, 0, st>>>(tmp.th, ntiles, tmp.totals);
    LAUNCH_CHECK();
    k_rs_scatter<Out, K, VALS, false><<<ntiles, RS_THREADS, 0, st>>>(kin, vin, out, n, shift, flip, tmp.th, tmp.totals,
                                                                    ntiles);
    LAUNCH_CHECK();
    return SI_OK;
}

// Ascending sort of n signed numbers given by their raw bits, by the digits with a bit of
// `varying` (at least one): in -> out, through the buffers k0 and k1.  in is not written; out may
// not be in, k0 or k1.
template <typename K>
int radix_sort_signed(const K* in, K* k0, K* k1, K* out, size_t n, uint64_t varying, const RsTemp& tmp,
                      hipStream_t st) {
    int last_d = -1;
    for (int d = 0; d < (int)sizeof(K); ++d)
        if (rs_digit_varies(varying, d)) last_d = d;
    const K* src = in;
    for (int d = 0; d <= last_d; ++d) {
        if (!rs_digit_varies(varying, d)) continue;
        const uint32_t flip = (d == (int)sizeof(K) - 1) ? 0x80u : 0u;
        K* const dst = (d == last_d) ? out : k0;
        const int rc = rs_pass<K, RS_NONE>(src, (const uint32_t*)nullptr, KeyOut<K>{dst}, n, 8 * d, flip, tmp, st);
        if (rc != SI_OK) return rc;
        src = dst;
        std::swap(k0, k1);
    }
    return SI_OK;
}

// Stable sort of (keys, vals) by key digits [digit_lo, digit_hi) (8-bit digits, least significant
// first) that hold a bit of `varying` (rs_varying_bits, or all of them, which needs no read-back,
// so that the sort can be captured in a graph).  tmp comes from rs_temp_carve.  On return
// *keys_sorted / *vals_sorted point at whichever buffer holds the result.
// With last (optional), the last pass run writes the sorted items through it instead of
// into the buffers, and *last_written says whether one ran; only if none ran are the
// items in *keys_sorted / *vals_sorted.
template <class LastOut = ArrayOut>
int radix_sort_pairs(uint64_t* k0, uint32_t* v0, uint64_t* k1, uint32_t* v1, size_t n,
                     int digit_lo, int digit_hi, const RsTemp& tmp, uint64_t** keys_sorted,
                     uint32_t** vals_sorted, hipStream_t st, uint64_t varying = ~0ull,
                     const LastOut* last = nullptr, bool* last_written = nullptr) {
    if (last_written) *last_written = false;
    *keys_sorted = k0;
    *vals_sorted = v0;
    if (n < 2) return SI_OK;

    uint64_t *ka = k0, *kb = k1;
    uint32_t *va = v0, *vb = v1;
    int last_d = -1;
    for (int d = digit_lo; d < digit_hi; ++d)
        if (rs_digit_varies(varying, d)) last_d = d;
    for (int d = digit_lo; d < digit_hi; ++d) {
        if (!rs_digit_varies(varying, d)) continue;
        int rc;
        if (last && d == last_d) {
            rc = rs_pass<uint64_t, RS_ARRAY>(ka, va, *last, n, 8 * d, 0u, tmp, st);
            if (last_written) *last_written = true;
        } else {
            rc = rs_pass<uint64_t, RS_ARRAY>(ka, va, ArrayOut{kb, vb}, n, 8 * d, 0u, tmp, st);
        }
        if (rc != SI_OK) return rc;
        std::swap(ka, kb);
        std::swap(va, vb);
    }
    *keys_sorted = ka;
    *vals_sorted = va;
    return SI_OK;
}

}  // namespace
}  // namespace sik
