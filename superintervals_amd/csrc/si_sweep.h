// si_sweep.h -- the fill pass as a sweep over query starts (included by si_query.hip).
//
// A query's hits are the run [lower_bound(s), upper_bound(e)], every position of which
// starts inside the query, and, below it, the positions p < lower_bound(s) with ends[p] >= s:
// the intervals that hold the point s.  That second set changes little between queries with
// neighbouring starts, so a wave takes a chunk of the plan's queries, orders them by start and
// carries the set along as a list in registers instead of walking down from every query:
//
//   window  the 64 positions [wbase, wbase + 64) that hold lower_bound - 1, one per lane;
//   list    the positions below wbase whose end reached the chunk's current start when they
//           were last looked at, ascending, at most SW_CAP of them, four registers per lane.
//
// A query then costs one compare and ballot per register and one store per register with
// hits, each covering consecutive output slots; its run is written 64 values a store.  When
// the starts leave the window, the survivors of list and window are packed together through
// LDS and the next line of ends becomes the window; a chunk's first query, and a query more
// than SW_GAP lines past the window, collects its list through the max tree (the lines with
// an end that reaches s, highest first).
//
// Where many queries with few hits share a window (SW_FEW), each lane answers its own: the
// wave goes through the window's and the list's entries once for all of them.
//
// What bounds it: on 10M int32 intervals x 10M queries (122 hits a query) it issues 33 vector
// and 39 scalar instructions a query, where the line walk with its shared emission chunks
// issued 140 and 62, and takes 2.44 ms (3.65 ms before), 2.0 TB/s of positions.  What is left is
// the writes: lists of 488 bytes that start anywhere leave two lines partly written each (the
// same segments aligned to 256 bytes are written in 0.8 ms by a kernel that does nothing else,
// unaligned in 1.8 ms).  100K queries on 10M: 66 us (143), 1M: 276 us (656), 4096: 14 us (111);
// 3M queries with 1.2 hits each on 100K intervals: 108 us (116).
//
// A query is left to k_sweep_shared, which continues below the run, when more than SW_CAP intervals
// hold its start, and when it ends below its own start's lower bound (start > end).
#pragma once

constexpr int SW_THREADS = 256;
constexpr int SW_WAVES = SW_THREADS / WAVE;
constexpr int SW_REGS = 4;                        // list registers per lane
constexpr uint32_t SW_CAP = SW_REGS * WAVE;       // entries of a list
constexpr uint32_t SW_CHUNK = 256;                // most queries of a wave
constexpr uint32_t SW_GAP = 8;                    // lines walked one by one before a list is collected anew

__device__ __forceinline__ uint32_t lanes_below(uint64_t m) {
    return __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
}

// A value that is the same in every lane, in a scalar register (the compiler takes values that
// leave a loop with ballots for lane-dependent ones; what they steer would then run on masks).
__device__ __forceinline__ uint32_t uniform(uint32_t v) { return (uint32_t)__builtin_amdgcn_readfirstlane((int)v); }

__device__ __forceinline__ int32_t read_lane(int32_t v, uint32_t l) { return __builtin_amdgcn_readlane(v, l); }
__device__ __forceinline__ uint32_t read_lane(uint32_t v, uint32_t l) {
    return (uint32_t)__builtin_amdgcn_readlane((int)v, l);
}
__device__ __forceinline__ uint64_t read_lane(uint64_t v, uint32_t l) {
    return (uint64_t)read_lane((uint32_t)(v >> 32), l) << 32 | read_lane((uint32_t)v, l);
}
__device__ __forceinline__ int64_t read_lane(int64_t v, uint32_t l) { return (int64_t)read_lane((uint64_t)v, l); }

// Ascending bitonic sort of 64 * NR keys, element r * 64 + lane in k[r].
template <int NR>
__device__ __forceinline__ void wave_sort(uint32_t (&k)[NR], int lane) {
#pragma unroll
    for (int K = 2; K <= WAVE * NR; K <<= 1) {
#pragma unroll
        for (int J = K >> 1; J >= 1; J >>= 1) {
            if (J >= WAVE) {
#pragma unroll
                for (int r = 0; r < NR; ++r) {
                    const int p = r | (J / WAVE);
                    if (p != r) {
                        const bool up = ((r * WAVE) & K) == 0;
                        const uint32_t lo = min(k[r], k[p]), hi = max(k[r], k[p]);
                        k[r] = up ? lo : hi;
                        k[p] = up ? hi : lo;
                    }
                }
            } else {
#pragma unroll
                for (int r = 0; r < NR; ++r) {
                    const uint32_t o = __shfl_xor(k[r], J, WAVE);
                    const bool up = ((r * WAVE + lane) & K) == 0, first = (lane & J) == 0;
                    k[r] = (up == first) ? min(k[r], o) : max(k[r], o);
                }
            }
        }
    }
}

// The positions below line `line0` (64 positions a line) with an end >= s, descending, at
// l_end / l_pay[0 .. n); returns n, or a number above SW_CAP when there are more (the entries
// are then incomplete).  The payload is the position, or its value.
template <typename S, bool VALUES>
__device__ __forceinline__ uint32_t collect_holding(const S* __restrict__ ends, const int32_t* __restrict__ vals,
                                                    const TreeDesc<S>& td, uint32_t line0, S s, int lane,
                                                    S* __restrict__ l_end, uint32_t* __restrict__ l_pay) {
    constexpr uint32_t NL = 4;   // lines with hits fetched per round trip
    if (line0 == 0u || td.nlev < 2) return 0u;
    const uint32_t hi_line = line0 - 1u;
    uint32_t g1 = hi_line & ~63u, n = 0;
    uint64_t rem = group_mask(td, g1, s, lane) & mask_upto(hi_line - g1);
    while (true) {
        if (rem == 0) {
            if (g1 == 0u) break;
            const uint32_t l = prev_line(td, g1, 0u, s, lane);
            if (l == NONE) break;
            g1 = l & ~63u;
            rem = group_mask(td, g1, s, lane) & mask_upto(l - g1);
            continue;
        }
        const uint32_t nv = min((uint32_t)__popcll(rem), NL);
        uint32_t pay[NL];
        S e[NL];
#pragma unroll
        for (uint32_t j = 0; j < NL; ++j) {
            const uint32_t b = rem ? 63u - (uint32_t)__builtin_clzll(rem) : 0u;
            if (rem) rem &= ~(1ull << b);
            const uint32_t p = (g1 + b) * 64u + 63u - (uint32_t)lane;   // (past the last line: the group's first, unused)
            e[j] = ends[p];
            pay[j] = VALUES ? (uint32_t)vals[p] : p;
        }
#pragma unroll
        for (uint32_t j = 0; j < NL; ++j) {
            const bool h = j < nv && e[j] >= s;
            const uint64_t m = __builtin_amdgcn_ballot_w64(h);
            const uint32_t cnt = (uint32_t)__popcll(m);
            if (n + cnt > SW_CAP) return n + cnt;   // wave-uniform
            if (h) {
                const uint32_t slot = n + lanes_below(m);
                l_end[slot] = e[j];
                l_pay[slot] = pay[j];
            }
            n += cnt;
        }
    }
    return n;
}

// The queries of one sweep group as its lanes hold them, and the list they are answered from.
template <typename S>
struct SweepGroup {
    S s;                 // query start
    uint32_t ub, lb;     // upper_bound of the end, lower_bound of the start
    uint64_t at;         // address of the query's first output slot
    uint32_t room;       // output slots it may write
    uint32_t found;      // its hits, written as they are found
};

// Answers the group's queries `todo` (a lane each): their run, then, with NB >= 0, the hits in
// the window (we, wp: position wbase + 63 - lane) and in the first NB list registers.  Every
// store goes through a buffer resource over the query's own slots, so slots past its room and
// lanes without a hit (offset 0xFFFFFFFF) are dropped by the hardware.
//
// Everything the loop reads is waited for before it: a load still in flight at the loop's head
// would put a wait for all memory operations, the stores of the query before included, into
// every turn of the loop.
template <typename S, int MODE, int NB>
__device__ __forceinline__ void sweep_emit(SweepGroup<S>& g, uint64_t todo, int lane, uint32_t wbase, S& we, uint32_t& wp,
                                           S (&le)[SW_REGS], uint32_t (&lp)[SW_REGS],
                                           const int32_t* __restrict__ vals) {
    constexpr bool VALUES = MODE == W_VALUES;
    constexpr int NL = NB > 0 ? NB : 0;
    const uint32_t lane4 = (uint32_t)lane * 4u;
    asm volatile("" : "+v"(g.s), "+v"(g.ub), "+v"(g.lb), "+v"(g.at), "+v"(g.room));
    if (NB >= 0) {
        asm volatile("" : "+v"(we), "+v"(wp));
#pragma unroll
        for (int r = 0; r < NL; ++r) asm volatile("" : "+v"(le[r]), "+v"(lp[r]));
    }
    while (todo) {
        const uint32_t j = (uint32_t)__builtin_ctzll(todo);
        todo &= todo - 1ull;
        const uint32_t ub = read_lane(g.ub, j), lb = read_lane(g.lb, j);
        uint32_t room = read_lane(g.room, j);
        uint64_t at = read_lane(g.at, j);
        uint64_t mw = 0, ml[NL + 1];
        uint32_t lead = ub + 1u - lb, total = lead;   // (NONE + 1 = 0)
        if (NB >= 0) {
            const S s = read_lane(g.s, j);
            const uint32_t d = (0u - lb) & 63u;   // window lanes from d on are below lb
            mw = __builtin_amdgcn_ballot_w64(we >= s) & (~0ull << d);
            total += (uint32_t)__popcll(mw);
#pragma unroll
            for (int r = 0; r < NL; ++r) {
                ml[r] = __builtin_amdgcn_ballot_w64(le[r] >= s);   // (lanes past the list hold the smallest value)
                total += (uint32_t)__popcll(ml[r]);
            }
            if (MODE == W_VECTOR) {
                // the leading run: [lb, ub] and the positions right below it that are hits
                const uint64_t miss = ~mw & (~0ull << d);
                if (miss) {
                    const uint32_t z = (uint32_t)__builtin_ctzll(miss);
                    lead += z - d;
                    mw &= ~0ull << z;
                } else {
                    lead += 64u - d;
                    mw = 0;
                    bool on = true;   // every position down to wbase is a hit: on into the list
#pragma unroll
                    for (int r = 0; r < NL; ++r) {
                        if (on) {
                            const uint64_t out_of = ~(ml[r] & __builtin_amdgcn_ballot_w64(
                                                                  lp[r] == wbase - 1u - (uint32_t)(r * WAVE + lane)));
                            if (out_of) {
                                const uint32_t z = (uint32_t)__builtin_ctzll(out_of);
                                lead += z;
                                ml[r] &= ~0ull << z;
                                on = false;
                            } else {
                                lead += 64u;
                                ml[r] = 0;
                            }
                        }
                    }
                }
            }
        }
        g.found = (uint32_t)lane == j ? total : g.found;
        // the (leading) run
        uint32_t p = (MODE == W_VECTOR) ? ub + 1u - lead + (uint32_t)lane : ub - (uint32_t)lane;
        uint32_t w = min(lead, room);
        if (w >= 8u * WAVE) {   // to a 256-byte boundary, then four values a lane and store
            global_u32* o = reinterpret_cast<global_u32*>((uintptr_t)at);
            constexpr uint32_t STEP = 4u * WAVE, UP = (MODE == W_VECTOR) ? 1u : 0u - 1u;   // (positions a slot)
            uint32_t done = (0u - (uint32_t)(at >> 2)) & 63u;
            if ((uint32_t)lane < done) o[(uint32_t)lane] = VALUES ? (uint32_t)vals[p] : p;
            p += UP * (done + 3u * (uint32_t)lane);
            o += done + 4u * (uint32_t)lane;
            if (VALUES) {
                for (; w - done >= 4u * STEP; done += 4u * STEP) {   // four loads before their stores
                    u32x4 v[4];
#pragma unroll
                    for (uint32_t x = 0; x < 4u; ++x) v[x] = *reinterpret_cast<const u32x4*>(vals + (p - x * STEP - 3u));
#pragma unroll
                    for (uint32_t x = 0; x < 4u; ++x) *reinterpret_cast<global_u32x4*>(o + x * STEP) = v[x].wzyx;
                    o += 4u * STEP;
                    p -= 4u * STEP;
                }
            }
            for (; w - done >= STEP; done += STEP) {
                const u32x4 v = VALUES ? (*reinterpret_cast<const u32x4*>(vals + (p - 3u))).wzyx
                                       : u32x4{p, p + UP, p + 2u * UP, p + 3u * UP};
                *reinterpret_cast<global_u32x4*>(o) = v;
                o += STEP;
                p += UP * STEP;
            }
            p -= UP * 3u * (uint32_t)lane;
            w -= done;
            at += (uint64_t)done * 4u;
            lead -= done;
            room -= done;
        }
        // (at most 2^28 slots: everything below is within a few thousand of `at`)
        {
            const __amdgpu_buffer_rsrc_t rs =
                __builtin_amdgcn_make_buffer_rsrc(reinterpret_cast<void*>(at), (short)0, (int)(w * 4u), 0x00020000);
            if (VALUES) {
                // two loads before their stores, as a load waits for the stores before it (2.5M queries on 3M int32
                // intervals that start at 60K places, 75 hits each: 594 us one by one, 541; the walk 466)
                for (uint32_t x = 0; x < w; x += 2u * WAVE) {
                    // (lanes past the run read a value too: position 0's)
                    const uint32_t a = (uint32_t)vals[x + (uint32_t)lane < w ? p : 0u];
                    const uint32_t b = (uint32_t)vals[x + (uint32_t)lane + WAVE < w ? p - (uint32_t)WAVE : 0u];
                    __builtin_amdgcn_raw_buffer_store_b32(a, rs, lane4 + x * 4u, 0, 0);
                    __builtin_amdgcn_raw_buffer_store_b32(b, rs, lane4 + (x + WAVE) * 4u, 0, 0);
                    p -= 2u * (uint32_t)WAVE;
                }
            } else {
                for (uint32_t x = 0; x < w; x += WAVE) {
                    __builtin_amdgcn_raw_buffer_store_b32(p, rs, lane4 + x * 4u, 0, 0);
                    p += (MODE == W_VECTOR) ? (uint32_t)WAVE : 0u - (uint32_t)WAVE;
                }
            }
        }
        if (NB >= 0) {
            const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
                reinterpret_cast<void*>(at), (short)0, (int)(min(room, 1u << 28) * 4u), 0x00020000);
            uint32_t k = lead;
            auto put = [&](uint64_t mask, uint32_t pay) {
                const uint32_t off = (lanes_below(mask) << 2) + k * 4u;
                __builtin_amdgcn_raw_buffer_store_b32(pay, rs, __builtin_amdgcn_inverse_ballot_w64(mask) ? off : 0xFFFFFFFFu,
                                                      0, 0);
                k += (uint32_t)__popcll(mask);
            };
            if (w == lead) {   // (else the room ended inside the run)
                put(mw, wp);
#pragma unroll
                for (int r = 0; r < NL; ++r) put(ml[r], lp[r]);
            }
        }
    }
}

// Queries with at most this many hits are answered a lane each, when enough of them share a
// window (sweep_lanes).
constexpr uint32_t SW_FEW = 16;

// Answers the queries `todo` a lane each: every lane writes its own run, then the wave goes
// through the window's and the list's entries that reach `from` once, highest first, and each
// lane takes those that reach its start.
template <typename S, int MODE, bool LIST>
__device__ __forceinline__ void sweep_lanes(SweepGroup<S>& g, uint64_t todo, int lane, uint32_t wbase, S from, const S& we,
                                            const uint32_t& wp, const S (&le)[SW_REGS], const uint32_t (&lp)[SW_REGS],
                                            uint32_t A, const int32_t* __restrict__ vals) {
    constexpr bool VALUES = MODE == W_VALUES;
    const bool mine = __builtin_amdgcn_inverse_ballot_w64(todo);
    const uint32_t c = mine ? g.ub + 1u - g.lb : 0u;
    const uint32_t d = (0u - g.lb) & 63u;   // window lanes from d on are below lb
    // the window's entries below the largest lb
    uint64_t cw = 0;
    if (LIST) cw = __builtin_amdgcn_ballot_w64(we >= from) & (~0ull << ((0u - uniform(wave_max(mine ? g.lb : 0u))) & 63u));
    // f(entry's end, payload, whether it lies below the lane's lb), highest position first
    auto entries = [&](auto&& f) {
        if (!LIST) return;
        for (uint64_t m = cw; m; m &= m - 1ull) {
            const uint32_t i = (uint32_t)__builtin_ctzll(m);
            f(read_lane(we, i), read_lane(wp, i), i >= d);
        }
#pragma unroll
        for (int r = 0; r < SW_REGS; ++r) {
            if (A <= (uint32_t)(r * WAVE)) break;
            uint64_t m = __builtin_amdgcn_ballot_w64(le[r] >= from && (uint32_t)(r * WAVE + lane) < A);
            for (; m; m &= m - 1ull) {
                const uint32_t i = (uint32_t)__builtin_ctzll(m);
                f(read_lane(le[r], i), read_lane(lp[r], i), true);
            }
        }
    };
    uint32_t lead = c;
    if (MODE == W_VECTOR)   // the leading run: [lb, ub] and the positions right below it that are hits
        entries([&](S e, uint32_t p, bool below) { lead += (mine && below && e >= g.s && p == g.ub - lead) ? 1u : 0u; });
    global_u32* const o = reinterpret_cast<global_u32*>((uintptr_t)g.at);
    for (uint32_t x = 0; __builtin_amdgcn_ballot_w64(x < lead); ++x) {
        const uint32_t p = (MODE == W_VECTOR) ? g.ub + 1u - lead + x : g.ub - x;
        if (x < min(lead, g.room)) o[x] = VALUES ? (uint32_t)vals[p] : p;
    }
    uint32_t k = lead;
    entries([&](S e, uint32_t p, bool below) {
        // (in vector order the entries of the leading run, above ub - lead, are written already)
        const bool h = mine && below && e >= g.s && (MODE != W_VECTOR || p < g.ub + 1u - lead);
        if (h && k < g.room) o[k] = p;
        k += h ? 1u : 0u;
    });
    g.found = mine ? k : g.found;
}

// The plan's queries t0 .. t0 + m - 1 (of one index), by one wave with its part of the LDS (see above).
// out: the positions or values as 32-bit words; only slots below cap and inside a query's segment
// [offsets[q], offsets[q + 1]) are written.  Queries left to k_sweep_shared go to the plan's heavy
// list from place + parked on, their run already written (not in vector order, where the run is
// part of the leading run); parked counts them.  bad: a query's hits differ from its offsets.
template <typename S, int MODE>
__device__ __forceinline__ void sweep_queries(const IndexView<S>& ix, const TreeDesc<S>& td, const PlanView<S>& pv,
                                                  uint32_t t0, uint32_t m, uint32_t place, uint32_t& parked, int lane,
                                                  S* __restrict__ l_end, uint32_t* __restrict__ l_pay,
                                                  uint32_t* __restrict__ l_key, const uint64_t* __restrict__ offsets,
                                                  uint32_t* __restrict__ out, const int32_t* __restrict__ vals,
                                                  uint64_t cap, bool& bad) {
    constexpr S SMIN = (sizeof(S) == 4) ? (S)INT32_MIN : (S)INT64_MIN;
    constexpr bool VALUES = MODE == W_VALUES;

    // ---- the chunk's queries in the order of their starts: keys (start - smallest) >> sh in
    // 24 bits, query in 8
    S smin;
    uint32_t sh = 0;
    {
        S sv[SW_REGS];
        S lo = pv.s[t0], hi = lo;
        uint32_t off_line = 0;   // a query whose window is not the first one's
        const uint32_t line0 = (uniform(pv.lb[t0]) - 1u) & ~63u;
#pragma unroll
        for (int r = 0; r < SW_REGS; ++r) {
            const uint32_t i = (uint32_t)(r * WAVE + lane);
            sv[r] = (i < m) ? pv.s[t0 + i] : lo;
            off_line |= ((i < m) ? (pv.lb[t0 + i] - 1u) & ~63u : line0) ^ line0;
        }
#pragma unroll
        for (int r = 0; r < SW_REGS; ++r) {
            lo = min(lo, sv[r]);
            hi = max(hi, sv[r]);
        }
        hi = wave_max(hi);
        // (~v reverses the order of a signed type without overflow)
        lo = (S)~wave_max((S)~lo);
        smin = lo;
        uint32_t key[SW_REGS];
        if (__builtin_amdgcn_ballot_w64(off_line != 0u) == 0ull) {
            // one window for all: no order is needed
#pragma unroll
            for (int r = 0; r < SW_REGS; ++r) key[r] = (uint32_t)(r * WAVE + lane);
        } else {
            const uint64_t span = (uint64_t)hi - (uint64_t)lo;
            const uint32_t bits = span ? 64u - (uint32_t)__builtin_clzll(span) : 0u;
            sh = uniform(bits > 24u ? bits - 24u : 0u);
#pragma unroll
            for (int r = 0; r < SW_REGS; ++r) {
                const uint32_t i = (uint32_t)(r * WAVE + lane);
                key[r] = (i < m) ? (uint32_t)(((uint64_t)sv[r] - (uint64_t)lo) >> sh) << 8 | i : 0xFFFFFFFFu;
            }
            if (m > (uint32_t)WAVE) {
                wave_sort<SW_REGS>(key, lane);
            } else if (m > 1u) {
                uint32_t k1[1] = {key[0]};
                wave_sort<1>(k1, lane);
                key[0] = k1[0];
            }
        }
#pragma unroll
        for (int r = 0; r < SW_REGS; ++r) l_key[r * WAVE + lane] = key[r];
        wave_lds_sync();
    }

    // ---- sweep
    uint32_t lp[SW_REGS] = {0u, 0u, 0u, 0u};   // list: payloads and ends, A entries, descending
    S le[SW_REGS] = {SMIN, SMIN, SMIN, SMIN};
    uint32_t A = 0, wbase = NONE;               // wbase NONE: no list yet
    S we = SMIN;                                // window: ends and payloads
    uint32_t wp = 0, full = 0;                  // full: a list outgrew SW_CAP, the chunk's other queries are left too

    // the packed entries l_end / l_pay[0 .. n) as the list
    auto take_list = [&](uint32_t n) {
        wave_lds_sync();
        A = n;
#pragma unroll
        for (int r = 0; r < SW_REGS; ++r) {
            const uint32_t i = (uint32_t)(r * WAVE + lane);
            le[r] = (i < n) ? l_end[i] : SMIN;
            lp[r] = (i < n) ? l_pay[i] : 0u;
        }
        wave_lds_sync();
    };
    auto load_window = [&]() {
        const uint32_t p = wbase + 63u - (uint32_t)lane;
        we = ix.ends[p];
        wp = VALUES ? (uint32_t)vals[p] : p;
    };

    for (uint32_t g0 = 0; g0 < m; g0 += WAVE) {
        // 64 queries in start order, one per lane
        const bool mine = g0 + (uint32_t)lane < m;
        const uint32_t gkey = l_key[min(g0 + (uint32_t)lane, m - 1u)];
        const uint32_t gk = t0 + (gkey & 255u);
        const uint32_t gq = pv.q[gk];
        SweepGroup<S> g;
        g.ub = pv.idx[gk];
        g.lb = pv.lb[gk];
        g.s = pv.s[gk];
        const uint64_t go0 = offsets[gq], go1 = offsets[gq + 1];
        const uint32_t gcnt = (uint32_t)(go1 - go0);
        const uint64_t go = min(go0, cap), goe = min(go1, cap);
        g.room = goe > go ? (uint32_t)min(goe - go, (uint64_t)0xFFFFFFFFu) : 0u;
        g.at = (uint64_t)(uintptr_t)(out + go);
        g.found = 0;
        const uint32_t gline = (g.lb - 1u) & ~63u;
        const bool ordered = g.lb <= g.ub + 1u;   // else start > end, with starts between the two
        // queries whose hits all lie in their run, those held by more intervals than a list takes (by
        // their counts), then those the list serves
        const uint64_t many =
            __builtin_amdgcn_ballot_w64(mine && ordered && g.lb != 0u && gcnt > SW_CAP && gcnt - (g.ub + 1u - g.lb) > SW_CAP);
        uint64_t todo = __builtin_amdgcn_ballot_w64(mine && ordered && g.lb != 0u) & ~many;
        uint64_t left = __builtin_amdgcn_ballot_w64(mine && !ordered && g.ub != NONE) | many;
        const uint64_t runs = __builtin_amdgcn_ballot_w64(mine && ordered && g.lb == 0u) | (MODE == W_VECTOR ? 0ull : many);
        const uint64_t few = __builtin_amdgcn_ballot_w64(mine && ordered && gcnt <= SW_FEW && g.ub + 1u - g.lb <= SW_FEW);
        if (runs) {
            const uint64_t rf = (uint32_t)__popcll(runs & few) >= 8u ? runs & few : 0ull;
            if (rf) sweep_lanes<S, MODE, false>(g, rf, lane, 0u, smin, we, wp, le, lp, 0u, vals);
            if (runs & ~rf) sweep_emit<S, MODE, -1>(g, runs & ~rf, lane, 0u, we, wp, le, lp, vals);
        }
        while (todo) {
            if (full) {
                if (MODE != W_VECTOR) sweep_emit<S, MODE, -1>(g, todo, lane, 0u, we, wp, le, lp, vals);
                left |= todo;
                break;
            }
            // the next query in start order, and all that share its window
            const uint32_t j = (uint32_t)__builtin_ctzll(todo);
            const uint32_t line = read_lane(gline, j);
            if (line != wbase) {
                // no start of the chunk's queries from here on is below this
                const S from = (S)((uint64_t)smin + ((uint64_t)(read_lane(gkey, j) >> 8) << sh));
                if (wbase == NONE || line < wbase || line - wbase > SW_GAP * 64u) {
                    wbase = line;
                    load_window();
                    const uint32_t n =
                        uniform(collect_holding<S, VALUES>(ix.ends, vals, td, line >> 6, from, lane, l_end, l_pay));
                    if (n > SW_CAP) full = 1u;
                    else take_list(n);
                } else {
                    do {
                        // survivors of the window, then of the list, packed
                        const uint64_t bw = __builtin_amdgcn_ballot_w64(we >= from);
                        uint64_t bl[SW_REGS];
                        uint32_t n = (uint32_t)__popcll(bw), at = n;
#pragma unroll
                        for (int r = 0; r < SW_REGS; ++r) {
                            // (lanes past the list hold SMIN, which a from of SMIN would keep)
                            bl[r] = __builtin_amdgcn_ballot_w64(le[r] >= from && (uint32_t)(r * WAVE + lane) < A);
                            n += (uint32_t)__popcll(bl[r]);
                        }
                        if (n > SW_CAP) {
                            full = 1u;
                            break;
                        }
                        if (__builtin_amdgcn_inverse_ballot_w64(bw)) {
                            l_end[lanes_below(bw)] = we;
                            l_pay[lanes_below(bw)] = wp;
                        }
#pragma unroll
                        for (int r = 0; r < SW_REGS; ++r) {
                            if (__builtin_amdgcn_inverse_ballot_w64(bl[r])) {
                                l_end[at + lanes_below(bl[r])] = le[r];
                                l_pay[at + lanes_below(bl[r])] = lp[r];
                            }
                            at += (uint32_t)__popcll(bl[r]);
                        }
                        wbase += 64u;
                        load_window();
                        take_list(n);
                    } while (wbase < line);
                }
                if (full) continue;
            }
            uint64_t same = todo & __builtin_amdgcn_ballot_w64(gline == wbase);
            todo &= ~same;
            // a query answered by the whole wave costs about 70 instructions, an entry that every lane looks at 20
            const uint64_t sf = same & few;
            const S low = (S)((uint64_t)smin + ((uint64_t)(read_lane(gkey, j) >> 8) << sh));   // no start is below
            if ((uint32_t)__popcll(sf) * 3u >= (uint32_t)__popcll(__builtin_amdgcn_ballot_w64(we >= low)) + A + SW_FEW) {
                sweep_lanes<S, MODE, true>(g, sf, lane, wbase, low, we, wp, le, lp, A, vals);
                same &= ~sf;
                if (same == 0) continue;
            }
            if (A == 0u) sweep_emit<S, MODE, 0>(g, same, lane, wbase, we, wp, le, lp, vals);
            else if (A <= (uint32_t)WAVE) sweep_emit<S, MODE, 1>(g, same, lane, wbase, we, wp, le, lp, vals);
            else if (A <= 2u * WAVE) sweep_emit<S, MODE, 2>(g, same, lane, wbase, we, wp, le, lp, vals);
            else sweep_emit<S, MODE, SW_REGS>(g, same, lane, wbase, we, wp, le, lp, vals);
        }
        const bool leave = (left >> lane) & 1ull;
        bad |= mine && !leave && g.found != gcnt;
        if (leave) {
            // (per lane, outside every wave-wide step; the run [lb, ub] is written, but for the vector order)
            const uint32_t c = ordered && MODE != W_VECTOR ? g.ub + 1u - g.lb : 0u;
            // (field by field: the first entry's pad is the chunk's number of them)
            HeavyEntry& he = pv.heavy[place + parked + lanes_below(left)];
            he.k = gk;
            he.cur = ordered ? g.lb - 1u : g.ub;
            he.top = g.ub;
            he.lead = MODE == W_VECTOR ? 1u : 0u;
            he.acc = go + min(c, g.room);
            he.left = gcnt - c;
        }
        parked += (uint32_t)__popcll(left);
    }
}

// One wave per chunk of `chunk` consecutive sorted queries.  MODE: W_DESC, W_VECTOR or W_VALUES.
// A chunk's heavy entries lie at its first query's place, their number in the first one's pad.
// either: the plan's counters say whether the sweep answers.
// MULTI: the plan's queries are sorted by their set (pv.set), a chunk's are answered set by set.
template <typename S, int MODE, bool MULTI = false>
__global__ __launch_bounds__(SW_THREADS) void k_sweep(IndexView<S> ix, TreeDesc<S> td, const SetView<S>* __restrict__ sets,
                                                      PlanView<S> pv, uint32_t nq, uint32_t chunk, bool either,
                                                      const uint64_t* __restrict__ offsets,
                                                      uint32_t* __restrict__ out, const int32_t* __restrict__ vals,
                                                      uint64_t cap) {
    if (either && uniform(pv.counter[2]) == 0u) return;   // the block walk answers
    __shared__ S s_end[SW_WAVES][SW_CAP];
    __shared__ uint32_t s_pay[SW_WAVES][SW_CAP];
    __shared__ uint32_t s_key[SW_WAVES][SW_CHUNK];
    const int lane = lane_id();
    const uint32_t wv = uniform(threadIdx.x / WAVE);
    const uint64_t t0w = (uint64_t)(blockIdx.x * (uint32_t)SW_WAVES + wv) * chunk;
    if (t0w >= nq) return;
    uint32_t t0 = (uint32_t)t0w;
    const uint32_t m = min(chunk, nq - t0);   // this wave's queries
    bool bad = false;
    uint32_t parked = 0;
    if (MULTI) {
        for (uint32_t n; t0 < (uint32_t)t0w + m; t0 += n) {
            const uint32_t g = uniform(pv.set[t0]);
            n = 0;
            for (uint64_t other = 0; other == 0 && t0 + n < (uint32_t)t0w + m;) {
                const uint32_t i = t0 + n + (uint32_t)lane;
                other = __builtin_amdgcn_ballot_w64(i >= (uint32_t)t0w + m || pv.set[i] != g);
                n += other ? (uint32_t)__builtin_ctzll(other) : (uint32_t)WAVE;
            }
            sweep_queries<S, MODE>(sets[g].v, sets[g].td, pv, t0, n, (uint32_t)t0w, parked, lane, s_end[wv], s_pay[wv],
                                   s_key[wv], offsets, out, nullptr, cap, bad);
        }
    } else {
        sweep_queries<S, MODE>(ix, td, pv, t0, m, t0, parked, lane, s_end[wv], s_pay[wv], s_key[wv], offsets, out, vals, cap,
                               bad);
    }
    if (lane == 0) {
        pv.heavy[(uint32_t)t0w].pad = parked;
        if (parked) pv.counter[1] = 1u;   // (a flag: an atomic a wave on one line took 70 us of 100K queries)
    }
    if (bad) atomicOr(&pv.counter[3], 1u);   // a query's hits differ from its offsets
}

// ---- the queries that the sweep left, several answered from one candidate list
//
// Where more than SW_CAP intervals hold a query's start, neighbouring queries share nearly all of
// them.  A workgroup takes a span of the plan's queries, orders those left by their starts
// (and sets) and cuts them into groups.  For a group its waves collect the candidates into LDS,
// highest first, CAP at a time; then each wave answers its queries from the list, two compares, a
// ballot and a store for 64 entries.  Two kinds of list:
//   all of it   the positions below the group's runs whose end reaches its first start: from
//               the index, through the max tree, down to the first start - len, from the long
//               list below that.  For starts close together (SH_NEAR);
//   far         only the long entries below each query's start - len (SH_SPREAD), the positions
//               above it read from the index for each query: long intervals lie thinly spread far
//               below (300 lines of 64 for 4100 hits, one in five a hit, in 20M int64 intervals
//               with 20 % of 10^5 .. 10^7 long) and are shared by starts further apart.
// The kind that takes in more queries is used.  A group of fewer than SH_LEAST queries would leave
// the other waves idle: each walks on its own (wave_walk).
//
// What bounds it: waits for memory, at 16 waves a CU (the lists' LDS).  100K queries on 20M such
// intervals: 0.77 ms (2.0 with a walk of the long list for each query), of which, far lists only,
// without the lists' stores 0.64, without the scan 0.48, without lists 0.33, without the index's
// positions too 0.21.  2000 queries on 20M: 0.13 ms (0.80).  1M queries that 320 of 10M intervals
// hold, none long: fill 0.83 ms (lane walk 1.06, a walk for each query 2.0); 50M on 200M intervals,
// two fifths of them held by 330: 26 ms (52; 76).  CAP 6144 (12 waves a CU) and 8 waves a workgroup
// were slower by 20 and 10 %, CAP 2048 by 10 %, but with payloads, which take another word of LDS
// an entry, faster by 15 %.  SH_SPREAD 512: 1.30 ms for the first fill, 1024: 1.10, 2048 and 4096:
// 1.00.  SH_NEAR 1024 and 4096: the same.  Spans of 64: 0.95 for the first, 0.12 against 0.21 for
// 100K queries that 400 of 1M hold.
constexpr int SH_THREADS = 256;
constexpr int SH_WAVES = SH_THREADS / WAVE;
constexpr uint32_t SH_SPREAD = 2048;     // long entries that start within a group's range
constexpr uint32_t SH_NEAR = 2048;       // positions between the starts of a group that shares all of its list
constexpr uint32_t SH_LEAST = 3;         // smallest group that shares a list
constexpr uint32_t SH_UNROLL = 4;        // groups of 64 candidates a wave looks at together
constexpr uint32_t sh_cap(int mode) { return mode == W_VALUES ? 2048u : 4096u; }
// Workgroups a CU, among which the spans are dealt: as many as its LDS holds, but for int64
// payloads, whose registers leave room for four.  (Six for payloads, more than fit, made the last
// ones wait with the spans dealt to them: 100K queries that 400 of 1M hold 200 us, now 181.)
template <typename S>
constexpr unsigned sh_wgs(int mode) { return mode == W_VALUES && sizeof(S) == 4 ? 5u : 4u; }
template <typename S>
constexpr size_t sh_lds(int mode, bool multi) {   // bytes of a workgroup (the arrays of k_sweep_shared)
    return (sh_cap(mode) + SH_UNROLL * WAVE) * 4u * (mode == W_VALUES ? 3u : 2u) +
           WAVE * (sizeof(S) + 8u + 7u * 4u + (multi ? 4u : 0u)) + 64u;
}
constexpr size_t CU_LDS = 160u << 10;

template <typename S, int MODE, bool MULTI = false>
__global__ __launch_bounds__(SH_THREADS) __attribute__((amdgpu_waves_per_eu(sh_wgs<S>(MODE)))) void k_sweep_shared(IndexView<S> ix_one, TreeDesc<S> td_one, UbTree<S> ub_one,
                                                             BucketView<S> tab, LongView<S> lv,
                                                             const SetView<S>* __restrict__ sets, PlanView<S> pv, uint32_t nq, uint32_t chunk,
                                                             uint32_t span, const uint64_t* __restrict__ offsets,
                                                             uint32_t* __restrict__ out_idx,
                                                             const int32_t* __restrict__ vals,
                                                             int32_t* __restrict__ out_val, uint64_t cap) {
    constexpr S SMIN = (sizeof(S) == 4) ? (S)INT32_MIN : (S)INT64_MIN;
    constexpr bool VALUES = MODE == W_VALUES;
    constexpr uint32_t CAP = sh_cap(MODE);            // candidates held at a time
    constexpr uint32_t LINES = (VALUES || sizeof(S) == 8) ? 4 : 8;   // lines a wave collects at a time (registers)
    constexpr uint32_t ROUND = SH_WAVES * LINES * 64u;   // most that one round of lines adds
    constexpr uint32_t UNROLL = SH_UNROLL;
    static_assert(SH_WAVES == 4, "a workgroup is one wave of each SIMD (amdgpu_waves_per_eu)");
    static_assert(sh_wgs<S>(MODE) * sh_lds<S>(MODE, MULTI) <= CU_LDS, "the workgroups dealt for fit a CU");
    __shared__ uint32_t c_rel[CAP + UNROLL * WAVE], c_pos[CAP + UNROLL * WAVE], c_val[VALUES ? CAP + UNROLL * WAVE : 1];
    __shared__ S q_s[WAVE];
    __shared__ uint64_t q_acc[WAVE];
    __shared__ uint32_t q_top[WAVE], q_p0[WAVE], q_j[WAVE], q_left[WAVE], q_room[WAVE], q_bound[WAVE];
    __shared__ uint32_t q_cur[WAVE], q_set[MULTI ? WAVE : 1];
    __shared__ uint32_t w_tot[2][SH_WAVES], s_n, s_work;
    if (uniform(pv.counter[1]) == 0u || uniform(pv.counter[2]) == 0u) return;   // nothing was left (by the sweep)
    const int lane = lane_id();
    const uint32_t wv = uniform(threadIdx.x / WAVE);
    EntryDeal deal(pv.counter + 8, (nq + span - 1u) / span, blockIdx.x, gridDim.x);
    // the next span of the plan's queries is taken by the last wave while the first prepares this one's
    if (wv == SH_WAVES - 1u) {
        const uint32_t first = deal.take(lane);
        if (lane == 0) s_work = first;
    }
    __syncthreads();
    uint32_t h = uniform(s_work);
    while (h != NONE) {
        const uint32_t k0 = h * span, kn = min(span, nq - k0);
        __syncthreads();   // (the span before is done with the lists, and s_work is read)
        if (wv == SH_WAVES - 1u) {
            const uint32_t then = deal.take(lane);
            if (lane == 0) s_work = then;
        }
        if (span == chunk && uniform(pv.heavy[k0].pad) == 0u) {
            __syncthreads();
            h = uniform(s_work);
            continue;
        }
        for (uint32_t b0 = 0; b0 < kn; b0 += WAVE) {
            if (b0) __syncthreads();   // (the batch before is done with the lists)
            if (wv == 0) {
                // up to 64 entries, in the order of their starts, with the part of the long list each needs
                const uint32_t t = b0 + (uint32_t)lane, i = t % chunk;
                const bool mine = t < kn && i < pv.heavy[k0 + t - i].pad;
                const uint64_t all = __builtin_amdgcn_ballot_w64(mine);
                const HeavyEntry* const he = pv.heavy + k0 + (mine ? t : 0u);
                S s = SMIN;
                uint32_t cur = 0, set = 0, top = 0, left = 0, room = 0;
                uint64_t acc = 0;
                if (mine) {
                    const uint32_t k = he->k;
                    cur = he->cur;
                    top = he->top;
                    left = he->left;
                    acc = he->acc;
                    s = pv.s[k];
                    if (MULTI) set = pv.set[k];
                    // (never below acc: offsets that decrease give an empty room, not a wrapped one)
                    room = (uint32_t)min(max(min(offsets[pv.q[k] + 1u], cap), acc) - acc, (uint64_t)0xFFFFFFFFu);
                }
                uint32_t rank = 0;
                for (uint64_t m = all; m; m &= m - 1ull) {
                    const uint32_t j = (uint32_t)__builtin_ctzll(m);
                    const S o = read_lane(s, j);
                    const bool below = o < s || (o == s && j < (uint32_t)lane);
                    if (MULTI) {
                        const uint32_t so = read_lane(set, j);
                        rank += (so < set || (so == set && below)) ? 1u : 0u;
                    } else {
                        rank += below ? 1u : 0u;
                    }
                }
                uint32_t p0 = 0;   // the first position starting at or after s - len (0: no long list)
                if (!MULTI && mine && lv.len > 0 && (int64_t)s > (int64_t)SMIN + lv.len) {
                    const S x = (S)((int64_t)s - lv.len - 1);
                    if (tab.tab) {
                        const BucketView<S> tt[1] = {tab};
                        const S* const v[1] = {ix_one.starts};
                        const S xs[1] = {x};
                        uint32_t r[1];
                        bucket_ranks<S, 1>(tt, v, ix_one.n, xs, r);
                        p0 = r[0];
                    } else {
                        for (uint32_t m = ix_one.n; m;) {
                            const uint32_t half = m >> 1;
                            if (ix_one.starts[p0 + half] <= x) {
                                p0 += half + 1u;
                                m -= half + 1u;
                            } else {
                                m = half;
                            }
                        }
                    }
                }
                if (mine) {
                    q_s[rank] = s;
                    q_top[rank] = top;
                    q_left[rank] = left;
                    q_acc[rank] = acc;
                    q_room[rank] = room;
                    q_bound[rank] = cur + 1u;
                    q_p0[rank] = p0;
                    q_j[rank] = (!MULTI && lv.len > 0) ? lv.lrank[min(p0, cur + 1u)] : 0u;
                    q_cur[rank] = cur;
                    if (MULTI) q_set[rank] = set;
                }
                if (lane == 0) s_n = (uint32_t)__popcll(all);
            }
            __syncthreads();
            const uint32_t n = uniform(s_n);
            h = uniform(s_work);
            const bool in = (uint32_t)lane < n;
            const uint32_t J = in ? q_j[lane] : 0u, C1 = in ? q_cur[lane] + 1u : 0u, G = (MULTI && in) ? q_set[lane] : 0u;
            const S sl = in ? q_s[lane] : SMIN;
            for (uint32_t g = 0, cnt = 0; g < n; g += cnt) {
                // the next queries that share a list: of all positions below them, or of the long entries
                const uint32_t Jg = read_lane(J, g), Cg = read_lane(C1, g), set = read_lane(G, g);
                const S smin = read_lane(sl, g);
                const bool same = in && G == set && (uint64_t)sl - (uint64_t)smin < 0xFFFFFFFFull;
                auto prefix = [&](bool fit) {
                    const uint64_t out_of = ~(__builtin_amdgcn_ballot_w64(fit) >> g);
                    return out_of ? (uint32_t)__builtin_ctzll(out_of) : (uint32_t)WAVE;
                };
                const uint32_t all = prefix(same && C1 - Cg + SH_NEAR <= 2u * SH_NEAR);
                const uint32_t far = (!MULTI && lv.len > 0) ? prefix(same && J - Jg + SH_SPREAD <= 2u * SH_SPREAD) : 0u;
                const bool near = all >= far;
                cnt = near ? all : far;
                const bool share = cnt >= SH_LEAST;
                const IndexView<S>& ix = [&]() -> const IndexView<S>& { if constexpr (MULTI) return sets[set].v; else return ix_one; }();
                const TreeDesc<S>& td = [&]() -> const TreeDesc<S>& { if constexpr (MULTI) return sets[set].td; else return td_one; }();
                const UbTree<S>& ub = [&]() -> const UbTree<S>& { if constexpr (MULTI) return sets[set].ub; else return ub_one; }();
                // without a list of all positions, their hits at and above s - len from the index; in vector
                // order the leading run; alone, everything
                for (uint32_t i = g; (!share || !near || MODE == W_VECTOR) && i < g + cnt; ++i) {
                    if (i % SH_WAVES != wv) continue;
                    const S s = read_lane(sl, i);
                    uint32_t cur = uniform(q_cur[i]), left = uniform(q_left[i]), bound = 0;
                    const uint32_t top = uniform(q_top[i]);
                    uint64_t acc = read_lane(q_acc[i], 0);
                    const uint64_t oend = acc + uniform(q_room[i]);
                    if (!share) {
                        wave_walk<S, MODE>(ix, td, ub, lv, lane, s, cur, top, MODE == W_VECTOR, acc, oend, left, out_idx,
                                           vals, out_val);
                        if (left != 0u) atomicOr(&pv.counter[3], 1u);
                        continue;
                    }
                    if (MODE == W_VECTOR) wave_lead(ix, lane, s, cur, top, acc, oend, left, out_idx);
                    if (cur != NONE) {
                        bound = cur + 1u;
                        if (!near) {
                            const uint32_t p0 = uniform(q_p0[i]);
                            wave_near<S, MODE>(ix, td, lane, s, cur, p0, acc, oend, left, out_idx, vals, out_val);
                            bound = min(p0, bound);
                        }
                    }
                    q_acc[i] = acc;
                    q_left[i] = left;
                    q_room[i] = (uint32_t)(oend - acc);
                    q_bound[i] = bound;   // (every lane stores the same values)
                }
                if (!share) continue;
                // ---- the positions from p0 on (near), then the long entries below the group's bounds, that
                // reach its first start, highest first
                const bool mine = (uint32_t)lane >= g && (uint32_t)lane < g + cnt;
                const uint32_t p0 = near ? uniform(q_p0[g]) : 0u;
                const uint32_t phi = near ? uniform(wave_max(mine ? C1 : 0u)) : 0u;
                uint32_t jmax = 0;
                if (!MULTI && lv.len > 0) jmax = near ? uniform(lv.lrank[p0]) : uniform(wave_max(mine ? J : 0u));
                uint32_t g1 = 0, par = 0, lo = 0, hi = 0;   // the source's entries [lo, hi) are looked at
                uint64_t rem = 0;
                int source = near ? 0 : 1;                  // 0: the index, 1: the long list
                auto lines_of = [&](uint32_t group) -> uint64_t {
                    if (source == 0) return td.nlev >= 2 ? group_mask(td, group, smin, lane) : 1ull;
                    return lv.td.nlev >= 2 ? group_mask(lv.td, group, smin, lane) : 1ull;
                };
                auto in_range = [&](uint64_t m, uint32_t group) {   // lines from lo's on
                    const uint32_t l = lo >> 6;
                    return l > group ? (l - group > 63u ? 0ull : m & (~0ull << (l - group))) : m;
                };
                auto open = [&]() {   // the source's last group of lines; false: it holds nothing
                    lo = source == 0 ? p0 : 0u;
                    hi = source == 0 ? phi : jmax;
                    rem = 0;
                    if (hi <= lo) return false;
                    const uint32_t hi_line = (hi - 1u) >> 6;
                    g1 = hi_line & ~63u;
                    rem = in_range(lines_of(g1) & mask_upto(hi_line - g1), g1);
                    return true;
                };
                bool more = open();
                if (!more && source == 0) {
                    source = 1;
                    more = open();
                }
                while (more) {
                    uint32_t C = 0;
                    while (C + ROUND <= CAP) {
                        if (rem == 0) {
                            uint32_t l = NONE;
                            if (g1 > (lo >> 6))
                                l = source == 0 ? prev_line(td, g1, lo >> 6, smin, lane) : prev_line(lv.td, g1, 0u, smin, lane);
                            if (l != NONE) {
                                g1 = l & ~63u;
                                rem = in_range(lines_of(g1) & mask_upto(l - g1), g1);
                                continue;
                            }
                            more = source == 0;
                            source = 1;
                            if (more) more = open();
                            if (!more) break;
                            continue;
                        }
                        uint32_t e32[LINES], pos[LINES], line[LINES];
                        S ev[LINES];
                        // the next SH_WAVES * LINES lines, a contiguous part for each wave
                        auto drop = [](uint64_t m, uint32_t n) {
                            for (; n && m; --n) m &= ~(1ull << (63u - (uint32_t)__builtin_clzll(m)));
                            return m;
                        };
                        uint64_t own = drop(rem, wv * LINES);
                        rem = drop(rem, SH_WAVES * LINES);
                        const uint32_t nl = min((uint32_t)__popcll(own), LINES);
#pragma unroll
                        for (uint32_t j = 0; j < LINES; ++j) {
                            const uint32_t b = own ? 63u - (uint32_t)__builtin_clzll(own) : 0u;
                            if (own) own &= ~(1ull << b);
                            line[j] = g1 + b;
                        }
#pragma unroll
                        for (uint32_t j = 0; j < LINES; ++j) {
                            const uint32_t p = line[j] * 64u + 63u - (uint32_t)lane;
                            if (source == 0) {
                                if (sizeof(S) == 8 && ix.ends32) e32[j] = ix.ends32[p];
                                else ev[j] = ix.ends[p];
                                pos[j] = p;
                            } else {
                                if (sizeof(S) == 8 && lv.ends32) e32[j] = lv.ends32[p];
                                else ev[j] = lv.ends[p];
                                pos[j] = lv.pos[p];
                            }
                        }
                        const bool by32 = sizeof(S) == 8 && (source == 0 ? ix.ends32 : lv.ends32) != nullptr;
                        const int64_t base32 = source == 0 ? ix.ends32_base : lv.ends32_base;
                        uint32_t rel[LINES], tot = 0;
                        uint64_t m[LINES];
#pragma unroll
                        for (uint32_t j = 0; j < LINES; ++j) {
                            const uint32_t p = line[j] * 64u + 63u - (uint32_t)lane;
                            const int64_t e = by32 ? (int64_t)((uint64_t)base32 + e32[j]) : (int64_t)ev[j];
                            const bool hit = j < nl && p >= lo && p < hi && e >= (int64_t)smin;
                            rel[j] = (uint32_t)min((uint64_t)e - (uint64_t)(int64_t)smin, (uint64_t)0xFFFFFFFFu);
                            m[j] = __builtin_amdgcn_ballot_w64(hit);
                            tot += (uint32_t)__popcll(m[j]);
                        }
                        if (lane == 0) w_tot[par][wv] = tot;
                        __syncthreads();
                        uint32_t at = C;
#pragma unroll
                        for (uint32_t w = 0; w < SH_WAVES; ++w) {
                            const uint32_t x = uniform(w_tot[par][w]);
                            at += w < wv ? x : 0u;
                            C += x;
                        }
                        par ^= 1u;
#pragma unroll
                        for (uint32_t j = 0; j < LINES; ++j) {
                            if (__builtin_amdgcn_inverse_ballot_w64(m[j])) {
                                const uint32_t slot = at + lanes_below(m[j]);
                                c_rel[slot] = rel[j];
                                c_pos[slot] = pos[j];
                                if (VALUES) c_val[slot] = (uint32_t)vals[pos[j]];
                            }
                            at += (uint32_t)__popcll(m[j]);
                        }
                    }
                    if (threadIdx.x < UNROLL * WAVE) c_pos[C + threadIdx.x] = NONE;   // (below no bound)
                    __syncthreads();
                    // ---- each query's hits among them
                    for (uint32_t i = g; i < g + cnt; ++i) {
                        if (i % SH_WAVES != wv) continue;
                        const uint32_t from = (uint32_t)((uint64_t)read_lane(sl, i) - (uint64_t)smin), bound = uniform(q_bound[i]);
                        const uint32_t room = uniform(q_room[i]);
                        const uint64_t acc = read_lane(q_acc[i], 0);
                        const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
                            (VALUES ? (uint32_t*)out_val : out_idx) + acc, (short)0, (int)(min(room, 1u << 28) * 4u), 0x00020000);
                        uint32_t k = 0;
                        for (uint32_t x = (uint32_t)lane; x < C + (uint32_t)lane; x += UNROLL * WAVE) {
                            uint32_t r[UNROLL], p[UNROLL], v[UNROLL];
#pragma unroll
                            for (uint32_t u = 0; u < UNROLL; ++u) {
                                r[u] = c_rel[x + u * WAVE];
                                p[u] = c_pos[x + u * WAVE];
                                v[u] = VALUES ? c_val[x + u * WAVE] : p[u];
                            }
#pragma unroll
                            for (uint32_t u = 0; u < UNROLL; ++u) {
                                const uint64_t m = __builtin_amdgcn_ballot_w64(r[u] >= from && p[u] < bound);
                                const uint32_t off = (lanes_below(m) + k) << 2;
                                __builtin_amdgcn_raw_buffer_store_b32(
                                    v[u], rs, __builtin_amdgcn_inverse_ballot_w64(m) ? off : 0xFFFFFFFFu, 0, SI_OUT_AUX);
                                k += (uint32_t)__popcll(m);
                            }
                        }
                        q_acc[i] = acc + min(k, room);
                        q_room[i] = room - min(k, room);
                        q_left[i] = uniform(q_left[i]) - k;
                    }
                    __syncthreads();
                }
                for (uint32_t i = g; i < g + cnt; ++i)
                    if (i % SH_WAVES == wv && uniform(q_left[i]) != 0u) atomicOr(&pv.counter[3], 1u);
            }
        }
    }
}
