// ksw2_thin.hip -- the stripe kernel's work for pairs whose latency counts:
// a lone pair, or a few that leave most of the device idle.
//
// Such a pair's time is its chain of steps, not the device's throughput, so
// its passes are thin: 128 rows each, two per lane, one wave per pass and
// (normally) one wave per SIMD, all passes of the pair in flight at once.
//  * Rows.  Lane k of pass p owns rows 128p + 2k (low half of every register)
//    and 128p + 2k + 1 (high half, one column behind); at step c the low half
//    is at column c - 2k.  Every input is an output of the step before: the
//    low half takes lane k-1's high half, the high half its own low half.  One
//    packed cell is all a step computes.
//  * Why 128 rows.  A pass trails the one above it by 128 steps of skew and
//    the hand-off, whatever its height, so a pair of n rows and m columns takes
//    about m + 170 n / 128R steps for R cells per lane; a step is 46
//    instructions at R = 1, 27.5 more for each further cell, at some 5.7 cycles
//    each (a wave alone on its SIMD waits 8 for the result it needs next).  R =
//    1 is the fastest up to some 5 kbp and spends half as many instructions
//    again per cell as the stripe kernel's eight rows, so plans that fill the
//    device do not come here.
//  * Hand-off.  Passes go to consecutive waves.  Inside a workgroup of four
//    (one wave per SIMD) a pass's bottom row goes to the next wave through a
//    ring in LDS, a column per step.  From one workgroup to the next it goes
//    through the pair's column buffer in device memory, 16 columns at a time:
//    x, x2, v and, in the low half of v's dword, the number of the pass that
//    reads it.  Those entries are single 8-byte device-scope stores; the reader
//    loads them 20 steps before it needs them and loads again while any does
//    not carry its number, so no count is published and nothing waits for a
//    store to complete.  A pass overwrites a column only after it has read it,
//    so one buffer serves all passes; it is cleared before the launch.  With
//    every hand-off through the column buffer a pass trailed by about 210
//    steps: a lone pair of 5 kbp took 1.58 ms of kernel, 1.53 with the rings
//    (22 us a pass of lag, 0.12 a step), and one of 300 bp 0.11 either way.
//  * All workgroups of a launch are resident together (launch_thin's caller
//    keeps them within its share of the device).  A wait on the column buffer
//    that outlasts 10 s gives up, raises the pair's late word, and the pair's
//    epilogue workgroup computes it again; waits on a ring are on waves of the
//    same workgroup, the earliest unfinished pass of which never waits on one.
//  * Stored bytes.  Four steps of a lane are 8 direction bytes (16 of tracks):
//    cell (row 128p + 2k + h, column j) is at step c = j + 2k + h, in chunk
//    c / 4, byte ((p * chunks + c / 4) * 64 + k) * 8 + 4 ((c & 3) / 2) + 2 h +
//    (c & 1); chunks = (columns + 127) / 4, the chunk past the last sharing the
//    first one's place (lanes 0-1 use the first, lanes 62-63 the other).
//
// Measured: see the figures at launch_thin's rule in ksw2_batch.cpp.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>
#include <type_traits>

#include "ksw2_cell.h"
#include "ksw2_common.h"
#include "ksw2_epilogue.h"
#include "ksw2_kernels.h"

namespace kswhip {

namespace {

using cell::bfi;
using cell::dpp_shl1;
using cell::dpp_shr1;
using cell::hi16;
using cell::lo16;
using cell::perm;
using cell::splat;

constexpr int kSkew = 2 * kWave;                 // the bottom row's column is handed on this many steps after
constexpr int kBlock = 16;                       // columns per hand-off
constexpr uint64_t kWaitTicks = 1000000000ull;  // 10 s of the 100 MHz real-time clock
constexpr int kDeviceLooks = 1024, kRingLooks = 16384;  // at an entry or a count, between two at the stop flag

__device__ __forceinline__ uint64_t load_entry(const int32_t *bnd, int col)
{
    return __hip_atomic_load((const uint64_t *)(bnd + 2 * col), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__device__ __forceinline__ void store_entry(int32_t *bnd, int col, uint32_t a, uint32_t b)
{
    __hip_atomic_store((uint64_t *)(bnd + 2 * col), (uint64_t)a | (uint64_t)b << 32, __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_AGENT);
}

// mqe partial of a pass (see ThinRec): the sum of its rows' u at the last
// column, the smallest running sum with ties to the later row, and that row.
__device__ __forceinline__ void pass_rec(uint32_t us, int p, int i0, int tlen, int lane, ThinRec *out)
{
    const int u0 = lo16(us) - p, u1 = hi16(us) - p;
    int incl = u0 + u1;
#pragma unroll
    for (int off = 1; off < kWave; off <<= 1) {
        const int o = __shfl_up(incl, off, kWave);
        if (lane >= off) incl += o;
    }
    const int s0 = incl - u1;
    int best = 0x7fffffff, best_r = -1;
    if (i0 < tlen) best = s0, best_r = 2 * lane;
    if (i0 + 1 < tlen && incl <= best) best = incl, best_r = 2 * lane + 1;
#pragma unroll
    for (int off = 1; off < kWave; off <<= 1) {
        const int ob = __shfl_xor(best, off, kWave), orow = __shfl_xor(best_r, off, kWave);
        if (ob < best || (ob == best && orow > best_r)) best = ob, best_r = orow;
    }
    const int total = __builtin_amdgcn_readlane(incl, kWave - 1);
    if (lane == 0) out->total = total, out->best_row = best << 7 | best_r;
}

// Hand-off rings in LDS.  Wave w of a workgroup reads its pass's upper boundary
// from ring w, one entry per column: x, x2 and v (in the high halves) and the
// column's score table (its query code, in the high half, when there is no
// table).  Wave w - 1 fills it as it goes, a step at a time; wave 0 fills its
// own, 16 columns at a time, from the column buffer (or row -1's boundary).
// The last wave of a workgroup writes the ring past its own and copies it to
// the column buffer.  Column j is entry j mod kRing of four arrays: a reader
// takes four columns of one in a load, and a writer's two stores per step take
// their operands where they are (as one 16-byte store they were moved to
// consecutive registers first, 4 of 39.5 vector instructions a step).
constexpr int kRing = 256;
struct ThinRing {
    uint32_t e[4][kRing];
    int32_t filled, taken;  // columns written and read: pass (of the wave) * (qlen + 1) + columns
    int32_t pad[14];
};
// The lanes that hold no bottom row write to the space after a workgroup's
// rings.
constexpr int kRingSpill = sizeof(uint32_t) * (3 * kRing + kWave + kBlock);
constexpr int ring_bytes(int waves) { return (waves + 1) * (int)sizeof(ThinRing) + kRingSpill; }

__device__ __forceinline__ int32_t ring_load(const int32_t *x)
{
    return __hip_atomic_load(x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
// (a wave's LDS operations complete in order, so a count stored after an
// entry is seen after it; the empty asm keeps the compiler to that order)
__device__ __forceinline__ void ring_store(int32_t *x, int32_t v)
{
    asm volatile("" ::: "memory");
    __hip_atomic_store(x, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

// One pass of one pair, computed by the calling wave (see the head of this
// file): the kk-th of wave w of a workgroup of `group`.  Lanes compute every
// step; a half's left state is set at its first column and its U kept at the
// last, as in the stripe kernel.  Blocks of 16 steps clear of starts and ends
// are unrolled whole, without their tests.  LAST: the last pass, which writes
// row tlen-1's v in place of the bottom row.
__device__ __forceinline__ uint32_t part(const uint4 &x, int k) { return k == 0 ? x.x : k == 1 ? x.y : k == 2 ? x.z : x.w; }

template <bool RIGHT, int MODE, bool LUT, bool LAST, bool FED, bool FEEDS>
__device__ __forceinline__ void thin_run(const StripeArgs &a, const typename CellOf<RIGHT, MODE>::type &kc, int p,
                                         const KswJob &jb, int qlen, int tlen, ThinRing *rings, int w, int group, int kk,
                                         int &late, int &stop)
{
    const KswScore &sc = a.sc;
    const int lane = threadIdx.x % kWave;
    const uint8_t *qs = a.seq + jb.q_off, *ts = a.seq + jb.t_off;
    int32_t *bnd = a.bnd + jb.bnd_off;
    const int nsteps = qlen + kSkew;
    const int chunks = thin_chunks(qlen);
    const int i0 = kThinRows * p + 2 * lane;
    uint32_t tb, us;
    {
        const int t0 = i0 < tlen ? (int)ts[i0] : 0, t1 = i0 + 1 < tlen ? (int)ts[i0 + 1] : 0;
        tb = LUT ? ((uint32_t)t0 | 12u << 8 | (uint32_t)(t1 + 4) << 16 | 12u << 24) : ((uint32_t)t0 | (uint32_t)t1 << 16);
        us = (uint32_t)(kc.diff(edge_diff(sc, i0)) & 0xffff) | (uint32_t)kc.diff(edge_diff(sc, i0 + 1)) << 16;
    }
    cell::Right st;
    st.u = us, st.y = kc.y0(), st.y2 = kc.y20();
    // (what comes from outside the pair's columns is any value: a column's
    // cells take nothing from the columns on its right)
    cell::Down down;
    down.x = kc.x0(), down.x2 = kc.x20(), down.v = splat(kc.p);
    const uint32_t tag = (uint32_t)p & 0xffffu;  // of the column-buffer entries this pass reads
    const uint32_t sx_rep = (uint32_t)(kc.sx & 0xff) * 0x01010101u, s_flip = (uint32_t)((kc.sm ^ kc.sx) & 0xff);
    const uint32_t sm2 = splat(kc.sm), sd2 = splat(kc.sx - kc.sm);
    uint32_t one = 0x00010001u;
    asm volatile("" : "+s"(one));
    const uint32_t tab0 = LUT ? sx_rep ^ s_flip : 0u;  // of code 0

    ThinRing &in = rings[w], &out = rings[w + 1];
    const int base = kk * (qlen + 1);
    auto stopped = [&]() {
        if (a.stop)
            stop = __builtin_amdgcn_readfirstlane(__hip_atomic_load(a.stop, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM));
        return stop != 0;
    };
    // while waiting it is looked at now and then, every millisecond or two: a
    // load over the bus on every look at a count made each wait last one, and a
    // thousand waves' loads filled the bus (38 pairs of 5 kbp in a server's
    // flight: 50 ms, 2.5 so).  A look at a ring takes a tenth of one at device
    // memory: with the same number between two loads, flights of 22 and 39
    // such pairs together still took 6-9 ms or 23-26, from run to run.
    int spins = 0;
    auto stopped_waiting = [&](int looks) { return (++spins & (looks - 1)) == 0 ? stopped() : stop != 0; };

    // ---- wave 0: column-buffer entries of a block, asked for 16 steps before
    // they are put into the ring and 20 before the first is used.  One set of
    // registers, filled and emptied at the same point of a block: the wait is
    // then for these loads alone, with the block's stores behind them still on
    // their way (two sets moved in turn waited for every store of the block
    // as well: 0.14 us a step, 0.12 so).
    uint64_t ne = 0;
    uint32_t nq = 0;  // the columns' query codes
    auto fetch = [&](int nb) {
        const int col = min(nb + min(lane, kBlock - 1), qlen - 1);
        if (p > 0) ne = load_entry(bnd, col);
        nq = qs[col];
    };
    auto fill = [&](int nb) {  // the block fetched
        const int col = nb + lane;
        const bool have = lane < kBlock && col < qlen;
        uint32_t x, x2, v;
        if (p == 0) {
            x = kc.x0(), x2 = kc.x20(), v = (uint32_t)kc.diff(edge_diff(sc, col)) << 16;
        } else {
            if (__builtin_expect(__ballot(have && (uint32_t)(ne >> 32 & 0xffffu) != tag) != 0 && !late && !stop, 0)) {
                // not all written yet: load again until they are
                const uint64_t t_start = wall_clock64();
                for (;;) {
                    if (have) ne = load_entry(bnd, col);
                    if (__ballot(have && (uint32_t)(ne >> 32 & 0xffffu) != tag) == 0 || stopped_waiting(kDeviceLooks)) break;
                    if (wall_clock64() - t_start > kWaitTicks) {
                        late = 1;
                        break;
                    }
                }
            }
            x = (uint32_t)ne, x2 = (uint32_t)ne << 16, v = (uint32_t)(ne >> 32);
        }
        const int k = col & (kRing - 1);
        if (have)
            in.e[0][k] = x, in.e[1][k] = x2, in.e[2][k] = v,
            in.e[3][k] = LUT ? sx_rep ^ (s_flip << (8 * nq)) : nq << 16;
    };

    // ---- this pass's boundary entries, four columns at a time
    int known = FED ? 0 : 0x7fffffff;
    auto read4 = [&](int c, uint4 (&e)[4]) {
        if (__builtin_expect(known < base + min(c + 4, qlen), 0)) {
            while ((known = __builtin_amdgcn_readfirstlane(ring_load(&in.filled))) < base + min(c + 4, qlen)) {
                if (stopped_waiting(kRingLooks)) break;
                __builtin_amdgcn_s_sleep(1);
            }
        }
        asm volatile("" ::: "memory");  // the entries are read after their count
#pragma unroll
        for (int k = 0; k < 4; ++k) e[k] = *(const uint4 *)&in.e[k][c & (kRing - 1)];
    };

    const int h_last = (tlen - 1) & 1, lane_last = ((tlen - 1) % kThinRows) / 2;
    const int out_lane = LAST ? lane_last : kWave - 1;
    uint32_t tab_lo = tab0, tab_hi = tab0;  // score table (or code) of each half's column
    uint8_t *dir = a.dir + jb.dir_off + ((uint64_t)p * chunks * kWave + lane) * kThinLane * (MODE == kTracks ? 2 : 1);
    // the halves at their first and at their last column: one after the other,
    // as values pass from row to row
    uint32_t start = lane == 0 ? 0x0000ffffu : 0u, last = 0;
    uint32_t *slot = nullptr;  // this lane's entry of the out ring for the block's first step

    // four steps from c (a multiple of 4) and their stored bytes; edge: 1 a
    // half may start in them, 2 may end
    auto steps4 = [&](int c, uint4 (&e)[4], auto edge) {
        constexpr bool START = decltype(edge)::value & 1, END = decltype(edge)::value & 2;
        cell::DirWord wd[4];
        uint32_t tv[4], tu[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            // the bottom row's outputs of the step before (its lane's high
            // half); in the last pass row tlen-1's v
            uint32_t *o = slot + (c + k & (kBlock - 1));
            if (!LAST) o[0] = down.x, o[kRing] = down.x2, o[3 * kRing] = tab_hi;
            o[2 * kRing] = LAST && !h_last ? down.v << 16 : down.v;
            cell::Down d;
            d.x = __builtin_amdgcn_alignbit(down.x, dpp_shr1(part(e[0], k), down.x), 16);
            d.x2 = __builtin_amdgcn_alignbit(down.x2, dpp_shr1(part(e[1], k), down.x2), 16);
            d.v = __builtin_amdgcn_alignbit(down.v, dpp_shr1(part(e[2], k), down.v), 16);
            const uint32_t up = dpp_shr1(part(e[3], k), tab_hi);
            tab_hi = tab_lo;
            tab_lo = up;
            if (START) {
                st.u = bfi(start, us, st.u), st.y = bfi(start, kc.y0(), st.y), st.y2 = bfi(start, kc.y20(), st.y2);
                start = __builtin_amdgcn_alignbit(start, dpp_shr1(0u, start), 16);
            }
            uint32_t s;
            if (LUT) {
                s = perm(tab_hi, tab_lo, tb);
            } else {
                // (codes travel in the high half of tab_lo and tab_hi)
                const uint32_t code = perm(tab_hi, tab_lo, 0x07060302u);
                const cell::v2u mm = __builtin_elementwise_min(__builtin_bit_cast(cell::v2u, tb ^ code),
                                                               __builtin_bit_cast(cell::v2u, one));
                s = __builtin_bit_cast(uint32_t, __builtin_bit_cast(cell::v2u, sm2) +
                                                     mm * __builtin_bit_cast(cell::v2u, sd2));
            }
            wd[k] = kc.step(s, d, st);
            down = d;
            tv[k] = d.v, tu[k] = st.u;
            if (END) {
                // lane 0's low half ends at the last column, the others in turn
                const uint32_t at = c + k == qlen - 1 ? 0xffff0000u : 0u;
                last = __builtin_amdgcn_alignbit(last, dpp_shr1(at, last), 16);
                us = bfi(last, st.u, us);
            }
        }
        if (MODE != kScoreOnly) {
            const int ch = c >> 2;
            // past the last chunk: lanes that may still be in their columns go
            // on from the first one's place, which they don't need, and the
            // others to the last one's
            const int at = !END || ch < chunks ? ch : lane < kWave / 2 ? chunks - 1 : ch - chunks;
            uint8_t *dst = dir + (uint64_t)at * kWave * kThinLane * (MODE == kTracks ? 2 : 1);
            if (MODE == kDirs) {
                uint2 o;
                o.x = kc.pack(wd[0], wd[1]), o.y = kc.pack(wd[2], wd[3]);
                *(uint2 *)dst = o;
            } else {
                uint4 o;
                o.x = perm(tv[1], tv[0], 0x06020400u), o.y = perm(tv[3], tv[2], 0x06020400u);
                o.z = perm(tu[1], tu[0], 0x06020400u), o.w = perm(tu[3], tu[2], 0x06020400u);
                *(uint4 *)dst = o;
            }
        }
    };

    if (!FED) {
        fetch(0);
        fill(0);
        fetch(kBlock);
    }
    uint4 e[4], f[4];
    read4(0, e);
    const int col_off = LAST ? 2 * lane_last + h_last + 1 : kSkew;  // a ring entry's column, behind its step
    uint32_t *spill = (uint32_t *)(rings + group + 1);
    int room = w + 1 < group ? __builtin_amdgcn_readfirstlane(ring_load(&out.taken)) : 0;
    // a block's entries from the ring to the column buffer, with the number of
    // the pass that reads it: taken and stored either side of the next block's
    // first steps
    uint32_t h0 = 0, h1 = 0, h2 = 0;
    auto take = [&](int cb) {
        asm volatile("" ::: "memory");
        const uint32_t *o = out.e[0] + (cb - kSkew & (kRing - 1)) + min(lane, kBlock - 1);
        h0 = o[0], h1 = o[kRing], h2 = o[2 * kRing];
    };
    auto hand_on = [&](int cb) {
        const int col = cb - col_off + lane;
        if (lane < kBlock && col >= 0 && col < qlen)
            store_entry(bnd, col, perm(h0, h1, 0x07060302u), bfi(0xffff0000u, h2, (tag + 1) & 0xffffu));
    };
#pragma unroll 1
    for (int c0 = 0; c0 < nsteps; c0 += kBlock) {
        // the host's stop flag, every 256 columns: end (nothing of this pair is
        // delivered; the waves that wait for this one read the flag too)
        if (__builtin_expect((c0 & 255) == 0 && stopped(), 0)) return;
        const int nb = c0 + kBlock;
        const bool writes = nb > col_off;  // the block has columns to hand on
        if (w + 1 < group && writes) {
            // the entries it overwrites have been read (the last pass, which
            // feeds no wave, too writes where the wave after it may still be
            // reading its pass before)
            const int need = max(FEEDS ? base + nb - kSkew - kRing : base, base);
            while (__builtin_expect(room < need, 0)) {
                if (stopped_waiting(kRingLooks)) return;
                __builtin_amdgcn_s_sleep(1);
                room = __builtin_amdgcn_readfirstlane(ring_load(&out.taken));
            }
        }
        const int taken = w + 1 < group ? ring_load(&out.taken) : 0;  // looked at a block later
        slot = lane == out_lane && writes ? out.e[0] + (c0 - kSkew & (kRing - 1)) : spill + lane;
        auto group4 = [&](int k, auto edge) {
            const int c = c0 + k;
            const int pr = FED ? ring_load(&in.filled) : 0;  // looked at after the steps
            if (!FED && k == kBlock / 2) {
                if (nb < qlen) fill(nb);
                fetch(nb + kBlock);
            }
            if (!FEEDS && k == 0) take(c0 - kBlock);
            read4(c + 4, f);
            steps4(c, e, edge);
            if (FEEDS) ring_store(&out.filled, base + min(max(c + 4 - kSkew, 0), qlen));
            if (FED) known = __builtin_amdgcn_readfirstlane(pr);
            if (!FEEDS && k == 0) hand_on(c0 - kBlock);
#pragma unroll
            for (int x = 0; x < 4; ++x) e[x] = f[x];
        };
        if (__builtin_expect(c0 >= 2 * kWave && nb + 4 <= qlen, 1)) {
#pragma unroll
            for (int k = 0; k < kBlock; k += 4) group4(k, std::integral_constant<int, 0>());
        } else {
            // (every pass waits for the one above it to start, so the start is
            // unrolled as well)
            if (nb + 4 <= qlen) {
#pragma unroll
                for (int k = 0; k < kBlock; k += 4) group4(k, std::integral_constant<int, 1>());
            } else {
#pragma unroll 1
                for (int k = 0; k < kBlock; k += 4) group4(k, std::integral_constant<int, 3>());
            }
        }
        if (FED) ring_store(&in.taken, base + min(nb, qlen));
        room = __builtin_amdgcn_readfirstlane(taken);
    }
    if (!FEEDS) {
        const int cb = nsteps - 1 & ~(kBlock - 1);
        take(cb), hand_on(cb);
    }
    if (FED) ring_store(&in.taken, base + qlen + 1);
    pass_rec(us, kc.p, i0, tlen, lane, (ThinRec *)(a.recs + jb.stripe_off) + p);
}

template <bool RIGHT, int MODE, bool LUT>
__device__ __forceinline__ void thin_pass(const StripeArgs &a, const typename CellOf<RIGHT, MODE>::type &kc, int p,
                                          const KswJob &jb, int qlen, int tlen, ThinRing *rings, int w, int group, int kk,
                                          int &late, int &stop)
{
    const bool last = p == thin_passes(tlen) - 1, feeds = !last && w + 1 < group;
    if (last && w)
        thin_run<RIGHT, MODE, LUT, true, true, false>(a, kc, p, jb, qlen, tlen, rings, w, group, kk, late, stop);
    else if (last)
        thin_run<RIGHT, MODE, LUT, true, false, false>(a, kc, p, jb, qlen, tlen, rings, w, group, kk, late, stop);
    else if (w && feeds)
        thin_run<RIGHT, MODE, LUT, false, true, true>(a, kc, p, jb, qlen, tlen, rings, w, group, kk, late, stop);
    else if (w)
        thin_run<RIGHT, MODE, LUT, false, true, false>(a, kc, p, jb, qlen, tlen, rings, w, group, kk, late, stop);
    else
        thin_run<RIGHT, MODE, LUT, false, false, true>(a, kc, p, jb, qlen, tlen, rings, w, group, kk, late, stop);
}

// Clears the rings' counts (by the whole workgroup, `n` rings).
__device__ __forceinline__ void open_rings(ThinRing *rings, int n)
{
    if ((int)threadIdx.x < n) rings[threadIdx.x].filled = rings[threadIdx.x].taken = 0;
    __syncthreads();
}

// Clears the column buffer of a pair with `n` threads of stride `stride`.
__device__ __forceinline__ void clear_entries(int32_t *bnd, int qlen, int t, int n)
{
    for (int c = t; c < qlen; c += n) store_entry(bnd, c, 0u, 0u);
}

// Singletrack tracks of one pair in the thin layout, in the reference's
// coordinates (i target, j query); as StripeTracks.
struct ThinTracks {
    const uint8_t *dir;
    const uint8_t *qs, *ts;
    int32_t chunks, mch, mis;
    bool tr;
    __device__ int32_t get(int track, int i, int j) const
    {
        if (tr) {
            const int t = i;
            i = j, j = t, track = 1 - track;
        }
        return -(int32_t)(int8_t)dir[thin_track_index(track, i, j, chunks)];
    }
    __device__ int forced(int, int) const { return 0; }
    __device__ int32_t cost(int i, int j) const { return ts[i] == qs[j] ? mch : mis; }
};

// The thin layout as the epilogue reads it.  The walk's tile is a pass (128
// rows) by 160 columns; each lane's columns are shifted by its skew, so a
// lane's chunks are staged from the one that holds the tile's first column.
// The first wave walks a tile while the others stage the one a diagonal path
// enters next, with 16 columns to spare on its right: a path of 5 kbp took
// 0.43 ms when every wave walked and then staged, most of it waiting for the
// tile's bytes, 0.29 ms so.
constexpr int kTileCols = 160, kTileMargin = 16, kTileChunks = kTileCols / 4 + 2;

template <int MODE>
struct ThinLayout {
    static constexpr int mode = MODE;
    typedef ThinTracks Tracks;
    uint2 *tile, *next;  // kTileChunks x 64 lanes each: the walk's, and the one staged meanwhile
    int *share;          // 16 ints
    const uint8_t *dir;
    int chunks;
    int r_lo, r_hi, c_lo, c_hi;  // the walk's tile: striped rows, swept columns

    __device__ ThinLayout(uint2 *t, int *s) : tile(t), next(t + kTileChunks * kWave), share(s) {}
    __device__ void open(const StripeArgs &a, const KswJob &jb)
    {
        dir = a.dir + jb.dir_off, chunks = thin_chunks(jb.qlen);
        r_lo = 1, r_hi = 0, c_lo = 1, c_hi = 0;
    }
    // score and mte from row tlen-1's v, which the last pass left in the
    // column buffer: each thread sums a run of columns, then the runs are
    // chained (largest H = smallest negated sum, ties to the later column)
    __device__ KswOut result(const StripeArgs &a, int, const KswJob &jb, int nthr) const
    {
        constexpr int SH = CellOf<false, MODE>::shift;
        const int tid = threadIdx.x, lane = tid % kWave, wv = tid / kWave, nw = nthr / kWave;
        const int qlen = jb.qlen, tlen = jb.tlen;
        const int bias = jb.flag & 0x02 ? 8 : 0;  // KSW_EZ_RIGHT
        const int vp = MODE == kDirs ? 8 * a.sc.G1 + bias : 0;
        const int32_t *bnd = a.bnd + jb.bnd_off;
        const int per = (qlen + nthr - 1) / nthr, c0 = tid * per, c1 = min(c0 + per, qlen);
        int sum = 0, best = 0x3fffffff, col = -1;
        constexpr int U = 8;
        for (int c = c0; c < c1; c += U) {
            uint32_t e[U];
#pragma unroll
            for (int k = 0; k < U; ++k) e[k] = (uint32_t)bnd[2 * min(c + k, c1 - 1) + 1];
#pragma unroll
            for (int k = 0; k < U; ++k) {
                if (c + k >= c1) break;
                sum += hi16(e[k]) - vp;
                if (sum <= best) best = sum, col = c + k;
            }
        }
        int incl = sum;
#pragma unroll
        for (int off = 1; off < kWave; off <<= 1) {
            const int o = __shfl_up(incl, off, kWave);
            if (lane >= off) incl += o;
        }
        if (lane == kWave - 1) share[wv] = incl;
        __syncthreads();
        int before = incl - sum, total = 0;
        for (int k = 0; k < nw; ++k) {
            if (k < wv) before += share[k];
            total += share[k];
        }
        if (col >= 0) best += before;
#pragma unroll
        for (int off = 1; off < kWave; off <<= 1) {
            const int ob = __shfl_xor(best, off, kWave), oc = __shfl_xor(col, off, kWave);
            if (ob < best || (ob == best && oc > col)) best = ob, col = oc;
        }
        __syncthreads();
        if (lane == 0) share[2 * wv] = best, share[2 * wv + 1] = col;
        __syncthreads();
        for (int k = 0; k < nw; ++k) {
            const int ob = share[2 * k], oc = share[2 * k + 1];
            if (ob < best || (ob == best && oc > col)) best = ob, col = oc;
        }
        __syncthreads();
        const int64_t h_anchor = (int64_t)a.sc.G1 - a.sc.qe_orig;
        const int h_left = (int)(h_anchor + edge_prefix(a.sc, tlen - 1));  // H(tlen-1, -1)
        KswOut o;
        o.score = h_left - (total >> SH), o.mte = h_left - (best >> SH), o.mte_q = col;
        o.mqe = KSW_NEG_INF_I, o.mqe_t = -1;
        o.max = 0, o.max_t = -1, o.max_q = -1;
        o.zdropped = 0, o.stopped = 0, o.reach_end = 0, o.n_cigar = 0;
        return o;
    }
    // the passes' partials in row order, 64 at a time (every wave alike)
    __device__ void last_column(const StripeArgs &a, const KswJob &jb, int, int &best, int &best_i) const
    {
        const ThinRec *recs = (const ThinRec *)(a.recs + jb.stripe_off);
        const int npass = thin_passes(jb.tlen), lane = threadIdx.x % kWave;
        int carry = 0;
        for (int p0 = 0; p0 < npass; p0 += kWave) {
            const int p = p0 + lane;
            int total = 0, b = 0x7fffffff, bi = -1;
            if (p < npass) {
                const ThinRec r = recs[p];
                total = r.total, b = r.best_row >> 7, bi = kThinRows * p + (r.best_row & 127);
            }
            int incl = total;
#pragma unroll
            for (int off = 1; off < kWave; off <<= 1) {
                const int o = __shfl_up(incl, off, kWave);
                if (lane >= off) incl += o;
            }
            if (bi >= 0) b += carry + incl - total;
#pragma unroll
            for (int off = 1; off < kWave; off <<= 1) {
                const int ob = __shfl_xor(b, off, kWave), oi = __shfl_xor(bi, off, kWave);
                if (ob < b || (ob == b && oi > bi)) b = ob, bi = oi;
            }
            if (bi >= 0 && b <= best) best = b, best_i = bi;
            carry += __builtin_amdgcn_readlane(incl, kWave - 1);
        }
    }
    __device__ bool has(int r, int c) const { return r >= r_lo && r <= r_hi && c >= c_lo && c <= c_hi; }
    __device__ int at(int r, int c) const
    {
        const int k = (r & (kThinRows - 1)) >> 1, h = r & 1, s = c + 2 * k + h;
        const int rel = (s >> 2) - ((c_lo + 2 * k) >> 2);
        return ((const uint8_t *)tile)[(rel * kWave + k) * kThinLane + 4 * (s >> 1 & 1) + 2 * h + (s & 1)];
    }
    // wave wv of nw stages pass p's columns up to c into `to`
    __device__ void stage(uint2 *to, int p, int c, int wv, int nw) const
    {
        const int lane = threadIdx.x % kWave, lo_c = max(c - (kTileCols - 1), 0);
        const uint2 *src = (const uint2 *)(dir + (uint64_t)p * chunks * kWave * kThinLane) + lane;
        const int first = (lo_c + 2 * lane) >> 2, last = (c + 2 * lane + 1) >> 2;
        const int lo = lo_c >> 2, hi = (c + 2 * (kWave - 1) + 1) >> 2;
        // whole chunk rows, all of a wave's in flight at once
        constexpr int U = 12;
        for (int ch = lo + wv; ch <= hi; ch += U * nw) {
            uint2 v[U];
#pragma unroll
            for (int k = 0; k < U; ++k) {
                const int x = ch + k * nw;
                if (x >= first && x <= last) v[k] = src[(uint64_t)(x == chunks ? 0 : x) * kWave];
            }
#pragma unroll
            for (int k = 0; k < U; ++k) {
                const int x = ch + k * nw;
                if (x >= first && x <= last) to[(x - first) * kWave + lane] = v[k];
            }
        }
    }
    __device__ void set_tile(int p, int c)
    {
        r_lo = kThinRows * p, r_hi = r_lo + kThinRows - 1;
        c_hi = c, c_lo = max(c - (kTileCols - 1), 0);
    }
    __device__ void walk(PathWalk &w, bool tr, int tid, int nthr)
    {
        const int wv = __builtin_amdgcn_readfirstlane(tid / kWave), nw = nthr / kWave;
        int next_p = -1, next_c = -1;  // the tile in `next`
        while (w.i >= 0 && w.j >= 0) {
            const int r = tr ? w.j : w.i, c = tr ? w.i : w.j, p = r / kThinRows;
            if (p == next_p && c <= next_c && c >= max(next_c - (kTileCols - 1), 0)) {
                uint2 *t = tile;
                tile = next, next = t;
                set_tile(p, next_c);
            } else {
                set_tile(p, c);
                stage(tile, p, c, wv, nw);
                __syncthreads();
            }
            // a diagonal path enters the pass above at this column
            next_p = p - 1, next_c = min(c - (r - r_lo) - 1 + kTileMargin, c);
            if (next_c < 0) next_p = -1;
            if (wv == 0) {
                walk_tile(*this, w, tr);
                if (tid == 0) share[0] = w.i, share[1] = w.j, share[2] = w.n;
            } else if (next_p >= 0) {
                stage(next, next_p, next_c, wv - 1, nw - 1);
            }
            __syncthreads();
            w.i = __builtin_amdgcn_readfirstlane(share[0]), w.j = __builtin_amdgcn_readfirstlane(share[1]);
            __syncthreads();  // read before the first wave writes them again
        }
        // the first wave's runs are the walk's: the others only need its length
        if (tid == 0) share[0] = w.run_op, share[1] = w.run_len, share[2] = w.n;
        __syncthreads();
        w.run_op = __builtin_amdgcn_readfirstlane(share[0]), w.run_len = __builtin_amdgcn_readfirstlane(share[1]);
        w.n = __builtin_amdgcn_readfirstlane(share[2]);
    }
    __device__ Tracks tracks(const StripeArgs &a, const KswJob &jb) const
    {
        const bool tr = jb.transposed != 0;
        Tracks A;
        A.dir = dir, A.chunks = chunks;
        A.qs = a.seq + (tr ? jb.t_off : jb.q_off), A.ts = a.seq + (tr ? jb.q_off : jb.t_off);
        A.mch = a.sc.mch, A.mis = a.sc.mis;
        A.tr = tr;
        return A;
    }
};

}  // namespace

// A pair's workgroups are the blocks wfirst[slot] .. wfirst[slot + 1] of the
// launch (one block per pair when wfirst is null); wave v of its W waves
// computes passes v, v + W, ...
template <bool RIGHT, int MODE, bool LUT>
__global__ void __launch_bounds__(kWave * kThinTeam) __attribute__((amdgpu_waves_per_eu(2)))
ksw_thin_kernel(StripeArgs a)
{
    extern __shared__ __align__(16) uint8_t thin_lds[];
    ThinRing *rings = (ThinRing *)thin_lds;  // one per wave and one more
    const int group = blockDim.x / kWave;
    int slot = blockIdx.x, blk = 0, blocks = 1;
    if (a.wfirst) {
        const int b = a.wfirst[0] + (int)blockIdx.x;
        int lo = 0, hi = a.njobs;
        while (hi - lo > 1) {
            const int mid = (lo + hi) >> 1;
            if (a.wfirst[mid] <= b) lo = mid;
            else hi = mid;
        }
        slot = lo, blk = b - a.wfirst[lo], blocks = a.wfirst[lo + 1] - a.wfirst[lo];
    }
    slot = __builtin_amdgcn_readfirstlane(slot);
    const int W = __builtin_amdgcn_readfirstlane(blocks * group);
    const int w = __builtin_amdgcn_readfirstlane((int)threadIdx.x / kWave), v = __builtin_amdgcn_readfirstlane(blk * group + w);
    open_rings(rings, group + 1);
    const int job = __builtin_amdgcn_readfirstlane(a.order[slot]);
    const KswJob jb = a.jobs[job];
    const typename CellOf<RIGHT, MODE>::type kc(a.sc, jb.transposed != 0);
    const int qlen = __builtin_amdgcn_readfirstlane(jb.qlen), tlen = __builtin_amdgcn_readfirstlane(jb.tlen);
    const int npass = thin_passes(tlen);
    int late = 0, stop = 0;
#pragma unroll 1
    for (int p = v, kk = 0; p < npass && !stop; p += W, ++kk)
        thin_pass<RIGHT, MODE, LUT>(a, kc, p, jb, qlen, tlen, rings, w, group, kk, late, stop);
    if ((late || a.force_late) && threadIdx.x % kWave == 0)
        __hip_atomic_store(a.wctl + (int64_t)slot * kWideCtl + kWideCtlLate, 1, __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_AGENT);
}

// Clears the late words and column buffers of a launch's pairs (blockIdx.y
// the pair) and, with clear_err, the plan's redo count.
__global__ void __launch_bounds__(256) ksw_thin_clear_kernel(StripeArgs a, bool clear_err)
{
    const KswJob &jb = a.jobs[a.order[blockIdx.y]];
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    clear_entries(a.bnd + jb.bnd_off, jb.qlen, t, gridDim.x * blockDim.x);
    if (t == 0) a.wctl[(int64_t)blockIdx.y * kWideCtl + kWideCtlLate] = 0;
    if (clear_err && t == 0 && blockIdx.y == 0) *a.werr = 0;
}

// The epilogue of a launch's pairs, one workgroup each, after all passes.  A
// pair whose late word is raised is computed again by its workgroup first.
template <bool RIGHT, int MODE, bool LUT>
__global__ void __launch_bounds__(kWave * kWideGroup) ksw_thin_epilogue_kernel(StripeArgs a)
{
    __shared__ __align__(16) uint2 tile[2 * kTileChunks * kWave];
    static_assert((int)sizeof(tile) >= ring_bytes(kWideGroup), "the rings of a redo share the tiles' space");
    __shared__ int share[16];
    __shared__ int shared_n;
    const int job = __builtin_amdgcn_readfirstlane(a.order[blockIdx.x]);
    const KswJob jb = a.jobs[job];
    const int late = __builtin_amdgcn_readfirstlane(__hip_atomic_load(
        a.wctl + (int64_t)blockIdx.x * kWideCtl + kWideCtlLate, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
    if (late) {
        const typename CellOf<RIGHT, MODE>::type kc(a.sc, jb.transposed != 0);
        const int qlen = __builtin_amdgcn_readfirstlane(jb.qlen), tlen = __builtin_amdgcn_readfirstlane(jb.tlen);
        clear_entries(a.bnd + jb.bnd_off, qlen, threadIdx.x, blockDim.x);
        __threadfence();
        __syncthreads();
        const int w = __builtin_amdgcn_readfirstlane((int)threadIdx.x / kWave);
        ThinRing *rings = (ThinRing *)tile;
        open_rings(rings, kWideGroup + 1);
        int late2 = 0, stop = 0;
#pragma unroll 1
        for (int p = w, kk = 0; p < thin_passes(tlen) && !stop; p += kWideGroup, ++kk)
            thin_pass<RIGHT, MODE, LUT>(a, kc, p, jb, qlen, tlen, rings, w, kWideGroup, kk, late2, stop);
        __threadfence();
        __syncthreads();
        if (threadIdx.x == 0) atomicAdd(a.werr, 1);
    }
    ThinLayout<MODE> lay(tile, share);
    pair_epilogue(a, job, jb, lay, &shared_n, (int)blockDim.x);
}

namespace {

template <bool RIGHT, int MODE, bool LUT>
struct Thin {
    static hipError_t passes(const StripeArgs &a0, const int32_t *h_wfirst, int max_wgs, int team, int kq, bool clear_err,
                             hipStream_t st)
    {
        StripeArgs a = a0;
        const dim3 clear((unsigned)std::min(std::max((kq + 1023) / 1024, 1), 64), 1);
        if (!h_wfirst) {
            a.wfirst = nullptr;
            hipLaunchKernelGGL(ksw_thin_clear_kernel, dim3(clear.x, a.njobs), dim3(256), 0, st, a, clear_err);
            hipLaunchKernelGGL((ksw_thin_kernel<RIGHT, MODE, LUT>), dim3(a.njobs), dim3(kWave * team),
                               ring_bytes(team), st, a);
            return hipGetLastError();
        }
        for (int off = 0; off < a0.njobs;) {
            // as many pairs as fit in max_wgs workgroups (at least one)
            int end = off + 1;
            while (end < a0.njobs && h_wfirst[end + 1] - h_wfirst[off] <= max_wgs) ++end;
            const int blocks = h_wfirst[end] - h_wfirst[off];
            if (blocks > max_wgs) return hipErrorInvalidConfiguration;
            a.order = a0.order + off, a.wfirst = a0.wfirst + off;
            a.wctl = a0.wctl + (int64_t)off * kWideCtl;
            a.njobs = end - off;
            hipLaunchKernelGGL(ksw_thin_clear_kernel, dim3(clear.x, a.njobs), dim3(256), 0, st, a,
                               clear_err && off == 0);
            hipLaunchKernelGGL((ksw_thin_kernel<RIGHT, MODE, LUT>), dim3(blocks), dim3(kWave * kWideGroup),
                               ring_bytes(kWideGroup), st, a);
            const hipError_t e = hipGetLastError();
            if (e != hipSuccess) return e;
            off = end;
        }
        return hipSuccess;
    }
    static hipError_t epilogue(const StripeArgs &a, hipStream_t st)
    {
        hipLaunchKernelGGL((ksw_thin_epilogue_kernel<RIGHT, MODE, LUT>), dim3(a.njobs), dim3(kWave * kWideGroup), 0, st,
                           a);
        return hipGetLastError();
    }
    static int per_cu()
    {
        int per_cu = 0;
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, (const void *)ksw_thin_kernel<RIGHT, MODE, LUT>,
                                                         kWave * kWideGroup, ring_bytes(kWideGroup)) !=
                hipSuccess)
            return 0;
        return per_cu;
    }
};

// F(variant) for a group and score form.
template <class F> auto by_thin(int group, bool lut, F f)
{
    switch (group) {
    case kGroupRight: return lut ? f(Thin<true, kDirs, true>()) : f(Thin<true, kDirs, false>());
    case kGroupScoreOnly: return lut ? f(Thin<false, kScoreOnly, true>()) : f(Thin<false, kScoreOnly, false>());
    case kGroupTracks: return lut ? f(Thin<false, kTracks, true>()) : f(Thin<false, kTracks, false>());
    default: return lut ? f(Thin<false, kDirs, true>()) : f(Thin<false, kDirs, false>());
    }
}

}  // namespace

hipError_t launch_thin(const StripeArgs &a, int group, bool lut, const int32_t *h_wfirst, int max_wgs, int team, int kq,
                       bool clear_err, hipStream_t st)
{
    if (a.njobs <= 0) return hipSuccess;
    if (!a.wctl || !a.werr || group < 0 || group >= kGroups || a.njobs > 65535) return hipErrorInvalidValue;
    if (h_wfirst) {
        if (!a.wfirst || max_wgs < 1) return hipErrorInvalidValue;
        for (int k = 0; k < a.njobs; ++k) {
            const int n = h_wfirst[k + 1] - h_wfirst[k];
            if (n < 1 || n * kWideGroup > kThinMaxTeam) return hipErrorInvalidValue;
        }
    } else if (team < 1 || team > kThinTeam) {
        return hipErrorInvalidValue;
    }
    return by_thin(group, lut, [&](auto v) { return v.passes(a, h_wfirst, max_wgs, team, kq, clear_err, st); });
}

hipError_t launch_thin_epilogue(const StripeArgs &a, int group, bool lut, hipStream_t st)
{
    if (a.njobs <= 0) return hipSuccess;
    if (!a.wctl || !a.werr || group < 0 || group >= kGroups) return hipErrorInvalidValue;
    return by_thin(group, lut, [&](auto v) { return v.epilogue(a, st); });
}

// Cached per variant: the occupancy query reads the device properties.
int thin_capacity(int group, bool lut)
{
    static int cache[kGroups][2] = {};
    if (group < 0 || group >= kGroups) group = kGroupLeft;
    int &c = cache[group][lut ? 1 : 0];
    int n = __atomic_load_n(&c, __ATOMIC_RELAXED);
    if (n <= 0) {
        n = by_thin(group, lut, [](auto v) { return v.per_cu(); });
        __atomic_store_n(&c, n, __ATOMIC_RELAXED);
    }
    return n * device_cus();
}

}  // namespace kswhip
