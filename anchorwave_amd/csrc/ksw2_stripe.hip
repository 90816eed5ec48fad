// ksw2_stripe.hip -- gfx950 kernels for unbanded ksw_extd2 (the fast path).
//
// Recurrence: the two-piece-affine difference recurrence of
// minimap2/ksw2_extd2_sse.c:43-71 and :237-331 (left/right gap alignment,
// score-only), evaluated for every cell (i = target, j = query).  This file
// evaluates it in a different order and representation than the reference:
//
//  * Stripes and passes.  The target is cut into stripes of 512 rows.  Lane
//    k of a wavefront owns 8 consecutive rows of a stripe and sweeps the
//    query; at step c it is at column j = c - k, so the cell above (i-1, j)
//    was produced by lane k-1 one step earlier and arrives through a DPP
//    wave rotate.  A wave computes two stripes at once (a "pass"): stripe 2p
//    in the low 16 bits of every register and stripe 2p+1 in the high 16
//    bits, 64 steps behind, so every VALU instruction of the cell is a
//    packed 16-bit operation on two cells.  The high stripe's lane 0 takes
//    the low stripe's lane-63 output of the previous step (the rotate wraps
//    it around); the low stripe's lane 0 takes the previous pass's bottom row
//    from a per-pair column buffer; the left neighbour (i, j-1) stays in
//    registers.
//  * Teams.  One workgroup of W waves computes one pair; wave w takes passes
//    w, w+W, ...  Pass p trails pass p-1 by at least two 64-column blocks:
//    the producer writes its bottom-row columns to the column buffer and then
//    publishes a column count in LDS (workgroup-scope release); the consumer
//    polls that count (workgroup-scope acquire) before it reads.  All waves
//    of a team share one CU, so no cache maintenance beyond the CU is
//    involved.  W = 1 (no waiting at all) for pairs that are small against
//    the batch; long pairs get up to 16 waves.  A pair's team may be smaller
//    than the launch's workgroups: the extra waves end at once.
//  * Wide teams (ksw_stripe_wide_kernel).  Above 16 waves, or to give each
//    wave a SIMD of its own, a pair's passes go to several 4-wave
//    workgroups on different CUs; the counts and column-buffer entries are
//    then device-scope accesses, and the epilogue runs in a launch of its
//    own.
//  * Cells (ksw2_cell.h): negated values on packed halves, with a scale and a
//    tag where direction bytes are wanted, plain for scores and tracks.
//    VALU issue bounds the kernel: a middle pass of eight rows takes 248
//    VALU instructions per step (16 cells per lane), 297 before the
//    three-input minimum, the constant-free candidates, the flag bits taken
//    two rows at a time and the score tables that travel between lanes.  The
//    fixed batch (4,096 x 2 kbp, bytes and walk) went from 12.76 to 9.15 ms a
//    launch, score only from 8.99 to 6.43, tracks (2,048 pairs) from 6.63 to
//    4.95; a lone 5 kbp pair on four rows per lane from 4.84 to 2.74 ms, the
//    plain blocks' unrolled steps helping it most.
//  * Exactness.  The reference computes on int8 lanes.  The host only routes
//    a call here when every in-band intermediate provably stays inside int8
//    (then 16-bit arithmetic gives the same values), the match score is 0
//    and no mismatch scores above it (then z = min(z, mat[0]) never binds and
//    H never exceeds 0, so ez->max stays 0), there is no band and no z-drop.
//
// Outputs per pair: the direction byte of every cell (bits as in
// minimap2/ksw2.h:156-159, layout dir_index()), or, for KSW_EZ_SINGLETRACK,
// the two difference tracks of every cell (the new v and u,
// minimap2/ksw2_extd2_avx.c:432-436, layout track_index()); and the H
// bookkeeping of minimap2/ksw2_extd2_sse.c:369-375 (score, mqe/mqe_t,
// mte/mte_q).
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

constexpr int kLag = kWave;      // steps the high stripe trails the low one
constexpr int kAhead = 16;       // steps before a block its boundary entries are loaded

using cell::bfi;
using cell::dpp_ror1;
using cell::dpp_shl1;
using cell::dpp_shr1;
using cell::hi16;
using cell::lo16;
using cell::perm;
using cell::splat;

// The value from the cell above for every lane: lane k takes lane k-1's
// (both halves); lane 0 takes lane 63's low half of the previous step into
// its high half, and the low stripe's boundary value (the high half of b_hi)
// into its low half.  m0 is all ones in lane 0 (a bit operation: a
// v_cndmask on a mask in VCC takes five times as long).
__device__ __forceinline__ uint32_t carry(uint32_t y, uint32_t b_hi, uint32_t m0)
{
    const uint32_t rot = dpp_ror1(y);
    return bfi(m0, __builtin_amdgcn_alignbit(rot, b_hi, 16), rot);
}

// Element i (the same in every lane) of a lane's array.
template <int R> __device__ __forceinline__ uint32_t row_of(const uint32_t (&v)[R], int i)
{
    uint32_t x = v[0];
#pragma unroll
    for (int r = 1; r < R; ++r) x = bfi(i == r ? ~0u : 0u, v[r], x);
    return x;
}

// Team progress: wave w publishes, for its k-th pass, k*(qlen+1) + the
// number of bottom-row columns written so far (monotonic per wave).
__device__ __forceinline__ void publish(int32_t *slot, int value)
{
    // every lane stores the same value (no divergent branch); the release
    // orders the preceding column-buffer stores before the count
    __hip_atomic_store(slot, value, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_WORKGROUP);
}

// Spins until the producer's published count reaches `need`.  The exit test
// uses lane 0's value, so the loop is uniform.  A producer always ends its
// pass at k*(qlen+1) + qlen, so `need` <= that bound terminates.
__device__ __forceinline__ int wait_count(const int32_t *slot, int need, int known)
{
    if (known >= need) return known;
    int seen = __builtin_amdgcn_readfirstlane(__hip_atomic_load(slot, __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_WORKGROUP));
    while (seen < need) {
        __builtin_amdgcn_s_sleep(1);
        seen = __builtin_amdgcn_readfirstlane(__hip_atomic_load(slot, __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_WORKGROUP));
    }
    return seen;
}

// Wide teams (waves on several CUs): counts and column-buffer entries are
// device-scope accesses, coherent across the XCDs' L2s; a count is stored
// only after the entries it covers are complete (s_waitcnt vmcnt(0)).
constexpr uint64_t kWaitTicks = 1000000000ull;  // 10 s of the 100 MHz real-time clock
constexpr int kStopCount = 0x3fffffff;          // published by a stopped wave: past every need

__device__ __forceinline__ void publish_wide(int32_t *slot, int value)
{
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0xF70);  // vmcnt(0)
    asm volatile("" ::: "memory");
    if (__lane_id() == 0) __hip_atomic_store(slot, value, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__device__ __forceinline__ int load_count_wide(const int32_t *slot)
{
    return __builtin_amdgcn_readfirstlane(__hip_atomic_load(slot, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
}

// As wait_count; past kWaitTicks (a workgroup the dispatcher could not
// place) it gives up, sets `late` and returns a count that satisfies every
// later wait, so every wave still runs to its end.
__device__ __forceinline__ int wait_count_wide(const int32_t *slot, int need, int known, int &late)
{
    if (known >= need) return known;
    int seen = load_count_wide(slot);
    if (seen < need) {
        const uint64_t t_start = wall_clock64();
        while (seen < need) {
            __builtin_amdgcn_s_sleep(1);
            seen = load_count_wide(slot);
            if (seen < need && wall_clock64() - t_start > kWaitTicks) {
                late = 1;
                seen = INT32_MAX;
            }
        }
    }
    asm volatile("" ::: "memory");  // the entry loads stay behind the wait
    return seen;
}

// Two column-buffer dwords (one entry): plain accesses within a workgroup,
// device-scope ones across CUs.
template <bool WIDE>
__device__ __forceinline__ void load_entry(const int32_t *src, uint32_t &a, uint32_t &b)
{
    if (WIDE) {
        const uint64_t v = __hip_atomic_load((const uint64_t *)src, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        a = (uint32_t)v, b = (uint32_t)(v >> 32);
    } else {
        a = (uint32_t)src[0], b = (uint32_t)src[1];
    }
}

template <bool WIDE>
__device__ __forceinline__ void store_entry(int32_t *dst, uint32_t a, uint32_t b)
{
    if (WIDE) {
        const uint64_t v = (uint64_t)a | (uint64_t)b << 32;
        __hip_atomic_store((uint64_t *)dst, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    } else {
        dst[0] = (int32_t)a, dst[1] = (int32_t)b;
    }
}

// mqe partial of one stripe from the snapshot of U at column qlen-1 (one
// half of Us, biased by p): H(i,qlen-1) = H(-1,qlen-1) + sum_{i'<=i} u(i'),
// kept negated and scaled as the state; the smallest running sum (largest H)
// with ties to the larger row, and the stripe total.
template <int R>
__device__ __forceinline__ void stripe_rec(const uint32_t (&Us)[R], bool hi, int p, int i0, int tlen, int lane,
                                           StripeRec *out)
{
    int u[R], lsum = 0;
#pragma unroll
    for (int r = 0; r < R; ++r) u[r] = (hi ? hi16(Us[r]) : lo16(Us[r])) - p, lsum += u[r];
    int incl = lsum;
#pragma unroll
    for (int off = 1; off < kWave; off <<= 1) {
        const int o = __shfl_up(incl, off, kWave);
        if (lane >= off) incl += o;
    }
    int run = incl - lsum;
    int best = 0x7fffffff, best_i = -1;
#pragma unroll
    for (int r = 0; r < R; ++r) {
        run += u[r];
        const int i = i0 + r;
        if (i < tlen && run <= best) best = run, best_i = i;
    }
#pragma unroll
    for (int off = 1; off < kWave; off <<= 1) {
        const int ob = __shfl_xor(best, off, kWave);
        const int oi = __shfl_xor(best_i, off, kWave);
        if (ob < best || (ob == best && oi > best_i)) best = ob, best_i = oi;
    }
    const int total = __builtin_amdgcn_readlane(incl, kWave - 1);
    if (lane == 0) {
        StripeRec rec;
        rec.total = total, rec.best = best, rec.best_i = best_i, rec.pad = 0;
        *out = rec;
    }
}

// What follows row tlen-1 over a pair's columns: the sum of v so far, its
// smallest value and the last column that has it (negated and scaled).
struct RowTrack {
    int acc = 0, best = 0x7fffffff, col = -1;
};

// Takes 64 columns of row tlen-1: lane l's v of column col (valid when
// 0 <= col < qlen, the columns ascending with the lane).
__device__ __forceinline__ void track_row(RowTrack &t, int v, int col, int qlen, int lane)
{
    const bool in = col >= 0 && col < qlen;
    int sum = in ? v : 0;
#pragma unroll
    for (int off = 1; off < kWave; off <<= 1) {
        const int o = __shfl_up(sum, off, kWave);
        if (lane >= off) sum += o;
    }
    sum += t.acc;
    int best = in ? sum : 0x7fffffff, at = in ? col : -1;
#pragma unroll
    for (int off = 1; off < kWave; off <<= 1) {
        const int ob = __shfl_xor(best, off, kWave), oa = __shfl_xor(at, off, kWave);
        if (ob < best || (ob == best && oa > at)) best = ob, at = oa;
    }
    t.acc = __builtin_amdgcn_readlane(sum, kWave - 1);
    if (best <= t.best && at >= 0) t.best = best, t.col = at;
}

// One pass (stripes 2p and 2p+1) of one pair, computed by the calling wave.
// Roles (uniform): the first pass takes row -1 as the low stripe's upper
// boundary instead of the column buffer; the last pass holds row tlen-1
// (score / mte) and publishes nothing; every other pass publishes the high
// stripe's bottom row.  Lanes compute every step; each half's left state is
// (re)initialised at its first column and U is snapshot at its last one, so
// the cells a half computes outside its columns never reach a result (they
// are cells of the same recurrence under a boundary of constant H, so they
// stay in range).
// Columns go in blocks of 64: the boundary entries and query codes of a block
// are loaded one per lane, kAhead steps before it, and move to lane 0 one
// step at a time.  A block clear of starts and ends runs several steps per
// loop iteration, without their tests.  LAST: the pass that holds row tlen-1.
// WIDE: the team spans several CUs (progress counts in device memory,
// kWideCtlStride dwords apart; a wait that gives up sets `late`).
template <bool RIGHT, int MODE, bool WIDE, bool LUT, int R, bool LAST>
__device__ __forceinline__ void pass_run(const StripeArgs &a, const typename CellOf<RIGHT, MODE>::type &kc, int job_id,
                                          int p, const KswJob &jb, int qlen, int tlen, int32_t *prog, int W, int &late,
                                          int &stop)
{
    constexpr int SR = kWave * R;           // rows per stripe
    constexpr int kUnroll = R == 8 ? 2 : 4;  // steps per iteration of a plain block
    const KswScore &sc = a.sc;
    const int nstripes = (tlen + SR - 1) / SR;
    const bool first = p == 0, has_hi = 2 * p + 1 < nstripes;
    const int lane = threadIdx.x % kWave;
    uint32_t m0 = lane == 0 ? ~0u : 0u;
    asm volatile("" : "+v"(m0));
    const uint8_t *qs = a.seq + jb.q_off;
    const uint8_t *ts = a.seq + jb.t_off;
    uint8_t *dir = a.dir + jb.dir_off;
    int32_t *bnd = a.bnd + jb.bnd_off;
    const int nsteps = qlen + kWave - 1 + kLag;
    // row tlen-1 (score, mte): stripe s_last, half h_last of the last pass
    const int h_last = ((tlen - 1) / SR) & 1;
    const int rho_last = (tlen - 1) % R;
    const int lane_last = ((tlen - 1) % SR) / R;
    // progress slots: pass p-1 is wave (p-1) % W's ((p-1)/W)-th pass
    constexpr int PS = WIDE ? kWideCtlStride : 1;
    const int32_t *prog_prev = prog + (p + W - 1) % W * PS;
    const int base_prev = first ? 0 : (p - 1) / W * (qlen + 1);
    int32_t *prog_mine = prog + p % W * PS;
    const int base_mine = p / W * (qlen + 1);

    const int ilo = 2 * p * SR + lane * R, ihi = ilo + SR;  // this lane's first rows
    uint32_t TB[R], Us[R];
    cell::Right st[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const int tl = ilo + r < tlen ? (int)ts[ilo + r] : 0, th = ihi + r < tlen ? (int)ts[ihi + r] : 0;
        // LUT: the v_perm selector of row r's two score bytes (table byte
        // tl of the low half's table, byte th of the high half's, zero high
        // bytes); else the two target codes
        TB[r] = LUT ? ((uint32_t)tl | 12u << 8 | (uint32_t)(th + 4) << 16 | 12u << 24)
                    : ((uint32_t)tl | (uint32_t)th << 16);
        Us[r] = (uint32_t)(kc.diff(edge_diff(sc, ilo + r)) & 0xffff) | (uint32_t)kc.diff(edge_diff(sc, ihi + r)) << 16;
        st[r].u = Us[r], st[r].y = kc.y0(), st[r].y2 = kc.y20();
    }
    const uint32_t p2 = splat(kc.p);  // v of a boundary of constant H
    cell::Down down;                  // this lane's bottom-row outputs
    down.x = kc.x0(), down.x2 = kc.x20(), down.v = p2;
    // The lane-0 queues: x (high half) and x2 of the boundary; its v (high
    // half), with the query code in the low half when there is no table; the
    // score table of the query code.
    const uint32_t entry0 = (kc.x0() & 0xffff0000u) | (kc.x20() & 0xffffu);
    // LUT: byte k of a half's table is the score candidate of target code k
    // against that half's query code (sm when equal, sx otherwise)
    const uint32_t sx_rep = (uint32_t)(kc.sx & 0xff) * 0x01010101u;
    const uint32_t s_flip = (uint32_t)((kc.sm ^ kc.sx) & 0xff);
    int known = 0;  // columns of pass p-1 known published
    auto load_block = [&](int nb, uint32_t &e0, uint32_t &e1, uint32_t &eq) {
        const int col = nb + lane;
        e0 = entry0, e1 = p2 & 0xffff0000u;
        if (first) {
            e1 = (uint32_t)kc.diff(edge_diff(sc, col)) << 16;
        } else {
            const int need = base_prev + min(nb + kWave, qlen);
            if (WIDE) known = wait_count_wide(prog_prev, need, known, late);
            else known = wait_count(prog_prev, need, known);
            if (col < qlen) load_entry<WIDE>(bnd + 2 * col, e0, e1);
        }
        eq = col < qlen ? (uint32_t)qs[col] : 0u;
        if (!LUT) e1 = (e1 & 0xffff0000u) | eq;
    };
    uint32_t bin0, bin1, binq, nx0 = 0, nx1 = 0, nxq = 0;
    load_block(0, bin0, bin1, binq);
    if (LUT) binq = sx_rep ^ (s_flip << (8 * binq));
    uint32_t tab_lo = sx_rep, tab_hi = sx_rep, code = 0;
    uint32_t out0 = 0, out1 = 0;  // lane-63 output queue; in the last pass out1 holds row tlen-1's v
    RowTrack row;
    uint32_t one = 0x00010001u;
    asm volatile("" : "+s"(one));
    const uint32_t sm2 = splat(kc.sm), sd2 = splat(kc.sx - kc.sm);
    uint8_t *dst = dir + ((uint64_t)p * nsteps * kWave + lane) * (MODE == kTracks ? 4 * R : 2 * R);

    auto step = [&](int c, auto edge) {
        constexpr bool EDGE = decltype(edge)::value;
        // this step's inputs from above, the queues one step on
        cell::Down d;
        d.x = carry(down.x, bin0, m0), d.x2 = carry(down.x2, bin0 << 16, m0), d.v = carry(down.v, bin1, m0);
        if (LUT) {
            tab_hi = dpp_shr1(dpp_ror1(tab_lo), tab_hi);
            const uint32_t q0 = binq;
            binq = dpp_shl1(binq, binq);
            tab_lo = dpp_shr1(q0, tab_lo);
        } else {
            code = carry(code, bin1 << 16, m0);
        }
        bin0 = dpp_shl1(bin0, bin0), bin1 = dpp_shl1(bin1, bin1);
        const int jl = c - lane;
        if (EDGE) {
            // a half starts at its first column: the lanes there take the
            // half's initial left state (U from Us, which holds it until the
            // half's last column)
            const uint32_t m = jl == 0 ? 0x0000ffffu : jl == kLag ? 0xffff0000u : 0u;
#pragma unroll
            for (int r = 0; r < R; ++r) {
                st[r].u = bfi(m, Us[r], st[r].u);
                st[r].y = bfi(m, kc.y0(), st[r].y), st[r].y2 = bfi(m, kc.y20(), st[r].y2);
            }
        }
        cell::DirWord w[R];
        uint32_t vr[R];
#pragma unroll
        for (int r = 0; r < R; ++r) {
            uint32_t s;
            if (LUT) {
                s = perm(tab_hi, tab_lo, TB[r]);
            } else {
                // min(t ^ q, ONE) with an opaque ONE stays one v_pk_min_u16 (0
                // match, 1 mismatch), the score one v_pk_mad_u16
                const cell::v2u mm = __builtin_elementwise_min(__builtin_bit_cast(cell::v2u, TB[r] ^ code),
                                                               __builtin_bit_cast(cell::v2u, one));
                s = __builtin_bit_cast(uint32_t, __builtin_bit_cast(cell::v2u, sm2) +
                                                     mm * __builtin_bit_cast(cell::v2u, sd2));
            }
            w[r] = kc.step(s, d, st[r]);
            vr[r] = d.v;
        }
        down = d;
        if (EDGE) {
            // a half ends at column qlen-1: keep U for the mqe partials
            const int je = jl - (qlen - 1);
            const uint32_t m = je == 0 ? 0x0000ffffu : je == kLag ? 0xffff0000u : 0u;
#pragma unroll
            for (int r = 0; r < R; ++r) Us[r] = bfi(m, st[r].u, Us[r]);
        }
        if (MODE == kDirs) {
            // 2R bytes per lane: byte 4g + 2h + (rho & 1) is row 2g + (rho & 1)
            // of half h
            if (R == 8) {
                uint4 o;
                o.x = kc.pack(w[0], w[1]), o.y = kc.pack(w[2], w[3]);
                o.z = kc.pack(w[4 % R], w[5 % R]), o.w = kc.pack(w[6 % R], w[7 % R]);
                *(uint4 *)dst = o;
            } else {
                uint2 o;
                o.x = kc.pack(w[0], w[1]), o.y = kc.pack(w[2], w[3]);
                *(uint2 *)dst = o;
            }
            dst += kWave * 2 * R;
        } else if (MODE == kTracks) {
            // 4R bytes per lane: the p track (new V) then the p2 track (new
            // U), each in the byte order of the direction bytes
            uint32_t tv[R / 2], tu[R / 2];
#pragma unroll
            for (int g = 0; g < R / 2; ++g) {
                tv[g] = perm(vr[2 * g + 1], vr[2 * g], 0x06020400u);
                tu[g] = perm(st[2 * g + 1].u, st[2 * g].u, 0x06020400u);
            }
            if (R == 8) {
                uint4 o;
                o.x = tv[0], o.y = tv[1], o.z = tv[2 % (R / 2)], o.w = tv[3 % (R / 2)];
                ((uint4 *)dst)[0] = o;
                o.x = tu[0], o.y = tu[1], o.z = tu[2 % (R / 2)], o.w = tu[3 % (R / 2)];
                ((uint4 *)dst)[1] = o;
            } else {
                uint2 o;
                o.x = tv[0], o.y = tv[1];
                ((uint2 *)dst)[0] = o;
                o.x = tu[0], o.y = tu[1];
                ((uint2 *)dst)[1] = o;
            }
            dst += kWave * 4 * R;
        }
        if (!LAST) {
            // lane 63 appends the high stripe's bottom-row output (column
            // c-127: x in the high half, x2 in the low half; v in the high
            // half) to the queue
            out0 = dpp_shl1(perm(down.x, down.x2, 0x07060302u), out0), out1 = dpp_shl1(down.v, out1);
        } else {
            // row tlen-1's v joins the queue
            out1 = dpp_shl1((uint32_t)__builtin_amdgcn_readlane((int)row_of<R>(vr, rho_last), lane_last), out1);
        }
    };

#pragma unroll 1
    for (int c0 = 0; c0 < nsteps; c0 += kWave) {
        if (a.stop && (c0 & 255) == 0) {
            // the host's stop flag: publish a count past every wait of the
            // team and end (nothing of this pair is delivered)
            stop = __builtin_amdgcn_readfirstlane(__hip_atomic_load(a.stop, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM));
            if (stop) {
                if (WIDE) publish_wide(prog_mine, kStopCount);
                else publish(prog_mine, kStopCount);
                return;
            }
        }
        const int c1 = min(c0 + kWave, nsteps), nb = c0 + kWave;
        const bool plain = c0 >= kWave + kLag && nb < qlen;
        // the next block's entries are waited for and loaded kAhead steps
        // before it starts (late enough that the producer need only be that
        // far ahead, early enough to hide the load)
        for (int c = c0, end = min(nb - kAhead, c1);; end = c1) {
            if (plain) {
#pragma unroll 1
                for (; c < end; c += kUnroll) {
#pragma unroll
                    for (int k = 0; k < kUnroll; ++k) step(c + k, std::integral_constant<bool, false>());
                }
            } else {
#pragma unroll 1
                for (; c < end; ++c) step(c, std::integral_constant<bool, true>());
            }
            if (c >= c1) break;
            load_block(nb, nx0, nx1, nxq);
        }
        bin0 = nx0, bin1 = nx1;
        if (LUT) binq = sx_rep ^ (s_flip << (8 * nxq));
        if (!LAST) {
            // the queue's columns go out, the newest in lane 63
            const int col = c1 - kWave - kLag - (kWave - 1) + lane;
            if (col >= 0 && col < qlen) store_entry<WIDE>(bnd + 2 * col, out0, out1);
            const int count = base_mine + max(0, min(c1 - (kWave - 1) - kLag, qlen));
            if (WIDE) publish_wide(prog_mine, count);
            else publish(prog_mine, count);
        } else {
            const int v = (h_last ? hi16(out1) : lo16(out1)) - kc.p, c = c1 - kWave + lane;
            track_row(row, v, c >= c0 ? c - lane_last - kLag * h_last : -1, qlen, lane);
        }
    }
    stripe_rec<R>(Us, false, kc.p, ilo, tlen, lane, a.recs + jb.stripe_off + 2 * p);
    if (has_hi) stripe_rec<R>(Us, true, kc.p, ihi, tlen, lane, a.recs + jb.stripe_off + 2 * p + 1);
    if (LAST && lane == 0) {
        constexpr int SH = CellOf<RIGHT, MODE>::shift;
        const int64_t h_anchor = (int64_t)sc.G1 - sc.qe_orig;
        const int h_left_last_row = (int)(h_anchor + edge_prefix(sc, tlen - 1));  // H(tlen-1, -1)
        KswOut o;
        o.score = h_left_last_row - (row.acc >> SH);
        o.mte = h_left_last_row - (row.best >> SH);
        o.mte_q = row.col;
        o.mqe = KSW_NEG_INF_I, o.mqe_t = -1;  // finalised by the backtrack kernel
        o.max = 0, o.max_t = -1, o.max_q = -1;
        o.zdropped = 0, o.stopped = 0, o.reach_end = 0, o.n_cigar = 0;
        a.out[job_id] = o;
    }
}

template <bool RIGHT, int MODE, bool WIDE, bool LUT, int R>
__device__ __forceinline__ void pass_body(const StripeArgs &a, const typename CellOf<RIGHT, MODE>::type &kc, int job_id,
                                          int p, const KswJob &jb, int qlen, int tlen, int32_t *prog, int W, int &late,
                                          int &stop)
{
    if (p == pass_count(tlen, R) - 1)
        pass_run<RIGHT, MODE, WIDE, LUT, R, true>(a, kc, job_id, p, jb, qlen, tlen, prog, W, late, stop);
    else
        pass_run<RIGHT, MODE, WIDE, LUT, R, false>(a, kc, job_id, p, jb, qlen, tlen, prog, W, late, stop);
}

}  // namespace

// One workgroup per pair of this launch's job list.  A pair's team is its
// own W waves (jb.team, at most blockDim.x / 64): the waves beyond it end at
// once (s_barrier then waits on the surviving waves only), so pairs of
// different team sizes share one launch.  Wave w computes passes w, w+W,
// ...; then the team runs the pair's epilogue (mqe, start cell, backtrack).
template <bool RIGHT, int MODE, int R, bool LUT>
__global__ void __launch_bounds__(kWave * kMaxTeam) ksw_stripe_kernel(StripeArgs a)
{
    constexpr int SR = kWave * R;
    __shared__ int32_t prog[kMaxTeam];
    __shared__ uint64_t tile[8][64];
    __shared__ int shared_n;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int job = __builtin_amdgcn_readfirstlane(a.order[blockIdx.x]);
    const KswJob jb = a.jobs[job];
    const int W = __builtin_amdgcn_readfirstlane(max(1, min(jb.team, (int)blockDim.x / kWave)));
    if (w >= W) return;
    prog[w] = 0;  // every lane of wave w writes the same zero
    __syncthreads();
    const typename CellOf<RIGHT, MODE>::type kc(a.sc, jb.transposed != 0);
    const int qlen = __builtin_amdgcn_readfirstlane(jb.qlen), tlen = __builtin_amdgcn_readfirstlane(jb.tlen);
    const int npass = ((tlen + SR - 1) / SR + 1) / 2;
    int late = 0, stop = 0;  // (no bounded waits within a workgroup)
    for (int p = w; p < npass && !stop; p += W)
        pass_body<RIGHT, MODE, false, LUT, R>(a, kc, job, p, jb, qlen, tlen, prog, W, late, stop);
    __syncthreads();  // every pass written: stripe partials, score / mte, direction bytes
    StripeLayout<R, MODE> lay(tile);
    pair_epilogue(a, job, jb, lay, &shared_n, W * kWave);
}

// Persistent one-wave workers over a device work queue.  The launch's job
// list is the queue, ordered longest first by the host (length-binned: the
// longest pairs are claimed first, short ones fill the tail); each wave
// claims the next entry with one device-scope atomic add on qhead, runs the
// pair's passes and its epilogue, and claims again until the list is
// exhausted, then ends.  No wave waits on another: a one-wave pair hands
// each pass to the next through the wave's own LDS count.  qhead is zero at
// launch (ksw_stripe_qhead_kernel, a fill kernel rather than a memset so a
// captured graph replays it).
template <bool RIGHT, int MODE, int R, bool LUT>
__global__ void __launch_bounds__(kWave) __attribute__((amdgpu_waves_per_eu(4)))
ksw_stripe_queue_kernel(StripeArgs a, int32_t *qhead)
{
    constexpr int SR = kWave * R;
    __shared__ int32_t prog[1];
    __shared__ uint64_t tile[8][64];
    __shared__ int shared_n;
    for (;;) {
        int idx = 0;
        if (threadIdx.x == 0) idx = __hip_atomic_fetch_add(qhead, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        idx = __builtin_amdgcn_readlane(idx, 0);
        if (idx >= a.njobs) return;
        const int job = __builtin_amdgcn_readfirstlane(a.order[idx]);
        const KswJob jb = a.jobs[job];
        prog[0] = 0;
        __syncthreads();
        const typename CellOf<RIGHT, MODE>::type kc(a.sc, jb.transposed != 0);
        const int qlen = __builtin_amdgcn_readfirstlane(jb.qlen), tlen = __builtin_amdgcn_readfirstlane(jb.tlen);
        const int npass = ((tlen + SR - 1) / SR + 1) / 2;
        int late = 0, stop = 0;
        for (int p = 0; p < npass && !stop; ++p)
            pass_body<RIGHT, MODE, false, LUT, R>(a, kc, job, p, jb, qlen, tlen, prog, 1, late, stop);
        __syncthreads();
        StripeLayout<R, MODE> lay(tile);
        pair_epilogue(a, job, jb, lay, &shared_n, kWave);
        __syncthreads();  // tile and prog are the next pair's
    }
}

// Zeroes the queue heads of a plan's queue launches.
__global__ void __launch_bounds__(64) ksw_stripe_qhead_kernel(int32_t *qhead, int n)
{
    if ((int)threadIdx.x < n) qhead[threadIdx.x] = 0;
}

// Wide teams: each pair has its own run of consecutive blocks (a.wfirst),
// which the dispatcher spreads over the XCDs' CUs; wave v of a team of W
// waves computes passes v, v+W, ...  A pair's control block holds one
// progress count per wave; a wave whose wait gave up raises its late word.
template <bool RIGHT, int MODE, int R, bool LUT>
__global__ void __launch_bounds__(kWave * kMaxTeam) ksw_stripe_wide_kernel(StripeArgs a)
{
    constexpr int SR = kWave * R;
    // the pair of this block: wfirst[slot] <= block < wfirst[slot + 1]
    const int blk = a.wfirst[0] + (int)blockIdx.x;
    int lo = 0, hi = a.njobs;
    while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (a.wfirst[mid] <= blk) lo = mid;
        else hi = mid;
    }
    const int slot = __builtin_amdgcn_readfirstlane(lo);
    const int first = __builtin_amdgcn_readfirstlane(a.wfirst[slot]);
    const int W = __builtin_amdgcn_readfirstlane(a.wfirst[slot + 1] - first) * kWideGroup;
    const int v = __builtin_amdgcn_readfirstlane((blk - first) * kWideGroup + (int)threadIdx.x / kWave);
    const int job = __builtin_amdgcn_readfirstlane(a.order[slot]);
    int32_t *ctl = a.wctl + (int64_t)slot * kWideCtl;
    const KswJob jb = a.jobs[job];
    const typename CellOf<RIGHT, MODE>::type kc(a.sc, jb.transposed != 0);
    const int qlen = __builtin_amdgcn_readfirstlane(jb.qlen), tlen = __builtin_amdgcn_readfirstlane(jb.tlen);
    const int npass = ((tlen + SR - 1) / SR + 1) / 2;
    int late = 0, stop = 0;
    for (int p = v; p < npass && !stop; p += W)
        pass_body<RIGHT, MODE, true, LUT, R>(a, kc, job, p, jb, qlen, tlen, ctl, W, late, stop);
    if ((late || a.force_late) && threadIdx.x % kWave == 0)
        __hip_atomic_store(ctl + kWideCtlLate, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Zeroes the control blocks of a wide launch's pairs (a fill kernel rather
// than a memset, so a captured graph replays it correctly).
__global__ void __launch_bounds__(256) ksw_stripe_wctl_kernel(int32_t *wctl)
{
    int32_t *ctl = wctl + (int64_t)blockIdx.x * kWideCtl;
    for (int k = threadIdx.x; k < kWideCtl; k += blockDim.x) ctl[k] = 0;
}

// The epilogue of every pair of a wide launch, one workgroup per pair, after
// all of the launch's passes.  A pair whose team gave up a wait (its late
// word is raised) is first recomputed by this workgroup as a one-workgroup
// team of kWideGroup waves (LDS progress counts, no cross-workgroup waits),
// into the same direction bytes, column buffer and stripe partials; the
// plan's redo word counts such pairs.
template <bool RIGHT, int MODE, int R, bool LUT>
__global__ void __launch_bounds__(kWave * kWideGroup) ksw_stripe_wide_epilogue_kernel(StripeArgs a)
{
    constexpr int SR = kWave * R;
    __shared__ int32_t prog[kWideGroup];
    __shared__ uint64_t tile[8][64];
    __shared__ int shared_n;
    const int slot = blockIdx.x;
    const int job = __builtin_amdgcn_readfirstlane(a.order[slot]);
    const KswJob jb = a.jobs[job];
    const int late = __builtin_amdgcn_readfirstlane(
        __hip_atomic_load(a.wctl + (int64_t)slot * kWideCtl + kWideCtlLate, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
    if (late) {
        const int w = __builtin_amdgcn_readfirstlane((int)threadIdx.x / kWave);
        prog[w] = 0;
        __syncthreads();
        const typename CellOf<RIGHT, MODE>::type kc(a.sc, jb.transposed != 0);
        const int qlen = __builtin_amdgcn_readfirstlane(jb.qlen), tlen = __builtin_amdgcn_readfirstlane(jb.tlen);
        const int npass = ((tlen + SR - 1) / SR + 1) / 2;
        int late2 = 0, stop = 0;
        for (int p = w; p < npass && !stop; p += kWideGroup)
            pass_body<RIGHT, MODE, false, LUT, R>(a, kc, job, p, jb, qlen, tlen, prog, kWideGroup, late2, stop);
        __syncthreads();
        if (threadIdx.x == 0) atomicAdd(a.werr, 1);
    }
    StripeLayout<R, MODE> lay(tile);
    pair_epilogue(a, job, jb, lay, &shared_n, (int)blockDim.x);
}

// Dispatch over the kernel variants: group (left, right, score-only,
// tracks), rows per lane (8 or 4) and score form (byte table or not).
template <template <bool, int, int, bool> class F, int R, bool LUT, typename... Args>
static auto by_group(int group, Args &&...args)
{
    switch (group) {
    case kGroupRight: return F<true, kDirs, R, LUT>::run(args...);
    case kGroupScoreOnly: return F<false, kScoreOnly, R, LUT>::run(args...);
    case kGroupTracks: return F<false, kTracks, R, LUT>::run(args...);
    default: return F<false, kDirs, R, LUT>::run(args...);
    }
}

template <template <bool, int, int, bool> class F, typename... Args>
static auto by_variant(int group, int R, bool lut, Args &&...args)
{
    if (R != 4) return lut ? by_group<F, 8, true>(group, args...) : by_group<F, 8, false>(group, args...);
    return lut ? by_group<F, 4, true>(group, args...) : by_group<F, 4, false>(group, args...);
}

template <bool RIGHT, int MODE, int R, bool LUT>
struct LaunchStripe {
    static hipError_t run(const StripeArgs &a, int team, hipStream_t st)
    {
        hipLaunchKernelGGL((ksw_stripe_kernel<RIGHT, MODE, R, LUT>), dim3(a.njobs), dim3(kWave * team), 0, st, a);
        return hipGetLastError();
    }
};

template <bool RIGHT, int MODE, int R, bool LUT>
struct LaunchQueue {
    static hipError_t run(const StripeArgs &a, int32_t *qhead, int workers, hipStream_t st)
    {
        hipLaunchKernelGGL((ksw_stripe_queue_kernel<RIGHT, MODE, R, LUT>), dim3(workers), dim3(kWave), 0, st, a, qhead);
        return hipGetLastError();
    }
};

template <bool RIGHT, int MODE, int R, bool LUT>
struct QueueWorkers {
    static int run()
    {
        int per_cu = 0, dev = 0;
        hipDeviceProp_t prop;
        if (hipGetDevice(&dev) != hipSuccess || hipGetDeviceProperties(&prop, dev) != hipSuccess) return 1024;
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, ksw_stripe_queue_kernel<RIGHT, MODE, R, LUT>, kWave, 0) !=
                hipSuccess ||
            per_cu <= 0)
            return prop.multiProcessorCount * 4;
        return per_cu * prop.multiProcessorCount;
    }
};

hipError_t launch_stripe_queue(const StripeArgs &a, int group, int R, bool lut, int32_t *qhead, hipStream_t st)
{
    if (a.njobs <= 0) return hipSuccess;
    if (!qhead || (R != 4 && R != 8) || group < 0 || group >= kGroups) return hipErrorInvalidValue;
    return by_variant<LaunchQueue>(group, R, lut, a, qhead, std::min(a.njobs, stripe_queue_workers(group, R)), st);
}

hipError_t clear_queue_heads(int32_t *qhead, int n, hipStream_t st)
{
    if (n < 1 || n > 64) return hipErrorInvalidValue;
    hipLaunchKernelGGL(ksw_stripe_qhead_kernel, dim3(1), dim3(64), 0, st, qhead, n);
    return hipGetLastError();
}

// Cached per variant: the occupancy query reads the device properties.
int stripe_queue_workers(int group, int R)
{
    static int cache[kGroups][2] = {};
    if (group < 0 || group >= kGroups) group = kGroupLeft;
    const int ri = R == 4 ? 1 : 0;
    if (cache[group][ri] > 0) return cache[group][ri];
    const int n = by_variant<QueueWorkers>(group, R, true);
    __atomic_store_n(&cache[group][ri], n, __ATOMIC_RELAXED);
    return n;
}

hipError_t launch_stripe(const StripeArgs &a, int group, int team, int R, bool lut, hipStream_t st)
{
    if (a.njobs <= 0) return hipSuccess;
    if (team < 1 || team > kMaxTeam || (R != 4 && R != 8) || group < 0 || group >= kGroups) return hipErrorInvalidValue;
    return by_variant<LaunchStripe>(group, R, lut, a, team, st);
}

namespace {

template <bool RIGHT, int MODE, int R, bool LUT>
struct LaunchWide {
    static hipError_t run(const StripeArgs &a0, const int32_t *h_wfirst, int max_wgs, hipStream_t st)
    {
        void (*fn)(StripeArgs) = ksw_stripe_wide_kernel<RIGHT, MODE, R, LUT>;
        StripeArgs a = a0;
        int off = 0;
        while (off < a0.njobs) {
            // as many pairs as fit in max_wgs workgroups (at least one)
            int end = off + 1;
            while (end < a0.njobs && h_wfirst[end + 1] - h_wfirst[off] <= max_wgs) ++end;
            const int blocks = h_wfirst[end] - h_wfirst[off];
            if (blocks > max_wgs) return hipErrorInvalidConfiguration;
            a.order = a0.order + off;
            a.wfirst = a0.wfirst + off;
            a.wctl = a0.wctl + (int64_t)off * kWideCtl;
            a.njobs = end - off;
            hipLaunchKernelGGL(ksw_stripe_wctl_kernel, dim3(a.njobs), dim3(256), 0, st, a.wctl);
            hipLaunchKernelGGL(fn, dim3(blocks), dim3(kWave * kWideGroup), 0, st, a);
            const hipError_t e = hipGetLastError();
            if (e != hipSuccess) return e;
            off = end;
        }
        return hipSuccess;
    }
};

template <bool RIGHT, int MODE, int R, bool LUT>
struct WideCapacity {
    static int run()
    {
        int dev = 0, cus = 0, per_cu = 0;
        if (hipGetDevice(&dev) != hipSuccess ||
            hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
            hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, (const void *)ksw_stripe_wide_kernel<RIGHT, MODE, R, LUT>,
                                                         kWave * kWideGroup, 0) != hipSuccess)
            return 0;
        return cus * per_cu;
    }
};

template <bool RIGHT, int MODE, int R, bool LUT>
struct LaunchWideEpilogue {
    static hipError_t run(const StripeArgs &a, hipStream_t st)
    {
        hipLaunchKernelGGL((ksw_stripe_wide_epilogue_kernel<RIGHT, MODE, R, LUT>), dim3(a.njobs), dim3(kWave * kWideGroup),
                           0, st, a);
        return hipGetLastError();
    }
};

template <bool RIGHT, int MODE, int R, bool LUT>
struct Resident {
    static int run()
    {
        int per_cu = 0, dev = 0;
        hipDeviceProp_t prop;
        if (hipGetDevice(&dev) != hipSuccess || hipGetDeviceProperties(&prop, dev) != hipSuccess) return 1024;
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, ksw_stripe_kernel<RIGHT, MODE, R, LUT>, kWave, 0) !=
                hipSuccess ||
            per_cu <= 0)
            return prop.multiProcessorCount * 4;
        return per_cu * prop.multiProcessorCount;
    }
};

}  // namespace

hipError_t launch_stripe_wide(const StripeArgs &a, int group, int R, bool lut, const int32_t *h_wfirst, int max_wgs,
                              hipStream_t st)
{
    if (a.njobs <= 0) return hipSuccess;
    if (!a.wfirst || !h_wfirst || !a.wctl || !a.werr || max_wgs < 1) return hipErrorInvalidValue;
    if ((R != 4 && R != 8) || group < 0 || group >= kGroups) return hipErrorInvalidValue;
    for (int k = 0; k < a.njobs; ++k) {
        const int n = h_wfirst[k + 1] - h_wfirst[k];
        if (n < 1 || n * kWideGroup > kMaxWide) return hipErrorInvalidValue;
    }
    return by_variant<LaunchWide>(group, R, lut, a, h_wfirst, max_wgs, st);
}

// Cached per variant: the occupancy query reads the device properties.
int stripe_wide_capacity(int group, int R, bool lut)
{
    static int cache[kGroups][2][2] = {};
    if (group < 0 || group >= kGroups) group = kGroupLeft;
    int &c = cache[group][R == 4 ? 1 : 0][lut ? 1 : 0];
    if (c > 0) return c;
    const int n = by_variant<WideCapacity>(group, R, lut);
    __atomic_store_n(&c, n, __ATOMIC_RELAXED);
    return n;
}

hipError_t clear_wide_err(int32_t *werr, hipStream_t st)
{
    hipLaunchKernelGGL(ksw_stripe_wctl_kernel, dim3(1), dim3(256), 0, st, werr);
    return hipGetLastError();
}

hipError_t launch_stripe_wide_epilogue(const StripeArgs &a, int group, int R, bool lut, hipStream_t st)
{
    if (a.njobs <= 0) return hipSuccess;
    if (!a.wctl || !a.werr) return hipErrorInvalidValue;
    if ((R != 4 && R != 8) || group < 0 || group >= kGroups) return hipErrorInvalidValue;
    return by_variant<LaunchWideEpilogue>(group, R, lut, a, st);
}

// Cached per variant: the occupancy query reads the device properties.
int stripe_resident_waves(int group, int R)
{
    static int cache[kGroups][2] = {};
    if (group < 0 || group >= kGroups) group = kGroupLeft;
    const int ri = R == 4 ? 1 : 0;
    if (cache[group][ri] > 0) return cache[group][ri];
    const int n = by_variant<Resident>(group, R, true);
    __atomic_store_n(&cache[group][ri], n, __ATOMIC_RELAXED);
    return n;
}

}  // namespace kswhip
