// ksw2_band.hip -- gfx950 kernel for banded ksw_extd2 calls inside the
// stripe kernel's exactness domain (match 0, mismatch <= 0, the scoring
// bounds that keep every int8 intermediate in range, no z-drop, no
// wildcard), from the narrow bands of certification to w = 4096 and beyond.
//
// The reference sweeps anti-diagonals r; on each it updates the positions
// t of the 16/64-rounded range [stB, en16] in place
// (minimap2/ksw2_extd2_avx.c:248-745): a cell reads x, v, x2 of position t-1
// and u, y, y2, s of position t as they were left by earlier anti-diagonals
// (stale outside the band), with the boundary rules of
// minimap2/ksw2_extd2_sse.c:158-172 (injection at st16, the AVX-512 lane
// wrap at a non-64-aligned start, row r re-initialised at column 0).  This
// kernel evaluates the same cells in (t, r) coordinates:
//
//  * Stripes.  The positions are cut into stripes of 128; lane k of a wave
//    holds positions t0 + 2k and t0 + 2k + 1 in the halves of its registers
//    (the in-place state u, v, x, y, x2, y2, the score s, and H in 32 bits)
//    and steps through the anti-diagonals that reach the stripe.  A position
//    takes the one above it through a DPP shift, the stripe's first from the
//    stripe above through a hand-off.  Every lane computes every step: a
//    position above en16 is set to the initial state when it enters the band,
//    and below stB nothing reads it.
//  * Why 128 positions.  A banded pair's time is its chain of anti-diagonals,
//    so what counts is the length of a step: one packed cell here (two, and
//    H of four positions, at 256 positions a stripe).  A stripe starts 256
//    anti-diagonals after the one above it, plus what the hand-off costs.
//  * Waves.  Wave w of a pair's W takes stripes w, w + W, ...; about
//    (2w + 420) / 256 are in flight.  They sit in workgroups of four, one wave
//    per SIMD.  A stripe's last position (x, x2, v, H, one entry per
//    anti-diagonal) goes to the next wave of a workgroup through a ring in
//    LDS, four anti-diagonals at a time, and from the last wave of a workgroup
//    to the first of the next through the pair's buffer in device memory, 16
//    at a time: two device-scope 8-byte stores per entry that carry the
//    reading stripe's number, which the reader looks for, so no count is
//    published and nothing waits for a store to complete.  One buffer
//    serves all stripes: an entry is overwritten three stripes and at least
//    three anti-diagonals after the block that holds it has been read.
//  * A wait on device memory that outlasts 10 s (a workgroup the dispatcher
//    could not place) gives up: the pair is flagged for the general kernel,
//    which recomputes it, and every wave still runs to its end.  Waits in LDS
//    are on waves of the same workgroup.
//  * Steps go in blocks of 16, aligned so that the band's end moves on even
//    steps and its start on odd ones.  A block in which neither end is near
//    the stripe, or only one of them, or clear of the rare rules (column 0,
//    t == r, the last position, row and anti-diagonal) runs unrolled without
//    the tests it does not need; the others go step by step with every rule.
//  * H bookkeeping (minimap2/ksw2_extd2_sse.c:332-375): H[en0] from the
//    position above plus u, H[t] += v on [st0, en0), mte on position tlen-1,
//    mqe where column qlen-1 is the band's start, the score at the last
//    anti-diagonal.  Held as -8 H + p r (p the bias of v and u), so one
//    v_dot2 adds a half of v.  The maximum is not tracked: H never exceeds
//    ez->max's initial 0.  (Every z is <= 0, capped at the match score.  Let
//    K(t, r) = H(t, r) - u(t, r).  A position enters the band with K = H of
//    the position above, and on the next anti-diagonal H = K + z and K grows
//    by the v it takes from above, as H of the position above does; where it
//    takes the initial v instead, at st16, K falls.  So K <= 0 and H <= 0.)
//  * Band exit (st > en) is pure geometry: the host passes the number of
//    anti-diagonals the reference completes.
//
// Outputs: direction bytes in the reference's row layout
// (p[r * n_col*64 + t - off[r]], off[r] = stB, off_end[r] = en16), so the
// general backtrack kernel walks them; the KswOut fields; the redo flag.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>
#include <type_traits>

#include "ksw2_cell.h"
#include "ksw2_common.h"
#include "ksw2_kernels.h"

namespace kswhip {

namespace {

using cell::add_hi;
using cell::add_lo;
using cell::bfi;
using cell::dpp_shr1;
using cell::hi16;
using cell::lo16;
using cell::perm;
using cell::sign2;
using cell::splat;
using cell::sub2;

constexpr int SR = kBandStripe;                 // positions per stripe
constexpr int kBlock = 16;                      // anti-diagonals per block
constexpr uint64_t kWaitTicks = 1000000000ull;  // 10 s of the 100 MHz real-time clock
constexpr int kDeviceLooks = 1024, kRingLooks = 16384;  // at an entry or a count, between two at the stop flag

struct Band {
    int st0, en0, st16, en16, stB, sc_end;
};

// Band of anti-diagonal r (minimap2/ksw2_extd2_sse.c:147-156) and the
// ranges derived from it: the 16-rounded start/end, the 64-block start and
// the last position whose score is written (16-byte groups from st0, or
// exactly en0 with KSW_EZ_GENERIC_SC, ksw2_extd2_sse.c:173-193).
__device__ __forceinline__ Band band_of(int r, int qlen, int tlen, int w, int tlenB, bool generic)
{
    int st = 0, en = tlen - 1;
    if (st < r - qlen + 1) st = r - qlen + 1;
    if (en > r) en = r;
    if (st < (r - w + 1) >> 1) st = (r - w + 1) >> 1;
    if (en > (r + w) >> 1) en = (r + w) >> 1;
    // (0 <= st <= en: the 16- and 64-roundings are masks)
    Band b;
    b.st0 = st, b.en0 = en;
    b.st16 = st & ~15, b.en16 = en | 15, b.stB = st & ~63;
    b.sc_end = generic ? en : min(st + ((en - st + 16) & ~15) - 1, tlenB - 1);
    return b;
}

// A wave's hand-off ring: the entries of the position above its stripe (x, x2
// and v in the high halves, H) and the query codes of its first position, one
// per anti-diagonal: entry c is the state as anti-diagonal c - 1 left it.  The
// wave above writes the entries (the first wave of a workgroup its own, from
// the pair's buffer; the last writes the ring past its own and copies it there).
constexpr int kRing = 256;
struct BandRing {
    uint32_t e[5][kRing];
    int32_t filled, taken;  // anti-diagonals written and read, counted from stripe kk of the wave at kk * span
    int32_t pad[14];
};
// The lanes that hold no stripe's last position write to the space after a
// workgroup's rings.
constexpr int ring_bytes(int waves)
{
    return (waves + 1) * (int)sizeof(BandRing) + (int)sizeof(uint32_t) * (3 * kRing + kWave + kBlock);
}

__device__ __forceinline__ int32_t ring_load(const int32_t *x)
{
    return __builtin_amdgcn_readfirstlane(__hip_atomic_load(x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP));
}
// (a wave's LDS operations complete in order, so a count stored after an
// entry is seen after it; the empty asm keeps the compiler to that order)
__device__ __forceinline__ void ring_store(int32_t *x, int32_t v)
{
    asm volatile("" ::: "memory");
    __hip_atomic_store(x, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

// Entry of the pair's buffer: two dwords with the reader's number in the low
// half of the second, and H with that number.
__device__ __forceinline__ uint64_t load_half(const int32_t *buf, int r, int k)
{
    return __hip_atomic_load((const uint64_t *)buf + 2 * r + k, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void store_half(int32_t *buf, int r, int k, uint32_t a, uint32_t b)
{
    __hip_atomic_store((uint64_t *)buf + 2 * r + k, (uint64_t)a | (uint64_t)b << 32, __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ uint32_t reader_tag(int s) { return (uint32_t)(s % 65535 + 1); }  // never 0

__device__ __forceinline__ uint32_t part(const uint4 &x, int k) { return k == 0 ? x.x : k == 1 ? x.y : k == 2 ? x.z : x.w; }

}  // namespace

// The band's blocks are placed so that (r + w) % 16 == 0 at their first
// anti-diagonal; `c` below is r + (w % 16).  What bounds it: the chain of a
// pair's anti-diagonals, a step of 54 (neither end of the band in the stripe)
// to 67 instructions (its start), and some 20 a step around them, of a wave
// alone on its SIMD.  Measured, against stripes of 256 positions handed on
// through progress counts in device memory: a pair of 20 kbp, w = 256, 1.1 and
// 0.24 us per anti-diagonal; 16 pairs of 60-120 kbp, w = 4096, 213 and 64 ms;
// 2,048 pairs of 2 kbp, w = 256, 26 ms on the general kernel and 4.5 ms here.
template <bool RIGHT, bool SCORE_ONLY>
__global__ void __launch_bounds__(kWave * kBandGroup) __attribute__((amdgpu_waves_per_eu(3))) ksw_band_kernel(BandArgs a)
{
    extern __shared__ __align__(16) uint8_t band_lds[];
    BandRing *rings = (BandRing *)band_lds;
    const int group = blockDim.x / kWave, lane = threadIdx.x % kWave;
    const int wgs = a.wgs, g = blockIdx.x % wgs;
    const int W = __builtin_amdgcn_readfirstlane(wgs * group);
    const int w = __builtin_amdgcn_readfirstlane((int)threadIdx.x / kWave);
    const int wv = __builtin_amdgcn_readfirstlane(g * group + w);
    if ((int)threadIdx.x <= group) rings[threadIdx.x].filled = rings[threadIdx.x].taken = 0;
    __syncthreads();
    const int job = __builtin_amdgcn_readfirstlane(a.order[blockIdx.x / wgs]);
    const GenJob jb = a.jobs[job];
    const int qlen = __builtin_amdgcn_readfirstlane(jb.qlen), tlen = __builtin_amdgcn_readfirstlane(jb.tlen);
    const int bw = __builtin_amdgcn_readfirstlane(jb.w), flag = __builtin_amdgcn_readfirstlane(jb.flag);
    const int tlenB = __builtin_amdgcn_readfirstlane(jb.tlenB), r_end = __builtin_amdgcn_readfirstlane(jb.r_end);
    const int ncolB = __builtin_amdgcn_readfirstlane(jb.ncolB);
    const bool generic = flag & 0x04;
    const int nr = qlen + tlen - 1;
    const KswScore &sc = a.sc.k;
    cell::DirCell<RIGHT> kc(sc, false);
    const uint8_t *qs = a.seq + jb.q_off, *ts = a.seq + jb.t_off;
    uint8_t *p = a.dir + jb.dir_off;
    int32_t *off = a.offs + jb.off_off, *off_end = off + nr;
    int32_t *ctl = a.bnd + jb.bnd_off;  // control block and buffer (cleared before the launch)
    int32_t *buf = ctl + kBandCtl;

    if (!SCORE_ONLY)
        for (int r = g * (int)blockDim.x + (int)threadIdx.x; r < r_end; r += wgs * (int)blockDim.x) {
            const Band b = band_of(r, qlen, tlen, bw, tlenB, generic);
            off[r] = b.stB, off_end[r] = b.en16;
        }

    uint32_t v_init = splat(kc.diff(-sc.G1)), sm2 = splat(kc.sm), sd2 = splat(kc.sx - kc.sm);
    // (in vector registers: the scalar ones run out, and are then kept in lanes)
    asm volatile("" : "+v"(v_init), "+v"(sm2), "+v"(sd2), "+v"(kc.cA2), "+v"(kc.cB2), "+v"(kc.zc), "+v"(kc.e1), "+v"(kc.e2));
    asm volatile("" : "+v"(kc.lA), "+v"(kc.lB), "+v"(kc.lA2), "+v"(kc.lB2), "+v"(kc.mA), "+v"(kc.mB), "+v"(kc.mA2));
    uint32_t one = 0x00010001u;
    asm volatile("" : "+s"(one));
    const int wofs = bw & 15, span = nr + 64;
    const int nstripes = (tlenB + SR - 1) / SR;
    // anti-diagonals that touch positions [t0, t0 + SR): computed when
    // stB <= t <= en16, scored when st0 <= t <= sc_end <= en0 + 15
    auto lo_of = [&](int t0) { return max(0, max(t0 - 16, 2 * t0 - 32 - bw)); };
    auto hi_of = [&](int t0) { return min(r_end - 1, min(qlen + t0 + SR - 2, 2 * (t0 + SR - 1) + bw)); };
    auto start_of = [&](int t0) { return lo_of(t0) + wofs & ~(kBlock - 1); };
    // (and two on, whose entries say what the last one left: the position after
    // the stripe can be the band's only one on both)
    auto end_of = [&](int t0) { return (hi_of(t0) + 2 + wofs | (kBlock - 1)) + 1; };

    // per-lane results over this wave's stripes
    int mqe_h = KSW_NEG_INF_I, mqe_t = -1, mte_h = KSW_NEG_INF_I, mte_q = -1, score = KSW_NEG_INF_I;
    int late = 0, stop = 0;
    auto stopped = [&]() {
        if (a.stop)
            stop = __builtin_amdgcn_readfirstlane(__hip_atomic_load(a.stop, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM));
        return stop != 0;
    };
    // (while waiting it is looked at now and then, every millisecond or two:
    // the load goes over the bus)
    int spins = 0;
    auto stopped_waiting = [&](int looks) { return (++spins & (looks - 1)) == 0 ? stopped() : stop != 0; };
    // one workgroup of as many waves as stripes in flight: the last hands on to
    // the first through the first's ring (with fewer, each would wait for room
    // in the next one's ring, the last for a stripe that the first has yet to
    // begin)
    const bool circle = wgs == 1 && group > 1 && 2 * bw + 420 <= 256 * W;
    BandRing &in = rings[w], &out = rings[circle && w + 1 == group ? 0 : w + 1];
    uint32_t *const spill = (uint32_t *)(rings + group + 1);
    auto has_stripe = [&](int s) { return s < nstripes && lo_of(s * SR) <= hi_of(s * SR); };
    // stripe s, the kk-th of this wave.  FED: its entries come from another
    // wave of the workgroup; LEAVES: its own go to the pair's buffer
    auto stripe = [&](int s, int kk, auto fed_by_wave, auto to_buffer) {
        constexpr bool FED = decltype(fed_by_wave)::value, LEAVES = decltype(to_buffer)::value;
        const int t0 = s * SR, tl = t0 + 2 * lane;
        const int r_hi = hi_of(t0), c_lo = start_of(t0), c_end = end_of(t0);
        const int base = kk * span, in_base = w > 0 ? base : base - span;  // of this stripe's counts and the one's above
        const int p_lo = s > 0 ? start_of(t0 - SR) : 0, p_end = s > 0 ? end_of(t0 - SR) : 0;
        const int p_hi = s > 0 ? hi_of(t0 - SR) : -2;
        const bool has_next = LEAVES || has_stripe(s + 1);
        const int n_lo = has_next ? start_of(t0 + SR) : 0;
        const bool feeds = !LEAVES && has_next, enters = !FED && s > 0;
        const uint32_t tag = reader_tag(s), next_tag = reader_tag(s + 1);

        cell::Right st;
        cell::Down dn;
        st.u = dn.v = v_init, st.y = kc.y0(), st.y2 = kc.y20(), dn.x = kc.x0(), dn.x2 = kc.x20();
        uint32_t sco = sm2;  // the score candidates (the match score until first written)
        int h0 = 0, h1 = 0;
        auto qcode = [&](int j) { return j >= 0 && j < qlen ? (uint32_t)qs[j] : 0u; };
        const uint32_t tb = (tl < tlen ? (uint32_t)ts[tl] : 0u) | (tl + 1 < tlen ? (uint32_t)ts[tl + 1] << 16 : 0u);
        uint32_t qb = qcode(c_lo - wofs - 1 - tl) | qcode(c_lo - wofs - 2 - tl) << 16;
        const uint32_t pos = ((uint32_t)tl & 0xffffu) | (uint32_t)(tl + 1) << 16;

        // ---- a block's query codes and (the first wave of a workgroup) its
        // entries from the pair's buffer: asked for a block ahead, put into
        // the ring 12 steps later
        uint64_t na = 0, nh = 0;
        uint32_t nq = 0;
        auto entry_valid = [&](int c) { return lane < kBlock && c >= p_lo && c - wofs >= 0 && c - wofs <= min(p_hi + 2, nr); };
        auto fetch = [&](int cb) {
            const int c = cb + lane, j = c - wofs - t0;
            nq = qs[min(max(j, 0), qlen - 1)];
            if (enters) {
                const int r = min(max(c - wofs, 0), nr);
                na = load_half(buf, r, 0), nh = load_half(buf, r, 1);
            }
        };
        auto fill = [&](int cb) {
            const int c = cb + lane, j = c - wofs - t0, k = c & (kRing - 1);
            if (lane < kBlock) in.e[4][k] = j >= 0 && j < qlen ? nq << 16 : 0u;
            if (enters) {
                const bool have = entry_valid(c);
                auto missing = [&]() {
                    return __ballot(have && ((uint32_t)(na >> 32 & 0xffffu) != tag || (uint32_t)(nh >> 32) != tag)) != 0;
                };
                if (__builtin_expect(missing() && !late && !stop, 0)) {
                    // not all written yet: load again until they are
                    const uint64_t t_start = wall_clock64();
                    for (;;) {
                        if (have) na = load_half(buf, c - wofs, 0), nh = load_half(buf, c - wofs, 1);
                        if (!missing() || stopped_waiting(kDeviceLooks)) break;
                        if (wall_clock64() - t_start > kWaitTicks) {
                            late = 1;
                            break;
                        }
                    }
                }
                if (lane < kBlock)
                    in.e[0][k] = (uint32_t)na, in.e[1][k] = (uint32_t)na << 16, in.e[2][k] = (uint32_t)(na >> 32),
                    in.e[3][k] = (uint32_t)nh;
            }
        };
        // ---- four anti-diagonals' entries
        int known = FED ? 0 : 0x7fffffff;
        // (what: the arrays that the steps after these can need)
        auto read4 = [&](int c, uint4 (&e)[5], auto what) {
            constexpr int WHAT = decltype(what)::value;
            if (FED && (WHAT & 7) && __builtin_expect(known < in_base + min(c + 4, p_end), 0)) {
                while ((known = ring_load(&in.filled)) < in_base + min(c + 4, p_end)) {
                    if (stopped_waiting(kRingLooks)) break;
                    __builtin_amdgcn_s_sleep(1);
                }
            }
            asm volatile("" ::: "memory");  // the entries are read after their count
#pragma unroll
            for (int k = 0; k < 5; ++k)
                if (WHAT >> k & 1) e[k] = *(const uint4 *)&in.e[k][c & (kRing - 1)];
        };
        // ---- a block's entries from the ring to the pair's buffer
        uint32_t b0 = 0, b1 = 0, b2 = 0, b3 = 0;
        auto take = [&](int cb) {
            asm volatile("" ::: "memory");
            const uint32_t *o = out.e[0] + (cb & (kRing - 1)) + min(lane, kBlock - 1);
            b0 = o[0], b1 = o[kRing], b2 = o[2 * kRing], b3 = o[3 * kRing];
        };
        auto hand_on = [&](int cb) {
            const int r = cb + lane - wofs;
            if (lane < kBlock && r >= 0 && r <= min(r_hi + 2, nr)) {
                store_half(buf, r, 0, perm(b0, b1, 0x07060302u), bfi(0xffff0000u, b2, next_tag));
                store_half(buf, r, 1, b3, next_tag);
            }
        };

        fetch(c_lo);
        fill(c_lo);
        uint4 e[5], f[5];
        read4(c_lo, e, std::integral_constant<int, 31>());
        int room = feeds ? ring_load(&out.taken) : 0;
        int slot[4];  // where this lane writes the block's first entry, as offsets in LDS
        // the state handed on, and the inputs from the position above
        uint32_t tx, tx2, tv;
        int th;
        auto begin = [&](int i, int k, const uint4 (&e)[5]) {
            auto o = [&](int x) -> uint32_t & { return *(uint32_t *)(band_lds + slot[x] + 4 * i); };
            o(0) = dn.x, o(1) = dn.x2, o(2) = dn.v, o(3) = (uint32_t)h1;
            qb = __builtin_amdgcn_alignbit(qb, dpp_shr1(part(e[4], k), qb), 16);
        };
        // the position above's x, x2 and v: the stripe's first position takes
        // the entry's
        auto from_above = [&](int k, const uint4 (&e)[5]) {
            tx = dpp_shr1(part(e[0], k), dn.x), tx2 = dpp_shr1(part(e[1], k), dn.x2), tv = dpp_shr1(part(e[2], k), dn.v);
        };
        auto score_of = [&]() {
            const cell::v2u mm = __builtin_elementwise_min(__builtin_bit_cast(cell::v2u, tb ^ qb),
                                                           __builtin_bit_cast(cell::v2u, one));
            return __builtin_bit_cast(uint32_t, __builtin_bit_cast(cell::v2u, sm2) + mm * __builtin_bit_cast(cell::v2u, sd2));
        };
        auto shift = [&]() {
            dn.x = __builtin_amdgcn_alignbit(dn.x, tx, 16), dn.x2 = __builtin_amdgcn_alignbit(dn.x2, tx2, 16);
            dn.v = __builtin_amdgcn_alignbit(dn.v, tv, 16);
        };
        // lanes whose positions enter the band: the initial state
        auto enter = [&](bool mine) {
            const uint32_t m = mine ? ~0u : 0u;
            st.u = bfi(m, v_init, st.u), st.y = bfi(m, kc.y0(), st.y), st.y2 = bfi(m, kc.y20(), st.y2);
            dn.v = bfi(m, v_init, dn.v), dn.x = bfi(m, kc.x0(), dn.x), dn.x2 = bfi(m, kc.x20(), dn.x2);
        };

#pragma unroll 1
        for (int cb = c_lo; cb < c_end; cb += kBlock) {
            // the host's stop flag, every 256 anti-diagonals: end (nothing of
            // this pair is delivered; the waves that wait read the flag too)
            if (__builtin_expect((cb & 255) == 0 && stopped(), 0)) break;
            const int r0 = cb - wofs, r15 = r0 + kBlock - 1, nb = cb + kBlock;
            if (feeds) {
                // the entries it overwrites have been read (by the stripe
                // after this one, or that wave's stripe before)
                const int need = nb - kRing > n_lo ? base + nb - kRing : base;
                while (__builtin_expect(room < need, 0)) {
                    if (stopped_waiting(kRingLooks)) break;
                    __builtin_amdgcn_s_sleep(1);
                    room = ring_load(&out.taken);
                }
            }
            slot[0] = (int)((uint8_t *)(lane == kWave - 1 && has_next ? out.e[0] + (cb & (kRing - 1)) : spill + lane) - band_lds);
#pragma unroll
            for (int k = 1; k < 4; ++k) {
                // (a register each: one base took an addition for each store)
                slot[k] = slot[k - 1] + 4 * kRing;
                asm volatile("" : "+v"(slot[k]));
            }
            // around each four steps
            int pr = 0;
            auto before4 = [&](int i, uint4 (&next)[5], auto what) {
                if (FED && (decltype(what)::value & 7)) pr = __hip_atomic_load(&in.filled, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                if (i == 0) {
                    if (LEAVES) take(cb - kBlock);
                    fetch(nb);
                }
                if (i == kBlock - 4) fill(nb);
                read4(cb + i + 4, next, what);
            };
            auto after4 = [&](int i, auto what) {
                if (feeds) ring_store(&out.filled, base + cb + i + 4);
                if (FED && (decltype(what)::value & 7)) known = __builtin_amdgcn_readfirstlane(pr);
                if (i == 0 && LEAVES && cb > c_lo) hand_on(cb - kBlock);
            };
            // the band's ends move as 2r -+ w, nothing rare in the block
            const int S0 = (r0 - bw) >> 1, E0 = (r0 + bw) >> 1;
            const bool plain = r0 >= 16 && E0 + 7 + 15 < tlenB && S0 >= 16 && bw < 30000 && r0 - E0 > 15 && E0 + 7 < tlen - 1 && r15 <= r_hi && r15 < nr - 1 &&
                               r15 - (S0 + 8) < qlen - 1;
            auto block = [&](auto edges) {
                constexpr bool START = decltype(edges)::value & 1, END = decltype(edges)::value & 2;
                const __amdgpu_buffer_rsrc_t rows =
                    __builtin_amdgcn_make_buffer_rsrc(p + (uint64_t)r0 * ncolB, 0, 0x7fffffff, 0x00027000);
                int soff = 0;               // of the anti-diagonal's row, less what stB moved by
                uint32_t m16 = 0, mB = 0;   // lanes of st16 (when it takes the initial values) and of a wrapped stB
                const int B0 = S0 & ~63;
                int voff = tl - B0;         // of this lane's bytes in the row (out of range: none stored)
                auto set_start = [&](int b_st, bool kept) {
                    const int stB = b_st & ~63, st16 = b_st & ~15;
                    m16 = !kept && tl == st16 ? ~0u : 0u;
                    mB = st16 != stB && tl == stB ? ~0u : 0u;
                    voff = tl < stB ? -1 : tl - B0;
                };
                auto move_start = [&](int b_st, bool kept) {
                    asm volatile("");  // (a branch, not selects)
                    const int cut = voff;
                    set_start(b_st, kept);
                    if (END) voff = cut < 0 ? cut : voff;
                };
                uint32_t below = 0;         // START: pos - st0
                uint32_t e0 = 0, e1 = 0;    // END: masks of the low and high position at en0
                if (START) set_start(S0, false), below = sub2(pos, splat(S0));
                if (END) {
                    if (__builtin_expect((E0 & 15) == 0, 0)) enter((unsigned)(tl - E0) < 16u);
                    voff = tl < (E0 | 15) ? voff : -1;
                    e0 = tl == E0 ? ~0u : 0u, e1 = tl + 1 == E0 ? ~0u : 0u;
                }
                // END: the last scored position - pos, on even and odd steps
                // (it is at most en0 + 15, short of tlenB in a plain block)
                uint32_t above0 = 0, above1 = 0;
                if (END) {
                    above0 = sub2(splat(S0 + (generic ? bw : ((bw + 16) & ~15) - 1)), pos);
                    above1 = sub2(splat(S0 + 1 + (generic ? bw - 1 : ((bw + 15) & ~15) - 1)), pos);
                }
                // four steps from i4; MOVES: st16 moves on in them
                auto steps4 = [&](int i4, auto moves, const uint4 (&e)[5]) {
                    constexpr bool MOVES = decltype(moves)::value;
                    const int s4 = S0 + (i4 >> 1);
#pragma unroll
                    for (int k = 0; k < 4; ++k) {
                        const int b_st = s4 + ((k + 1) >> 1);
                        begin(i4 + k, k, e);
                        if (k % 2 == 1) {
                            // (stB moves on only where st16 does)
                            if (MOVES || !START) soff -= (b_st & 63) == 0 ? 64 : 0;
                            if (START) below = sub2(below, one);
                        }
                        if (MOVES && k > 0 && __builtin_expect((b_st & 15) == 0, 0)) {
                            // (st16 - 1 was computed on the anti-diagonal before)
                            move_start(b_st, k % 2 == 1);
                        }
                        if (END && k % 2 == 0) th = (int)dpp_shr1(part(e[3], k), (uint32_t)h1);
                        // (START alone: the stripe's first position is below the
                        // start or takes its values)
                        if (START && !END)
                            tx = cell::dpp_shr1_0(dn.x), tx2 = cell::dpp_shr1_0(dn.x2), tv = cell::dpp_shr1_0(dn.v);
                        else
                            from_above(k, e);
                        if (START) {
                            // (position stB + 15 is seven lanes after stB's, lane 0 or 32)
                            tx = bfi(m16, kc.x0(), bfi(mB, cell::dpp_row_shl7(dn.x), tx));
                            tx2 = bfi(m16, kc.x20(), bfi(mB, cell::dpp_row_shl7(dn.x2), tx2));
                            tv = bfi(m16, v_init, bfi(mB, cell::dpp_row_shl7(dn.v), tv));
                        }
                        shift();
                        const uint32_t sn = score_of();
                        uint32_t keep = 0;  // halves that keep their score
                        if (START) keep = below;
                        if (END) {
                            uint32_t &above = k % 2 ? above1 : above0;
                            keep = START ? keep | above : above;
                            above = cell::add2(above, one);
                        }
                        sco = START || END ? bfi(sign2(keep), sco, sn) : sn;
                        const cell::DirWord o = kc.template step<true>(sco, dn, st);
                        if (END && k % 2 == 0) {
                            // en0 is one on from the step before: H from the
                            // position above (on odd steps H + v is the same)
                            const int c0 = add_lo(st.u, th), c1 = add_hi(st.u, h0);
                            h0 = (int)bfi(e0, (uint32_t)c0, (uint32_t)add_lo(dn.v, h0));
                            h1 = (int)bfi(e1, (uint32_t)c1, (uint32_t)add_hi(dn.v, h1));
                            const uint32_t t = e0;  // where it moves to
                            e0 = cell::dpp_shr1_0(e1), e1 = t;
                        } else {
                            h0 = add_lo(dn.v, h0), h1 = add_hi(dn.v, h1);
                        }
                        if (!SCORE_ONLY)
                            __builtin_amdgcn_raw_buffer_store_b16((short)cell::DirCell<RIGHT>::pack1(o), rows, voff, soff, 0);
                        soff += ncolB;
                    }
                };
#pragma unroll
                for (int i4 = 0; i4 < kBlock; i4 += 4) {
                    // (a group's entries are loaded during the one before it,
                    // into the arrays in turn)
                    const int s4 = S0 + (i4 >> 1);
                    const uint4 (&now)[5] = i4 & 4 ? f : e;
                    const auto what = std::integral_constant<int, END ? 31 : START ? 16 : 23>();
                    before4(i4, i4 & 4 ? e : f, what);
                    if (START && i4 > 0 && __builtin_expect((s4 & 15) == 0, 0)) move_start(s4, false);
                    if (START && END) steps4(i4, std::true_type(), now);
                    else if (START && __builtin_expect((s4 + 2 & 15) < 2, 0)) steps4(i4, std::true_type(), now);
                    else steps4(i4, std::false_type(), now);
                    after4(i4, what);
                }
            };
            if (__builtin_expect(plain, 1)) {
                const bool starts = S0 + 8 >= t0, ends = t0 + SR - 1 >= E0;
                if (!starts && !ends) block(std::integral_constant<int, 0>());
                else if (!ends && S0 > t0) block(std::integral_constant<int, 1>());
                else if (!starts) block(std::integral_constant<int, 2>());
                else block(std::integral_constant<int, 3>());
            } else {
                // every rule
                int lst16 = -1, len16 = -1;  // st16, en16 of anti-diagonal r-1
                if (r0 > 0 && r0 <= r_hi) {
                    const Band bp = band_of(r0 - 1, qlen, tlen, bw, tlenB, generic);
                    lst16 = bp.st16, len16 = bp.en16;
                }
#pragma unroll 1
                for (int i4 = 0; i4 < kBlock; i4 += 4) {
                    before4(i4, f, std::integral_constant<int, 31>());
#pragma unroll
                    for (int k = 0; k < 4; ++k) {
                        const int r = r0 + i4 + k;
                        begin(i4 + k, k, e);
                        if (r < 0 || r > r_hi) {
                            h0 += kc.p, h1 += kc.p;  // H stays
                            continue;
                        }
                        from_above(k, e);
                        const Band b = band_of(r, qlen, tlen, bw, tlenB, generic);
                        th = (int)dpp_shr1(part(e[3], k), (uint32_t)h1);
                        if (b.en16 != len16) {
                            // (what lane 0 takes from the stripe above is that
                            // position's, whatever enters)
                            enter(tl > len16 && tl <= b.en16);
                            from_above(k, e);
                        }
                        const bool keep_prev = b.st16 > 0 && b.st16 - 1 >= lst16 && b.st16 - 1 <= len16;
                        const uint32_t edge = splat(kc.diff(edge_diff(sc, r)));
                        if (b.st16 != b.stB) {
                            const int wl = (b.stB + 15 - t0) / 2 & (kWave - 1);
                            const uint32_t wx = (uint32_t)__builtin_amdgcn_readlane((int)dn.x, wl);
                            const uint32_t wx2 = (uint32_t)__builtin_amdgcn_readlane((int)dn.x2, wl);
                            const uint32_t wvv = (uint32_t)__builtin_amdgcn_readlane((int)dn.v, wl);
                            if (tl == b.stB) tx = wx, tx2 = wx2, tv = wvv;
                        }
                        if (tl == b.st16 && !keep_prev) tx = kc.x0(), tx2 = kc.x20(), tv = b.st16 == 0 ? edge : v_init;
                        if (b.en16 >= r) {
                            const uint32_t m = tl == r ? 0x0000ffffu : tl + 1 == r ? 0xffff0000u : 0u;
                            st.u = bfi(m, edge, st.u), st.y = bfi(m, kc.y0(), st.y), st.y2 = bfi(m, kc.y20(), st.y2);
                        }
                        shift();
                        const uint32_t scored = (tl >= b.st0 && tl <= b.sc_end ? 0x0000ffffu : 0u) |
                                                (tl + 1 >= b.st0 && tl + 1 <= b.sc_end ? 0xffff0000u : 0u);
                        sco = bfi(scored, score_of(), sco);
                        const cell::DirWord o = kc.template step<true>(sco, dn, st);
                        // H on [st0, en0]; elsewhere it stays
                        int n0 = h0 + (tl >= b.st0 && tl < b.en0 ? lo16(dn.v) : kc.p);
                        int n1 = h1 + (tl + 1 >= b.st0 && tl + 1 < b.en0 ? hi16(dn.v) : kc.p);
                        if (r == 0) {
                            if (tl == 0) n0 = lo16(dn.v) - kc.p + 8 * sc.qe_orig;
                        } else if (b.en0 == 0) {
                            if (tl == 0) n0 = h0 + lo16(dn.v);
                        } else {
                            if (tl == b.en0) n0 = th + lo16(st.u);
                            if (tl + 1 == b.en0) n1 = h0 + hi16(st.u);
                        }
                        h0 = n0, h1 = n1;
                        const int q0 = (kc.p * r - h0) >> 3, q1 = (kc.p * r - h1) >> 3;  // H
                        if (b.en0 == tlen - 1 && (tl | 1) == (b.en0 | 1)) {
                            const int h = b.en0 & 1 ? q1 : q0;
                            if (h >= mte_h) mte_h = h, mte_q = r - b.en0;
                            if (r == nr - 1) score = h;
                        }
                        if (r - b.st0 == qlen - 1 && (tl | 1) == (b.st0 | 1)) {
                            const int h = b.st0 & 1 ? q1 : q0;
                            if (h >= mqe_h) mqe_h = h, mqe_t = b.st0;
                        }
                        if (!SCORE_ONLY && tl >= b.stB && tl < b.en16)
                            *(uint16_t *)(p + (uint64_t)r * ncolB + (tl - b.stB)) =
                                (uint16_t)cell::DirCell<RIGHT>::pack1(o);
                        lst16 = b.st16, len16 = b.en16;
                    }
                    after4(i4, std::integral_constant<int, 31>());
#pragma unroll
                    for (int k = 0; k < 5; ++k) e[k] = f[k];
                }
            }
            if (FED) ring_store(&in.taken, in_base + (nb >= p_end ? span : nb));
            if (feeds) room = ring_load(&out.taken);
        }
        if (LEAVES) take(c_end - kBlock), hand_on(c_end - kBlock);
        if (FED) ring_store(&in.taken, in_base + span);
    };
#pragma unroll 1
    for (int s = wv, kk = 0; has_stripe(s) && !stop; s += W, ++kk) {
        const bool fed = s > 0 && (w > 0 || circle), leaves = w + 1 == group && !circle && has_stripe(s + 1);
        if (fed && !leaves) stripe(s, kk, std::true_type(), std::false_type());
        else if (fed) stripe(s, kk, std::true_type(), std::true_type());
        else if (!leaves) stripe(s, kk, std::false_type(), std::false_type());
        else stripe(s, kk, std::false_type(), std::true_type());
    }

    // ---- results: mte and the score come from one position; mqe keeps the
    // largest H, ties to the later anti-diagonal (the larger t)
#pragma unroll
    for (int o = 1; o < kWave; o <<= 1) {
        const int oh = __shfl_xor(mqe_h, o, kWave), ot = __shfl_xor(mqe_t, o, kWave);
        if (oh > mqe_h || (oh == mqe_h && ot > mqe_t)) mqe_h = oh, mqe_t = ot;
        const int th = __shfl_xor(mte_h, o, kWave), tq = __shfl_xor(mte_q, o, kWave);
        if (tq >= 0 && (mte_q < 0 || th > mte_h)) mte_h = th, mte_q = tq;
        score = max(score, __shfl_xor(score, o, kWave));
    }
    // each wave leaves its record; the last to take a ticket combines them
    // in wave order and writes the pair's results
    int32_t *rec = ctl + kBandCtlRec;
    int last = 0;
    if (lane == 0) {
        int32_t *m = rec + 8 * wv;
        m[0] = mqe_h, m[1] = mqe_t, m[2] = mte_h, m[3] = mte_q, m[4] = score, m[5] = late;
        last = __hip_atomic_fetch_add(ctl + kBandCtlTicket, 1, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT) == W - 1;
    }
    if (lane == 0 && last) {
        mqe_h = KSW_NEG_INF_I, mqe_t = -1, mte_h = KSW_NEG_INF_I, mte_q = -1, score = KSW_NEG_INF_I;
        for (int k = 0; k < W; ++k) {
            const int32_t *m = rec + 8 * k;
            if (m[0] > mqe_h || (m[0] == mqe_h && m[1] > mqe_t)) mqe_h = m[0], mqe_t = m[1];
            if (m[3] >= 0 && (mte_q < 0 || m[2] > mte_h)) mte_h = m[2], mte_q = m[3];
            score = max(score, m[4]);
            late |= m[5];
        }
        KswOut o;
        o.score = score, o.mqe = mqe_h, o.mqe_t = mqe_t, o.mte = mte_h, o.mte_q = mte_q;
        o.max = 0, o.max_t = -1, o.max_q = -1;
        o.zdropped = r_end < nr ? 1 : 0, o.stopped = 0, o.reach_end = 0, o.n_cigar = 0;
        a.out[jb.out] = o;
        a.redo[job] = late | a.force_redo;
    }
}

// Clears the control blocks and buffers of a launch's jobs (blockIdx.y).
__global__ void __launch_bounds__(256) ksw_band_ctl_kernel(int32_t *bnd, const GenJob *jobs, const int32_t *order)
{
    const GenJob &jb = jobs[order[blockIdx.y]];
    int32_t *ctl = bnd + jb.bnd_off;
    // (64 bits: 536 million letters of both are 2^31 dwords)
    const int64_t n = kBandCtl + 4 * ((int64_t)jb.qlen + jb.tlen);
    for (int64_t k = blockIdx.x * blockDim.x + threadIdx.x; k < n; k += gridDim.x * blockDim.x) ctl[k] = 0;
}

namespace {

// Workgroups of one band-kernel variant that the device holds at once.
int band_capacity(const void *fn, int threads, int lds)
{
    int dev = 0, cus = 0, per_cu = 0;
    if (hipGetDevice(&dev) != hipSuccess) return 0;
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) return 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, fn, threads, lds) != hipSuccess) return 0;
    return cus * per_cu;
}

}  // namespace

hipError_t launch_band(const BandArgs &a0, int team, bool right, bool score_only, hipStream_t st)
{
    if (a0.njobs <= 0) return hipSuccess;
    if (team < 1 || team > kBandTeam) return hipErrorInvalidValue;
    BandArgs a = a0;
    const int wpg = team < kBandGroup ? team : kBandGroup;
    a.wgs = (team + wpg - 1) / wpg;
    const int threads = kWave * wpg, lds = ring_bytes(wpg);
    void (*fn)(BandArgs) = score_only ? ksw_band_kernel<false, true>
                           : right    ? ksw_band_kernel<true, false>
                                      : ksw_band_kernel<false, false>;
    // half the device's capacity per launch: the workgroups of a pair wait on
    // one another, so all of them must be resident together, beside the
    // kernels of other streams (which finish on their own) and one other
    // waiting launch of at most half the device (the caller's admission).
    // One workgroup per pair waits for no other: all pairs in one launch
    int chunk = a0.njobs;
    if (a.wgs > 1) {
        const int cap = band_capacity((const void *)fn, threads, lds);
        if (cap < 2 * a.wgs) return hipErrorInvalidConfiguration;
        chunk = cap / 2 / a.wgs;
    }
    chunk = std::min(chunk, 65535);
    for (int off = 0; off < a0.njobs; off += chunk) {
        a.order = a0.order + off;
        a.njobs = a0.njobs - off < chunk ? a0.njobs - off : chunk;
        hipLaunchKernelGGL(ksw_band_ctl_kernel, dim3(std::max(1, std::min(64, 1024 / a.njobs)), a.njobs), dim3(256), 0, st,
                           a.bnd, a.jobs, a.order);
        hipLaunchKernelGGL(fn, dim3(a.njobs * a.wgs), dim3(threads), lds, st, a);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

}  // namespace kswhip
