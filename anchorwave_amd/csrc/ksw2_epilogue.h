// ksw2_epilogue.h -- what follows a pair's passes: the H bookkeeping's last
// folds, the start cell, the walk and the result, for the kernels whose
// passes store direction bytes or Singletrack tracks by rows of lanes.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>
#include "ksw2_cell.h"
#include "ksw2_common.h"
#include "ksw2_kernels.h"
#include "ksw2_walk.h"

namespace kswhip {

// Singletrack tracks of one stripe-kernel pair (layout of the tracks mode),
// read in the reference's coordinates (i target, j query).  A transposed
// pair stores cell (i, j) at (j, i) and its horizontal and vertical
// differences exchanged.
template <int R>
struct StripeTracks {
    static constexpr int SR = kWave * R;
    const uint8_t *dir;
    const uint8_t *qs, *ts;   // the reference's query and target
    uint64_t nsteps;
    int32_t mch, mis;
    bool tr;
    __device__ int32_t get(int track, int i, int j) const
    {
        if (tr) {
            const int t = i;
            i = j, j = t, track = 1 - track;
        }
        const int s = i / SR, pp = s >> 1, h = s & 1, k = (i % SR) / R, rho = i % R;
        const uint64_t c = (uint64_t)(j + k + kWave * h);
        const uint8_t b =
            dir[((pp * nsteps + c) * kWave + k) * (4 * R) + track * (2 * R) + 4 * (rho >> 1) + 2 * h + (rho & 1)];
        return -(int32_t)(int8_t)b;
    }
    __device__ int forced(int, int) const { return 0; }
    __device__ int32_t cost(int i, int j) const { return ts[i] == qs[j] ? mch : mis; }
};

// The state of a walk: the cell (i, j) in the reference's coordinates, the
// state machine's state, the open CIGAR run and the words written so far (by
// the threads with `writer` set).  Uniform over a wave.
struct PathWalk {
    int i, j, state, run_op, run_len, n;
    uint32_t *cig;
    bool writer;
    __device__ __forceinline__ void push(int op, int len)
    {
        if (op == run_op) {
            run_len += len;
            return;
        }
        if (run_len > 0) {
            if (writer) cig[n] = (uint32_t)run_len << 4 | (uint32_t)run_op;
            ++n;
        }
        run_op = op, run_len = len;
    }
};

// Walks until the path leaves the staged tile or the matrix.  From state 0
// the walk stays in state 0 and moves diagonally while each cell's argmax (its
// low three bits) is 0; state s (1-4) stays while each cell's continuation bit
// (s + 2) is set, moving i (s = 1, 3) or j (s = 2, 4) back by one, which is one
// stored row or one column.  So lane k tests the k-th cell of such a run, a
// ballot finds the first that ends it, and that cell's byte (already in its
// lane) gives the step after the run: one LDS read per run and turn.
template <class L>
__device__ __forceinline__ void walk_tile(const L &lay, PathWalk &w, bool tr)
{
    const int lk = threadIdx.x & (kWave - 1);
    while (w.i >= 0 && w.j >= 0) {
        const int r = tr ? w.j : w.i, c = tr ? w.i : w.j;  // stored coordinates of cell (i, j)
        if (!lay.has(r, c)) return;
        const int s = w.state;
        const bool di = s == 0 || s == 1 || s == 3, dj = s == 0 || s == 2 || s == 4;
        const bool dr = tr ? dj : di, dc = tr ? di : dj;
        // the last step of a run that is inside the tile and the matrix
        const int lim = min(min(dr ? r - lay.r_lo : kWave, dc ? c - lay.c_lo : kWave),
                            min(di ? w.i : kWave, dj ? w.j : kWave));
        int byte = 0, end = 1;
        if (lk <= lim) {
            byte = lay.at(dr ? r - lk : r, dc ? c - lk : c);
            end = s == 0 ? (byte & 7) != 0 : !(byte >> (s + 2) & 1);
        }
        const uint64_t eb = __ballot(end);
        const int run = eb ? (int)__builtin_ctzll(eb) : kWave;
        if (run > 0) {
            w.push(s == 0 ? 0 : di ? 2 : 1, run);
            if (di) w.i -= run;
            if (dj) w.j -= run;
        }
        if (run > min(lim, kWave - 1)) continue;
        w.state = __builtin_amdgcn_readlane(byte, run) & 7;
        if (w.state == 0) w.push(0, 1), --w.i, --w.j;
        else if (w.state == 1 || w.state == 3) w.push(2, 1), --w.i;
        else w.push(1, 1), --w.j;
    }
}

// The stripe kernel's stored layout (dir_index() and track_index() of
// ksw2_common.h) as the epilogue reads it.  The walk's tile is 8 lanes x 64
// columns (up to 64 rows x 64 columns of one stripe).
template <int R, int MODE>
struct StripeLayout {
    static constexpr int SR = kWave * R;  // rows per stripe
    static constexpr int mode = MODE;
    typedef StripeTracks<R> Tracks;
    uint64_t (*tile)[64];
    const uint8_t *dir;
    uint64_t nsteps;
    int r_lo, r_hi, c_lo, c_hi;  // the staged cells: striped rows, swept columns

    __device__ StripeLayout(uint64_t (*t)[64]) : tile(t) {}
    __device__ void open(const StripeArgs &a, const KswJob &jb)
    {
        dir = a.dir + jb.dir_off;
        nsteps = pass_steps(jb.qlen);
        r_lo = 1, r_hi = 0, c_lo = 1, c_hi = 0;
    }
    // the passes have left the result so far (score, mte) in a.out
    __device__ KswOut result(const StripeArgs &a, int job, const KswJob &, int) const { return a.out[job]; }
    // the largest H of the last swept column, negated and scaled, and its row
    // (ties to the later row): the stripes' partials in row order
    __device__ void last_column(const StripeArgs &a, const KswJob &jb, int, int &best, int &best_i) const
    {
        const int nstripes = stripe_count(jb.tlen, R);
        int carry = 0;
        for (int s = 0; s < nstripes; ++s) {
            const StripeRec rec = a.recs[jb.stripe_off + s];
            if (rec.best_i >= 0 && carry + rec.best <= best) best = carry + rec.best, best_i = rec.best_i;
            carry += rec.total;
        }
    }
    __device__ bool has(int r, int c) const { return r >= r_lo && r <= r_hi && c >= c_lo && c <= c_hi; }
    // the byte of a staged cell
    __device__ int at(int r, int c) const
    {
        const int rel = r - r_lo;
        return (int)(tile[rel / R][c - c_lo] >> (8 * (rel % R))) & 0xff;
    }
    // stages lanes kb..k of stripe s (rows up to r) x columns c-63..c
    __device__ void stage(int r, int c, int tid, int nthr)
    {
        const int s = r / SR, k = (r - s * SR) / R, kb = k >= 7 ? k - 7 : 0;
        const int pp = s >> 1, h = s & 1;
        r_lo = s * SR + kb * R, r_hi = s * SR + k * R + R - 1;
        c_hi = c, c_lo = c >= 63 ? c - 63 : 0;
        const int s_lo = c_lo + kb + kWave * h, s_hi = c_hi + k + kWave * h;
        __syncthreads();  // the previous tile is no longer read
        for (int cc = s_lo + tid; cc <= s_hi; cc += nthr) {
            const uint8_t *src = dir + (((uint64_t)pp * nsteps + (uint64_t)cc) * kWave + kb) * (2 * R);
            for (int kr = 0; kr <= k - kb; ++kr) {
                const int jj = cc - kWave * h - (kb + kr);
                if (jj >= c_lo && jj <= c_hi) {
                    // the R row bytes of half h: bytes 2h, 2h+1 of each dword
                    const unsigned sel = h ? 0x07060302u : 0x05040100u;
                    if (R == 8) {
                        const uint4 w = ((const uint4 *)src)[kr];
                        const uint32_t lo = __builtin_amdgcn_perm(w.y, w.x, sel);
                        const uint32_t hi = __builtin_amdgcn_perm(w.w, w.z, sel);
                        tile[kr][jj - c_lo] = (uint64_t)hi << 32 | lo;
                    } else {
                        const uint2 w = ((const uint2 *)src)[kr];
                        tile[kr][jj - c_lo] = __builtin_amdgcn_perm(w.y, w.x, sel);
                    }
                }
            }
        }
        __syncthreads();
    }
    // every thread walks, staging a tile when the path leaves the last
    __device__ void walk(PathWalk &w, bool tr, int tid, int nthr)
    {
        while (w.i >= 0 && w.j >= 0) {
            const int r = tr ? w.j : w.i, c = tr ? w.i : w.j;
            if (!has(r, c)) stage(r, c, tid, nthr);
            walk_tile(*this, w, tr);
        }
    }
    __device__ Tracks tracks(const StripeArgs &a, const KswJob &jb) const
    {
        const bool tr = jb.transposed != 0;
        Tracks A;
        A.dir = dir;
        A.qs = a.seq + (tr ? jb.t_off : jb.q_off), A.ts = a.seq + (tr ? jb.q_off : jb.t_off);
        A.nsteps = nsteps;
        A.mch = a.sc.mch, A.mis = a.sc.mis;
        A.tr = tr;
        return A;
    }
};

// Epilogue of one pair, run by the whole workgroup once every pass is done:
// folds the per-stripe mqe partials in row order (ties to the later row, the
// '>=' of minimap2/ksw2_extd2_sse.c:371), picks the start cell as in
// minimap2/ksw2_extd2_sse.c:398-418 and walks the direction bytes with the
// state machine of ksw_backtrack (minimap2/ksw2.h:160-192) for an unbanded
// matrix (no cell of the path can leave the band there, so the off/off_end
// forcing never triggers).  The walk reads a tile of the layout L staged in
// LDS by the workgroup; when the path leaves the tile the next one is staged,
// so HBM latency is paid once per tile rather than once per step.  Every thread runs the same walk
// (uniform control flow, LDS broadcast reads) while other workgroups keep the
// SIMDs busy; thread 0 writes the run-length encoded CIGAR, which is reversed
// at the end unless KSW_EZ_REV_CIGAR.  With a host mirror, the result and the
// CIGAR are then copied to pinned host memory and the pair's completion flag
// is raised (system-scope release), so a caller can take this pair's result
// while the launch still runs.
//
// With the two Singletrack tracks instead of direction bytes, the first wave
// runs the Singletrack walk (track_walk) for a global alignment; with
// KSW_EZ_EXTZ_ONLY or KSW_EZ_SEMIGLOBAL_END the result is zdropped with no
// path (minimap2/ksw2_extd2_avx.c:752-760), and a failed walk reports
// n_cigar = -1 (no CIGAR, zdropped).
template <class L>
__device__ __forceinline__ void pair_epilogue(const StripeArgs &a, int job_id, const KswJob &jb, L &lay,
                                              int *shared_n, int nthr)
{
    constexpr bool tracks = L::mode == kTracks;
    const int tid = threadIdx.x;
    // the host's stop flag, read once for the whole workgroup: a stopped
    // pair's passes may have ended early, so it takes no walk
    int stopped = 0;
    if (a.stop) {
        if (tid == 0) *shared_n = __hip_atomic_load(a.stop, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        __syncthreads();
        stopped = *shared_n;
        __syncthreads();
    }
    lay.open(a, jb);
    KswOut o = lay.result(a, job_id, jb, nthr);
    if (stopped) o.stopped = 1;
    const int flag = jb.flag;
    // kq, kt: the swept and striped lengths; qlen, tlen: the reference's
    const bool tr = __builtin_amdgcn_readfirstlane(jb.transposed) != 0;
    const int kq = jb.qlen, kt = jb.tlen;
    const int qlen = tr ? kt : kq, tlen = tr ? kq : kt;
    {
        int best = 0x7fffffff, best_i = -1;
        lay.last_column(a, jb, nthr, best, best_i);
        const int64_t h_anchor = (int64_t)a.sc.G1 - a.sc.qe_orig;
        const int h_top_last_col = (int)(h_anchor + edge_prefix(a.sc, kq - 1));  // H(-1, kq-1)
        const int col_max = h_top_last_col - (best >> CellOf<false, L::mode>::shift);
        if (!tr) {
            o.mqe = col_max, o.mqe_t = best_i;
        } else {
            // the last swept column is the reference's last row (mte) and the
            // last striped row, tracked by the last pass, its last column (mqe)
            o.mqe = o.mte, o.mqe_t = o.mte_q;
            o.mte = col_max, o.mte_q = best_i;
        }
    }
    int i0 = -1, j0 = -1;
    int n = 0;
    uint32_t *cig = a.cig + jb.cig_off;
    if (stopped) {
        // no walk: the passes, the stripe partials and this pair's result
        // slot may be incomplete
    } else if (tracks) {
        if (!o.stopped && !o.zdropped && !(flag & (0x40 | 0x800))) {
            if (tid < kWave) {
                const typename L::Tracks A = lay.tracks(a, jb);
                const WalkGaps g = {-a.sc.q, -a.sc.e, -a.sc.q2, -a.sc.e2};
                const int nn = track_walk(A, qlen, tlen, g, cig);
                if (tid == 0) *shared_n = nn;
            }
            __syncthreads();
            n = *shared_n;
            if (n < 0) o.zdropped = 1;
        } else if (!o.stopped && !o.zdropped) {
            o.zdropped = 1;
        }
    } else if (!(flag & 0x01)) {  // KSW_EZ_SCORE_ONLY: no path
        if (!o.stopped && !o.zdropped && (flag & 0x800)) {          // SEMIGLOBAL_END
            if (o.mqe > o.mte) o.score = o.mqe, i0 = o.mqe_t, j0 = qlen - 1;
            else o.score = o.mte, i0 = tlen - 1, j0 = o.mte_q;
        } else if (!o.stopped && !o.zdropped && !(flag & 0x40)) {   // global
            i0 = tlen - 1, j0 = qlen - 1;
        } else if (!o.zdropped && (flag & 0x40) && o.mqe + jb.end_bonus > o.max) {  // EXTZ_ONLY
            o.reach_end = 1, i0 = o.mqe_t, j0 = qlen - 1;
        } else if (o.max_t >= 0 && o.max_q >= 0) {
            i0 = o.max_t, j0 = o.max_q;
        }
    }
    if (i0 >= 0 || j0 >= 0) {
        PathWalk w;
        w.i = __builtin_amdgcn_readfirstlane(i0), w.j = __builtin_amdgcn_readfirstlane(j0);
        w.state = 0, w.run_op = -1, w.run_len = 0, w.n = 0;
        w.cig = cig, w.writer = tid == 0;
        lay.walk(w, tr, tid, nthr);
        if (w.i >= 0) w.push(2, w.i + 1);
        if (w.j >= 0) w.push(1, w.j + 1);
        w.push(-2, 0);  // flush the last run
        n = w.n;
        __syncthreads();
        if (!(flag & 0x80))
            for (int x = tid; x < (n >> 1); x += nthr) {
                const uint32_t t = cig[x];
                cig[x] = cig[n - 1 - x];
                cig[n - 1 - x] = t;
            }
    }
    o.n_cigar = n;
    if (tid == 0) a.out[job_id] = o;
    if (a.host_flag) {
        __syncthreads();
        uint32_t *hc = a.host_cig + jb.cig_off;
        if (n < 0) n = 0;
        for (int x = tid; x < n; x += nthr) hc[x] = cig[x];
        if (tid == 0) a.host_out[job_id] = o;
        __threadfence_system();
        __syncthreads();
        if (tid == 0) __hip_atomic_store(a.host_flag + job_id, 1, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
    }
}

}  // namespace kswhip
