// bf16 MFMA forward kernels (head_dim 64 / 128 / 256; at 256 the one-sweep kernel only: two K / V tile pairs are 128 KB of LDS).
// Replace the reference's `_forward_one_row` sweep (sb_varlen/sb_varlen_fwd.py:81-215):
// one workgroup per (sequence, head, 128-query row-block), keys swept right-to-left from
// the diagonal in steps of 64, K/V tiles double-buffered in LDS, running product of
// (1 - beta) per query in a register.  Layout and arithmetic: sba_mfma.h.
#include "sba_mfma.h"

namespace sba {
inline namespace SBA_ELEM_NS {

// One sweep step of one wave: 32 queries x 64 keys.  Scores (from the pre-scaled Q fragments),
// mask on the diagonal, weights, O^T += V^T P^T.  kFast: the one-reciprocal chain; it may refuse
// the step (returns false, nothing changed), see forward_weights_fast().  lane_carry: the product of
// (1 - beta) over all keys right of this LANE's 32 keys (the right half-wave's is the carry that entered
// the step), which is what the carry tables keep.
template <int D, bool kCarryOnly, bool kFast, bool kPinBase>
__device__ inline bool fwd_step(const char* ktile, const char* vtile, const LaneOffsets<D>& lo,
                                const h16x8 (&qf)[D / 16], f32x16 (&oacc)[D / 32], float& R, int lane,
                                int key0, int q0w, int qi, int strict, float& lane_carry) {
    const int h = lane >> 5;
    float x[32];
    score_tiles_ps<D>(x, ktile, lo, qf);
    if (key0 + 63 + strict > q0w) mask_step(x, key0 + 32 * h, qi, strict);     // diagonal region
    h16x8 pf[4];
    if (kFast) {
        if (!forward_weights_fast<!kCarryOnly>(x, pf, R, lane, lane_carry)) return false;
    } else {
        float dummy[1];
        stick_weights<false>(x, dummy, R, lane, &lane_carry);
        if (!kCarryOnly) {
#pragma unroll
            for (int c = 0; c < 4; ++c) pf[c] = pack8(&x[8 * c]);
        }
    }
    if (!kCarryOnly) {
#pragma unroll
        for (int c2 = 0; c2 < 2; ++c2) {   // operands of two key groups requested together, ahead of their MFMAs
            h16x8 vt[2][D / 32];
#pragma unroll
            for (int cc = 0; cc < 2; ++cc)
#pragma unroll
                for (int db = 0; db < D / 32; ++db) vt[cc][db] = fetch_cols_o<D, kPinBase>(vtile, lo, db, 2 * c2 + cc);
            if (kWide<D>) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int cc = 0; cc < 2; ++cc)
#pragma unroll
                for (int db = 0; db < D / 32; ++db) oacc[db] = mfma(vt[cc][db], pf[2 * c2 + cc], oacc[db]);
        }
    }
    return true;
}

template <int D>
__device__ inline void store_o_rows(char* stage, const KParams& p, const Job& job, int head, int q0w, int lane, const f32x16 (&oacc)[D / 32]) {
    store_query_rows<D>(stage, oacc, 1.0f, p.o, slice_offset(p.o, job.seq, head, job.tok0),
                        q0w, job.len, lane, p.cols);
}

// kCarryOnly: write the carry table and nothing else (no P*V, no o / rem): the backward's way of
// getting the table when the forward kept none.
// Params, wave_, lane_: launches that draw their jobs hand them in anew for each job (see draw_jobs()).  The others take the parameters by value and their own thread
// index: then the compiler makes of it what it makes of a kernel's body (head_dim 256 by reference and from outside: 721 -> 725 us at H=16 T=10008, 46.8 -> 47.4 at B=4 H=8 T=1024).
template <int D, bool kCarryOnly, Sharing kSharing, class Params, class Draw>
__device__ __forceinline__ void fwd_job(Params p, const int block, const int wave_, const int lane_, Draw draw) {
    const int lane = kSharing == kDrawn ? lane_ : (int)(threadIdx.x & 63);
    const int wave = kSharing == kDrawn ? wave_ : __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    constexpr int kTile = 64 * kPitch<D> * 2;            // bytes per K or V tile
    __shared__ __attribute__((aligned(16))) char lds[4 * kTile + (kCarryOnly ? 0 : 32)];   // K0 V0 K1 V1 | words
    int (*const done_waves)[4] = (int (*)[4])(lds + (kCarryOnly ? kTile : 4 * kTile));     // [parity of the step][wave]

    const int n = lane & 31, h = lane >> 5;
    LaneOffsets<D> lo;
    lo.init(lane);
    const int head = head_of_block<kSharing>(p, block);
    const Job job = decode_job<D == 64>(p, order_job(slot_of_block(p, block), p.n_jobs, false));
    const int strict = p.attend_current ? 0 : 1;
    const int m0 = job.rb * kRowBlock;
    const int q0w = m0 + 32 * wave;              // first query of this wave
    const int qi = q0w + n;                      // this lane's query
    const bool rows_full = q0w + 31 < job.len;   // wave-uniform
    const int64_t qbase = slice_offset(p.q, job.seq, head, job.tok0);
    const int64_t kbase = slice_offset(p.k, job.seq, head, job.tok0);
    const int64_t vbase = slice_offset(p.v, job.seq, head, job.tok0);

    h16x8 qf[D / 16];
    load_row_frags<D>(qf, p.q, qbase, q0w, n, job.len, lane, p.cols);
    prescale_frags(qf, p.scale2);

    f32x16 oacc[D / 32];
#pragma unroll
    for (int db = 0; db < D / 32; ++db) oacc[db] = f32x16{0};
    float R = qi < job.len ? 1.0f : 0.0f;
    // This wave has no more weights to give: its rows' carries are exactly 0, or it has no rows at all.
    bool done = q0w >= job.len;
    const int thread = kSharing == kDrawn ? 64 * wave + lane : (int)threadIdx.x;
    if (thread < 8) done_waves[thread >> 2][thread & 3] = 0;

    const int imax = min(m0 + kRowBlock - 1, job.len - 1);
    const int kmax = imax - strict;                       // last key any row of the block sees
    const int n_steps = kmax >= 0 ? kmax / kKeyBlock + 1 : 0;
    const int64_t tabq = tab_index(p, head, job, job.rb, 0) + 32 * wave + n;   // + step * kRowBlock

    TileDma<D> kc, vc;
    kc.init(lane, wave, p.k, kbase, p.cols);
    vc.init(lane, wave, p.v, vbase, p.cols);
#pragma unroll
    for (int b = 0; b < 2; ++b) {
        kc.clear(lds + b * 2 * kTile);
        vc.clear(lds + b * 2 * kTile + kTile);
    }
    if (n_steps > 0) {
        kc.issue((n_steps - 1) * kKeyBlock, job.len, lds);
        if (!kCarryOnly) vc.issue((n_steps - 1) * kKeyBlock, job.len, lds + kTile);
    }
    wait_global_memory();
    __syncthreads();

    // Carry tables: the right half-wave's carries go to `rtab`, the left one's to `rmid` (one store of the whole
    // wave).  A step's carries are only known after its chain (the left half's contain the right half's
    // product) and are stored at the top of the NEXT step, in front of its tile loads: vector-memory
    // operations retire in order, so the wait for those loads at the end of that step also covers the store,
    // long after it has completed, and no wait ever falls on a fresh store.
    float* const my_tab = h ? p.rtab : p.rmid;
    const bool both_tables = D == 256 || p.rmid;          // (without rmid the backward makes it)
    float carry_out = 1.0f;
    int carry_step = -1;                       // wave-uniform: the step whose carries wait to be stored
    auto store_carries = [&]() {
        if (carry_step >= 0 && p.save) {
            if (rows_full && both_tables) my_tab[tabq + carry_step * kRowBlock] = carry_out;      // no lane mask
            else if (qi < job.len && (both_tables || h)) my_tab[tabq + carry_step * kRowBlock] = carry_out;
        }
        carry_step = -1;
    };
    // what a step does before its arithmetic
    auto open_step = [&](int step, int buf) {
        store_carries();
        if (step > 0) {   // next tiles, straight into the other buffer (free since the last barrier);
                          // every tile left of the sweep's first lies inside the sequence
            kc.issue_full((step - 1) * kKeyBlock, lds + (buf ^ 1) * 2 * kTile);
            if (!kCarryOnly) vc.issue_full((step - 1) * kKeyBlock, lds + (buf ^ 1) * 2 * kTile + kTile);
        }
    };
    // The sweep runs with the one-reciprocal chain until a step refuses it (logits too large for
    // it); from that step on this wave continues with the reciprocal-per-key chain.  Every wave
    // executes one barrier per step whichever loop it is in.
    // A wave that is done only copies its share of the tiles and enters zero carries; the sweep ends after the step in which the
    // last of the four is done (live_index() says why).  A wave with work left pays one comparison per step for this: only a
    // wave that is done looks at what the others have said.  Their words are kept by parity of the step, so that none can
    // be about a later one; they are never taken back.
    const float nothing = p.early_end ? 0.f : -1.f;
    // (the number of iterations is a variable of the loops' only exit: with a break of its own the accumulators would meet copies
    // of themselves behind the loops, 32 registers more)
    int it = 0, iterations = n_steps;
    auto close_step = [&](int step, int buf) {
        wait_global_memory();                  // the next tiles have landed
        if (__builtin_amdgcn_ballot_w64(R != nothing) != 0) {
            __syncthreads();
            return;
        }
        done = true;
        if (q0w < job.len && carry_step < 0) { carry_out = 0.f; carry_step = step; }
        if (lane == 0) done_waves[buf][wave] = 1;
        __syncthreads();
        if (__builtin_amdgcn_readfirstlane(done_waves[buf][0] & done_waves[buf][1] & done_waves[buf][2] & done_waves[buf][3])) iterations = it + 1;
    };
    int buf = 0;
    bool redo = false;
    for (; it < iterations; ++it, buf ^= 1) {
        const int step = n_steps - 1 - it;
        const char* ktile = lds + buf * 2 * kTile;
        const int key0 = step * kKeyBlock;
        // whole step right of this wave's last query, or all of this wave's queries past the end of the sequence
        const bool skip = key0 + strict > q0w + 31 || done;
        open_step(step, buf);
        if (!skip) {
            if (!fwd_step<D, kCarryOnly, true, kWide<D>>(ktile, ktile + kTile, lo, qf, oacc, R, lane, key0, q0w, qi, strict, carry_out)) {
                redo = true;
                break;
            }
            carry_step = step;
        }
        close_step(step, buf);
    }
    for (; it < iterations; ++it, buf ^= 1) {
        const int step = n_steps - 1 - it;
        const char* ktile = lds + buf * 2 * kTile;
        const int key0 = step * kKeyBlock;
        const bool skip = key0 + strict > q0w + 31 || done;
        if (!redo) open_step(step, buf);
        redo = false;
        if (!skip) {
            fwd_step<D, kCarryOnly, false, kWide<D>>(ktile, ktile + kTile, lo, qf, oacc, R, lane, key0, q0w, qi, strict, carry_out);
            carry_step = step;
        }
        close_step(step, buf);
    }
    draw();
    store_carries();
    if (p.save && thread == 0) set_first_live(p, head, job, n_steps - iterations);

    if (!kCarryOnly) {
        store_o_rows<D>(lds + wave * kRowStage<D>, p, job, head, q0w, lane, oacc);       // (the tiles are free)
        if (h == 0 && qi < job.len)
            Elem16::store(p.rem.ptr, (int64_t)job.seq * p.rem.sb + (int64_t)head * p.rem.sh + job.tok0 + qi, R);
    }
}

template <int D, bool kCarryOnly>
__global__ __launch_bounds__(kThreads) void mfma_fwd_kernel(KParams p) {
    fwd_job<D, kCarryOnly, kSharedCu, KParams>(p, blockIdx.x, 0, 0, [] {});
}

template <int D, bool kCarryOnly>
__global__ __launch_bounds__(kThreads, 2) void mfma_fwd_drawing_kernel(KParams) {
    __shared__ int words[2];
    draw_jobs(words, [&](const KParams& p, int block, int wave, int lane, auto draw) { fwd_job<D, kCarryOnly, kDrawn, const KParams&>(p, block, wave, lane, draw); });
}

// ---------------------------------------------------------------- small grids: G segments per sweep
// A launch of a few hundred workgroups cannot fill the SIMDs with one-sweep-per-workgroup work,
// and lasts as long as its longest sweep.  Here a workgroup has G groups of four waves, and the
// sweep of its 128 queries is cut into G CONTIGUOUS segments of keys, one per group (group 0 the
// rightmost, with the diagonal).  Every group runs the ordinary sweep over its segment from a
// carry of 1 - nothing couples the segments but one number per query, the product of (1 - beta)
// over a whole segment - and at the end
//     O = sum_g F_g O_g,   F_g = product of the totals of the segments right of g,
// is formed through LDS, the carry-table entries that a group wrote relative to its own right
// edge are multiplied by F_g, and rem is the product of all totals.  No exchange inside the
// sweep; the groups only share the workgroup barrier that hands over the tiles.
template <int D, int G, bool kCarryOnly>
__global__ __launch_bounds__(G * kThreads) void mfma_fwd_seg_kernel(KParams p) {
    constexpr int kTile = 64 * kPitch<D> * 2;
    // tile(grp, buf, kv) = lds + ((grp * 2 + buf) * 2 + kv) * kTile
    __shared__ __attribute__((aligned(16))) char lds[G * 4 * kTile];
    __shared__ float totals[G][kRowBlock];
    __shared__ int done_waves[2][4 * G];
    __shared__ int first_live;

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int grp = wave >> 2, qs = wave & 3;
    const int n = lane & 31, h = lane >> 5;
    LaneOffsets<D> lo;
    lo.init(lane);
    const int head = head_of_block<G == 2 && D == 64 ? kSharedCu : kOnePerCu>(p, blockIdx.x);
    const Job job = decode_job<D == 64 && G == 2>(p, order_job(slot_of_block(p, blockIdx.x), p.n_jobs, false));
    const int strict = p.attend_current ? 0 : 1;
    const int m0 = job.rb * kRowBlock;
    const int q0w = m0 + 32 * qs;
    const int qi = q0w + n;
    const bool rows_full = q0w + 31 < job.len;      // wave-uniform
    const int64_t qbase = slice_offset(p.q, job.seq, head, job.tok0);
    const int64_t kbase = slice_offset(p.k, job.seq, head, job.tok0);
    const int64_t vbase = slice_offset(p.v, job.seq, head, job.tok0);

    h16x8 qf[D / 16];
    load_row_frags<D>(qf, p.q, qbase, q0w, n, job.len, lane, p.cols);
    prescale_frags(qf, p.scale2);
    f32x16 oacc[D / 32];
#pragma unroll
    for (int db = 0; db < D / 32; ++db) oacc[db] = f32x16{0};
    float R = qi < job.len ? 1.0f : 0.0f;

    const int imax = min(m0 + kRowBlock - 1, job.len - 1);
    const int kmax = imax - strict;
    const int n_steps = kmax >= 0 ? kmax / kKeyBlock + 1 : 0;
    const int chunk = (n_steps + G - 1) / G;              // iterations of every group
    const int hi = n_steps - grp * chunk;                  // this group sweeps steps hi-1 .. low
    const int low = max(hi - chunk, 0);
    const int64_t tabq = tab_index(p, head, job, job.rb, 0) + 32 * qs + n;   // + step * kRowBlock
    char* my_tiles = lds + grp * 4 * kTile;                // + buf * 2 * kTile

    TileDma<D> kc, vc;
    kc.init(lane, qs, p.k, kbase, p.cols);
    vc.init(lane, qs, p.v, vbase, p.cols);
#pragma unroll
    for (int b = 0; b < 2; ++b) {
        kc.clear(my_tiles + b * 2 * kTile);
        vc.clear(my_tiles + b * 2 * kTile + kTile);
    }
    if (hi - 1 >= low) {
        kc.issue((hi - 1) * kKeyBlock, job.len, my_tiles);
        if (!kCarryOnly) vc.issue((hi - 1) * kKeyBlock, job.len, my_tiles + kTile);
    }
    // A segment ends early as the sweep of mfma_fwd_kernel does, once its own product is exactly 0 for all rows; the workgroup's
    // loop ends when every wave is done or at the end of its segment.
    bool done = q0w >= job.len, group_done = false;
    int reached = low;                                     // leftmost step for which this wave had weights to give
    const float nothing = p.early_end ? 0.f : -1.f;
    if (threadIdx.x < 8 * G) done_waves[threadIdx.x / (4 * G)][threadIdx.x % (4 * G)] = 0;
    if (threadIdx.x == 0) first_live = n_steps;
    wait_global_memory();
    __syncthreads();

    // carry tables as in mfma_fwd_kernel (right half-wave -> rtab, left -> rmid, stored a step late), here
    // relative to the segment's right edge
    float* const my_tab = h ? p.rtab : p.rmid;
    const bool both_tables = D == 256 || p.rmid;          // (without rmid the backward makes it)
    float carry_out = 1.0f;
    int carry_step = -1;
    auto store_carries = [&]() {
        if (carry_step >= 0 && p.save) {
            if (rows_full && both_tables) my_tab[tabq + carry_step * kRowBlock] = carry_out;
            else if (qi < job.len && (both_tables || h)) my_tab[tabq + carry_step * kRowBlock] = carry_out;
        }
        carry_step = -1;
    };
    auto open_step = [&](int step, int buf) {
        store_carries();
        if (step - 1 >= low && !group_done) {
            kc.issue_full((step - 1) * kKeyBlock, my_tiles + (buf ^ 1) * 2 * kTile);
            if (!kCarryOnly) vc.issue_full((step - 1) * kKeyBlock, my_tiles + (buf ^ 1) * 2 * kTile + kTile);
        }
    };
    int it = 0, iterations = chunk;
    auto close_step = [&](int step, int buf) {
        wait_global_memory();
        if (__builtin_amdgcn_ballot_w64(R != nothing) != 0 && step > low) {
            __syncthreads();
            return;
        }
        // nothing more to come from this wave: at the end of its segment, or done
        if (__builtin_amdgcn_ballot_w64(R != nothing) == 0) {
            if (!done) reached = max(step, low);
            done = true;
            if (step >= low && q0w < job.len && !group_done && carry_step < 0) { carry_out = 0.f; carry_step = step; }
        }
        if (lane == 0) done_waves[buf][wave] = done ? 1 : 2;
        __syncthreads();
        // one lane per wave's word
        const int said = done_waves[buf][lane % (4 * G)];
        const uint64_t group = UINT64_C(0xf) << (4 * grp);
        if ((__builtin_amdgcn_ballot_w64(said == 1) & group) == group) group_done = true;
        if (__builtin_amdgcn_ballot_w64(said == 0) == 0) iterations = it + 1;
    };
    int buf = 0;
    bool redo = false;
    for (; it < iterations; ++it, buf ^= 1) {
        const int step = hi - 1 - it;
        const char* ktile = my_tiles + buf * 2 * kTile;
        const int key0 = step * kKeyBlock;
        const bool skip = step < low || key0 + strict > q0w + 31 || done;
        open_step(step, buf);
        if (!skip) {
            if (!fwd_step<D, kCarryOnly, true, true>(ktile, ktile + kTile, lo, qf, oacc, R, lane, key0, q0w, qi, strict, carry_out)) {
                redo = true;
                break;
            }
            carry_step = step;
        }
        close_step(step, buf);
    }
    for (; it < iterations; ++it, buf ^= 1) {       // reciprocal-per-key chain from the refused step on
        const int step = hi - 1 - it;
        const char* ktile = my_tiles + buf * 2 * kTile;
        const int key0 = step * kKeyBlock;
        const bool skip = step < low || key0 + strict > q0w + 31 || done;
        if (!redo) open_step(step, buf);
        redo = false;
        if (!skip) {
            fwd_step<D, kCarryOnly, false, true>(ktile, ktile + kTile, lo, qf, oacc, R, lane, key0, q0w, qi, strict, carry_out);
            carry_step = step;
        }
        close_step(step, buf);
    }
    store_carries();
    wait_global_memory();                      // the group's last entries are in memory before they are rescaled below

    // ---- segment totals -> F (what this group's results are relative to) and rem
    if (h == 0) totals[grp][32 * qs + n] = R;
    __syncthreads();
    float F = 1.0f, all = 1.0f;
#pragma unroll
    for (int g = 0; g < G; ++g) {
        const float t = totals[g][32 * qs + n];
        if (g < grp) F *= t;
        all *= t;
    }
    // (rows for which nothing is left of the stick to the right of this segment have all their live entries there)
    if (__builtin_amdgcn_ballot_w64(F != 0.f && qi < job.len) != 0 && lane == 0) atomicMin(&first_live, reached);
    // carry-table entries of this group, written relative to its own right edge: times F.  Every lane
    // rescales the entries it wrote (the half-waves have a table each); the loads go out in batches so that
    // their latencies overlap.  Its stores have completed (wait above).
    if (p.save && grp > 0 && qi < job.len && (both_tables || h)) {
        for (int s0 = reached; s0 < hi; s0 += 8) {
            float v[8];
#pragma unroll
            for (int j = 0; j < 8; ++j)
                if (s0 + j < hi) v[j] = my_tab[tabq + (s0 + j) * kRowBlock];
#pragma unroll
            for (int j = 0; j < 8; ++j)
                if (s0 + j < hi) my_tab[tabq + (s0 + j) * kRowBlock] = v[j] * F;
        }
    }
    if (kCarryOnly) {
        __syncthreads();
        if (p.save && threadIdx.x == 0) set_first_live(p, head, job, p.early_end ? first_live : 0);
        return;
    }

    // ---- O = sum_g F_g O_g: groups 1.. park their scaled accumulators in LDS (the tiles are free
    // since the last barrier of the sweep), group 0 adds them up
    float* park = (float*)lds;                              // [grp - 1][qs][db][r][lane]
    if (grp > 0) {
#pragma unroll
        for (int db = 0; db < D / 32; ++db)
#pragma unroll
            for (int r = 0; r < 16; ++r)
                park[((((grp - 1) * 4 + qs) * (D / 32) + db) * 16 + r) * 64 + lane] = oacc[db][r] * F;
    }
    __syncthreads();
    if (p.save && threadIdx.x == 0) set_first_live(p, head, job, p.early_end ? first_live : 0);
    if (grp == 0) {
#pragma unroll
        for (int g = 1; g < G; ++g)
#pragma unroll
            for (int db = 0; db < D / 32; ++db)
#pragma unroll
                for (int r = 0; r < 16; ++r)
                    oacc[db][r] += park[((((g - 1) * 4 + qs) * (D / 32) + db) * 16 + r) * 64 + lane];
        static_assert(kRowStage<D> <= (D / 32) * 16 * 64 * 4, "a wave's own accumulators were parked there");
        store_o_rows<D>((char*)(park + qs * (D / 32) * 16 * 64), p, job, head, q0w, lane, oacc);
        if (h == 0 && qi < job.len)
            Elem16::store(p.rem.ptr, (int64_t)job.seq * p.rem.sb + (int64_t)head * p.rem.sh + job.tok0 + qi, all);
    }
}

}  // inline namespace SBA_ELEM_NS
}  // namespace sba

// Key segments per sweep for the forward: 4 or 2 (head_dim 128: 2), or 0 = one sweep per workgroup.
//
// What decides is how long the launch's longest sweep is against the work of an average workgroup slot, the tail
// ratio r of sba_tail_ratio().  Two segments halve the longest sweep at 8 waves per workgroup (two workgroups per CU),
// four quarter it at 16 waves (one workgroup per CU: worth it only while the grid is at most two rounds of them).
// Measured on MI355X, forward time in us, one sweep / two segments / four segments:
//     B=1 H=16 T=3584 (r 4.4)   64.8 / 55.8 / 51.1      B=2 H=16 T=2304 (r 3.4)   47.7 / 42.6 / 52.4
//     B=1 H=16 T=4096 (r 3.9)   74.5 / 63.9 / 60.4      B=4 H=16 T=1024 (r 3.6, 512 workgroups)  26.2 / 26.1 / 29.7
//     B=1 H=16 T=4224 (r 3.8)   76.5 / 66.9 / 69.6      B=8 H=16 T=512  (r 3.2, 512 workgroups)  18.5 / 18.8 / 24.9
//     B=1 H=16 T=5120 (r 3.1)   95.7 / 82.8 / 93.3      B=1 H=32 T=4096 (r 1.9)   96.8 / 96.6 / 112.8
//     B=1 H=16 T=6144 (r 2.6)  115.8 / 110.0 / 120.0    B=2 H=16 T=4096 (r 1.9)   98.4 / 97.3 / 112.7
//     B=1 H=16 T=8192 (r 2.0)  179.8 / 170.9 / 181.9    B=5 H=16 T=2048 (r 1.5)   65.4 / 70.8 / -
//     B=1 H=16 T=10240 (r 1.6) 253.7 / 248.6 / -        B=3 H=16 T=4096 (r 1.3)  127.6 / 132.5 / -
//     packs of log-normal documents, H=16 (tokens, longest document, r): one sweep / two segments
//         8192, 2802, r 3.2   57.7 / 51.2 (four: 69.8)     8192, 4096, r 2.8   81.5 / 72.3     4096, 1393, r 4.7   31.0 / 28.0
//         6000, 1162, r 3.3   30.5 / 31.5                  10000, 2243, r 2.4  51.1 / 56.0     12288, 2069, r 1.9  56.4 / 64.7
// Two segments pay from r = 1.7 on for dense batches but lose 10-16 % on packs (one long document among many short
// ones) up to r = 2.4: the rule takes them from 2.7 on.
// SBA_FWD_GROUPS=2|3|4 forces the number of segments where the rule picks any; SBA_TWO_STEP_MAX_GRID=n replaces
// the rule by "segments (4, or as forced) up to n workgroups".
static int forward_segments(const sba::KParams& kp, unsigned grid) {
    if (kp.head_dim == 256) return 0;      // two K / V tile pairs are 128 KB of LDS: one group of waves per workgroup
    if (kp.head_dim == 128 || kp.head_dim == 96) {
        // head_dim 128: the one-sweep kernel holds two workgroups per CU, the two-segment one (8 waves, 129 KB of
        // LDS) one; it pays while the grid is at most two rounds of those and the longest sweep dominates.  B=1,
        // H=16, one sweep / two segments in us: T=1024 29.8 / 26.2, T=2048 50.4 / 41.6, T=3072 77.2 / 60.0, T=4096
        // 105.5 / 91.8, T=5120 131.1 / 138.7, T=8192 276.2 / 291.7; B=2 T=2048 60.0 / 57.0; H=8 T=4096 89.7 / 70.8.
        // Long dense sequences somewhat beyond.  Two segments over one sweep, mean logits 0 .. -6 over the heads in this order and in two random
        // ones / all at -6:  T=4400 (r 3.6) 0.83-0.86 / 0.86, T=4800 (3.3) 0.87-0.92 / 0.90, T=5000 (3.1) 0.88-0.94 / 0.915, H=12 T=6500 (3.3)
        // 0.79-0.82 / 0.90, H=10 T=8000 (3.2) 0.82-0.97 / 0.885, H=8 T=10000 (3.2) 0.92-1.00 / 0.89, B=2 H=8 T=4800 (3.3) 0.98 / 0.92; beyond that
        // H=8 T=11000 (2.9) 0.90-1.09 / 0.93;  with fewer heads H=4 T=20000 (3.2) 0.97-0.98 / 0.88;  shorter ones H=32 T=2500 (3.1) 1.02-1.08 / 1.02.
        // At head_dim 80, whose steps are shorter, the same rule is about even: T=4400 0.91-0.93 / 0.97, T=4800 0.94-0.99 / 1.05, T=5000 0.97-1.01 / 1.07,
        // H=12 T=6500 0.85-0.87 / 1.01, H=10 T=8000 0.90-1.06 / 1.03, H=8 T=10000 0.96-1.06 / 1.00, B=2 H=8 T=4800 1.08 / 1.03.
        if (sba_two_step_env() >= 0) return grid <= (unsigned)sba_two_step_env() ? 2 : 0;
        const double r = sba_tail_ratio(kp, grid);
        if (!kp.cu_seqlens && kp.n_heads >= 8 && kp.seq_len > 32 * sba::kRowBlock && r >= 3.1) return 2;
        return grid <= 2u * (unsigned)sba_cu_count() && r >= 3.7 ? 2 : 0;
    }
    const char* e = getenv("SBA_FWD_GROUPS");
    const int forced = e ? atoi(e) : 0;
    const bool force = forced == 2 || forced == 3 || forced == 4;
    if (sba_two_step_env() >= 0) return grid <= (unsigned)sba_two_step_env() ? (force ? forced : 4) : 0;
    const double r = sba_tail_ratio(kp, grid);
    const int segments = (r >= 3.8 && grid <= 2u * (unsigned)sba_cu_count()) ? 4 : (r >= 2.7 ? 2 : 0);
    return segments && force ? forced : segments;
}

template <bool kCarryOnly>
static void launch_seg(int groups, dim3 grid, hipStream_t s, const sba::KParams& kp) {
    using namespace sba;
    if (kp.head_dim == 96) hipLaunchKernelGGL((mfma_fwd_seg_kernel<96, 2, kCarryOnly>), grid, dim3(2 * kThreads), 0, s, kp);
    else if (kp.head_dim == 128) hipLaunchKernelGGL((mfma_fwd_seg_kernel<128, 2, kCarryOnly>), grid, dim3(2 * kThreads), 0, s, kp);
    else if (groups == 2) hipLaunchKernelGGL((mfma_fwd_seg_kernel<64, 2, kCarryOnly>), grid, dim3(2 * kThreads), 0, s, sba_turning(kp, 2));
    else if (groups == 3) hipLaunchKernelGGL((mfma_fwd_seg_kernel<64, 3, kCarryOnly>), grid, dim3(3 * kThreads), 0, s, kp);
    else hipLaunchKernelGGL((mfma_fwd_seg_kernel<64, 4, kCarryOnly>), grid, dim3(4 * kThreads), 0, s, kp);
}

#ifdef SBA_ELEM_F16
int sba_launch_mfma_f16_fwd(const sba::KParams& kp_in, hipStream_t s) {
#else
int sba_launch_mfma_fwd(const sba::KParams& kp_in, hipStream_t s) {
#endif
    using namespace sba;
    dim3 grid((unsigned)kp_in.n_jobs * kp_in.n_heads);
    const int segments = forward_segments(kp_in, grid.x);
    KParams kp = kp_in;
    kp.queue_stride = sba_queue_stride(kp);
    float* const table = kp.save ? kp.rtab : nullptr;
    if (segments) {
        if (kp.carry_only) launch_seg<true>(segments, grid, s, kp);
        else launch_seg<false>(segments, grid, s, kp);
    } else if (kp.head_dim == 64) {
        if (kp.carry_only) hipLaunchKernelGGL((mfma_fwd_kernel<64, true>), grid, dim3(kThreads), 0, s, sba_turning(kp, 4));
        else hipLaunchKernelGGL((mfma_fwd_kernel<64, false>), grid, dim3(kThreads), 0, s, sba_turning(kp, 4));
    } else if (kp.head_dim == 96) {
        if (kp.carry_only) sba_launch_drawing((mfma_fwd_kernel<96, true>), (mfma_fwd_drawing_kernel<96, true>), grid.x, kThreads, 2, kp, table, kForwardQueue, false, s);
        else sba_launch_drawing((mfma_fwd_kernel<96, false>), (mfma_fwd_drawing_kernel<96, false>), grid.x, kThreads, 2, kp, table, kForwardQueue, false, s);
    } else if (kp.head_dim == 128) {
        if (kp.carry_only) sba_launch_drawing((mfma_fwd_kernel<128, true>), (mfma_fwd_drawing_kernel<128, true>), grid.x, kThreads, 2, kp, table, kForwardQueue, false, s);
        else sba_launch_drawing((mfma_fwd_kernel<128, false>), (mfma_fwd_drawing_kernel<128, false>), grid.x, kThreads, 2, kp, table, kForwardQueue, false, s);
    } else {
        if (kp.carry_only) hipLaunchKernelGGL((mfma_fwd_kernel<256, true>), grid, dim3(kThreads), 0, s, kp);
        else hipLaunchKernelGGL((mfma_fwd_kernel<256, false>), grid, dim3(kThreads), 0, s, kp);
    }
    return hipGetLastError() == hipSuccess ? SBA_OK : SBA_ERR_LAUNCH;
}
