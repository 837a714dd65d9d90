// bf16 MFMA backward kernels (head_dim 64 / 128 / 256): two passes, no atomics, deterministic.
//
// The reference (`_backward_one_row`, sb_varlen/sb_varlen_bwd.py:274-456) owns a query
// row-block, keeps dq in registers and adds every dk/dv tile into global memory under a
// spin lock (`locked_add`, :13-52).  Here the two reductions are separated instead:
//
//   pass 1  (row owner, like the forward): recomputes the weights of each 64-key step from
//           the forward's carry table, forms dz, accumulates dQ in registers, and records
//           for every (query, key block) the prefix  sum_{j left of the block} g_ij  in a
//           second table.  g_ij = a_ij * (dO_i . v_j) here: the gradient of rem enters as the
//           constant d_rem_i * rem_i that every prefix of row i starts from, which is all it
//           contributes to dz (sum_j a_ij + rem_i = 1), so pass 2 never reads d_rem.
//   pass 2  (key owner): the owner of a block of keys sweeps the query blocks at or below the
//           diagonal, recomputes weights and dz of its tiles from the tables, transposes them
//           through LDS and accumulates dK = dZ^T Q and dV = P^T dO in registers.  Four
//           kernels, chosen by grid size and head_dim: every wave owning 32 keys outright
//           (d = 64, large grids), two waves sharing 32 keys (d = 128, large grids), a resident
//           producer/consumer stream over 64-key items (d = 64, small grids), one workgroup
//           per 64-key block (d = 128, small grids).  d = 256: every wave on its own 32 keys, two
//           workgroups per key block that each take half of the columns of dK and dV.
//
// Every element of the score matrix is therefore evaluated twice in the backward (once per
// pass); in exchange nothing is reduced through memory.
#include <string.h>
#include <atomic>
#include <type_traits>
#include "sba_mfma.h"

namespace sba {
inline namespace SBA_ELEM_NS {

// The dQ pass leaves its pre-scaled Q fragments (q times scale * log2 e, rounded to bf16: the operand every
// row-owner kernel multiplies with) behind for the key-owner stream and the paired kernel in its place, which then need no scaling of their
// own and see bit for bit the logits that the forward's carries were made from.  Row qi of q_scaled gets this
// lane's four 16-byte chunks (columns 16 ks + 8 h ..).  head_dim 64 only, and only where the launcher asks for it.
template <int D>
__device__ inline void store_scaled_q(const KParams& p, const Job& job, int head, int qi, int lane,
                                      const h16x8 (&qf)[D / 16]) {
    if (D != 64 || !p.q_scaled.ptr || qi >= job.len) return;
    char* row = p.q_scaled.ptr + 2 * ((int64_t)job.seq * p.q_scaled.sb + (int64_t)head * p.q_scaled.sh +
                                      (int64_t)(job.tok0 + qi) * p.q_scaled.st + 8 * (lane >> 5));
#pragma unroll
    for (int ks = 0; ks < D / 16; ++ks) *(u32x4*)(row + 32 * ks) = __builtin_bit_cast(u32x4, qf[ks]);
}

// ---------------------------------------------------------------- pass 1: dQ + prefix table
// kLean (head_dim 64): the register-lean arrangement of the step that head_dim 128 always uses, held to three waves
// per SIMD.  Ahead on large launches, whose SIMDs it fills better (the packed benchmark's dQ -5.6 %, short documents
// -6 %); on launches that last as long as their longest sweep the plain arrangement's shorter step is ahead.
// kMid: the forward kept `rtab` alone (KParams::makes_mid).  The left half-wave starts its chain from 1, the right half-wave's product
// completes it, and is the entry of `rmid`: 32 multiplications a step.
template <int D, bool kLean, bool kMid, Sharing kSharing, class Draw>
__device__ __forceinline__ void dq_job(const KParams& p, const int block, const int wave, const int lane, Draw draw) {
    static_assert(!kMid || kWide<D> || kLean, "the arrangement that takes the carry into g alone");
    constexpr int kTile = 64 * kPitch<D> * 2;
    __shared__ __attribute__((aligned(16))) char lds[4 * kTile];   // K0 V0 K1 V1

    const int n = lane & 31, h = lane >> 5;
    LaneOffsets<D> lo;
    lo.init(lane);
    lo.rebase(lds);                        // absolute addresses: the loop below runs in one copy per tile buffer
    const int head = head_of_block<kSharing>(p, block);
    const Job job = decode_job<D == 64>(p, order_job(slot_of_block(p, block), p.n_jobs, false));
    const int strict = p.attend_current ? 0 : 1;
    const int m0 = job.rb * kRowBlock;
    const int q0w = m0 + 32 * wave;
    const int qi = q0w + n;
    const bool row_ok = qi < job.len;
    const int64_t qbase = slice_offset(p.q, job.seq, head, job.tok0);
    const int64_t kbase = slice_offset(p.k, job.seq, head, job.tok0);
    const int64_t vbase = slice_offset(p.v, job.seq, head, job.tok0);
    const int64_t dobase = slice_offset(p.d_o, job.seq, head, job.tok0);

    if (block == 0 && wave == 0) clear_words(p, lane);     // error word of the launch pair, see wait_for_count(), and the second one's queues
    h16x8 qf[D / 16], dof[D / 16];
    load_row_frags<D>(qf, p.q, qbase, q0w, n, job.len, lane, p.cols);
    prescale_frags(qf, p.scale2);          // the score MFMAs then deliver base-2 logits
    load_row_frags<D>(dof, p.d_o, dobase, q0w, n, job.len, lane, p.cols);

    f32x16 dqacc[D / 32];
#pragma unroll
    for (int db = 0; db < D / 32; ++db) dqacc[db] = f32x16{0};
    float Gc = 0.f;

    const int imax = min(m0 + kRowBlock - 1, job.len - 1);
    const int kmax = imax - strict;
    const int n_steps = kmax >= 0 ? kmax / kKeyBlock + 1 : 0;
    const int first = first_live_block(p, head, job);      // the sweep's first step, see live_index()

    TileDma<D, false, D == 64 && kLean> kc, vc;
    kc.init(lane, wave, p.k, kbase, p.cols);
    vc.init(lane, wave, p.v, vbase, p.cols);
#pragma unroll
    for (int b = 0; b < 2; ++b) {
        kc.clear(lds + b * 2 * kTile);
        vc.clear(lds + b * 2 * kTile + kTile);
    }
    if (n_steps > 0) {
        kc.seek(first * kKeyBlock);
        kc.issue_here(first * kKeyBlock, job.len, lds);
        vc.seek(first * kKeyBlock);
        vc.issue_here(first * kKeyBlock, job.len, lds + kTile);
    }
    if (wave == 3) close_live_ranges(p, head, job, lane, first);

    // carry-table traffic is kept off the critical path: the value of the NEXT step is loaded
    // while this one is computed, and this step's prefix is stored before the tile loads are
    // issued (vector memory operations retire in order)
    // Per lane ONE cursor into the tables: the entry of (this query, the step at hand) in the table of the forward
    // that holds the carry entering this LANE's 32 keys (right half-wave: rtab, left: rmid).  The prefix entering
    // the same 32 keys goes to the same entry of gmid / gtab, which lies the same distance from the cursor for
    // both half-waves (gmid - rtab == gtab - rmid: the library lays the tables out that way).
    constexpr int64_t tstride = kRowBlock;
    const float* rcur = (h ? p.rtab : p.rmid) + tab_index(p, head, job, job.rb, first) + 32 * wave + n;
    // (kMid: rtab is the caller's, so that the distances differ)
    const int64_t g_from_r = kMid && h ? (const char*)p.gmid - (const char*)p.rtab : (const char*)p.gtab - (const char*)p.rmid;
    // kMid at head_dim 64: a table's entry is a scalar base and the lane's row.  Cursor and distance are three registers more, which its step does not
    // have: the distance came back from scratch in every step, and a reload waits for all memory (the kernel alone at H=16, T=16384: 775 us, 721 this
    // way; forward and backward at B=4 H=16 T=8192 2155, 2138).  At head_dim 128, where there is room, the two extra stores cost 0.5 %.
    constexpr bool kByBase = kMid && kLean;
    int64_t column = tab_index(p, head, job, job.rb, first);
    const uint32_t table_row = 32 * wave + n;
    auto entry_of = [&](float* table, int64_t at) __attribute__((always_inline)) -> float& {
        table += at;
        asm("" : "+s"(table));                // (a scalar base: its sum with the row would be two registers)
        return table[table_row];
    };
    float Rnext = 1.0f;
    if (row_ok && n_steps > 0) {
        if (kByBase && h) Rnext = entry_of(p.rtab, column);
        if (!kByBase && (!kMid || h)) Rnext = *rcur;
    }
    float Gstore = 0.f, Mstore = 0.f;
    bool g_pending = false;
    auto store_prefixes = [&]() __attribute__((always_inline)) {
        if (!g_pending || !row_ok) return;
        if (!kByBase) {
            *(float*)((char*)(rcur - tstride) + g_from_r) = Gstore;
            if (kMid && !h) *const_cast<float*>(rcur - tstride) = Mstore;
        } else if (h) {
            entry_of(p.gmid, column - tstride) = Gstore;
        } else {
            entry_of(p.gtab, column - tstride) = Gstore;
            entry_of(p.rmid, column - tstride) = Mstore;
        }
    };
    // (last of the prologue's loads: its conversion waits for it, and with it for everything requested before)
    float dr = 0.f;
    if (row_ok && p.d_rem.ptr)
        dr = Elem16::load(p.d_rem.ptr, (int64_t)job.seq * p.d_rem.sb + (int64_t)head * p.d_rem.sh + job.tok0 + qi);
    if (first > 0) Gc = dr * 0.f;              // nothing left of the stick there: 0, and NaN where dr is no number, as in a full sweep
    wait_global_memory();
    __syncthreads();
    // (behind the prologue's loads: a store in front of them would keep the compiler from issuing them together,
    // and the wait above would fall on it; here it retires under the first step)
    store_scaled_q<D>(p, job, head, qi, lane, qf);
    auto do_step = [&](int step, auto buf_c) __attribute__((always_inline)) {
        constexpr int buf = decltype(buf_c)::value;
        constexpr TileAt ktile = {buf * 2 * kTile};
        constexpr TileAt vtile = {buf * 2 * kTile + kTile};
        const bool more = step + 1 < n_steps;
        const int key0 = step * kKeyBlock;
        const bool skip = key0 + strict > q0w + 31 || q0w >= job.len;     // nothing visible, or no query of this wave inside the sequence
        // the prefixes that entered the previous step (the first block's are only known once that
        // block's weights are: they start at d_rem * rem, see below)
        store_prefixes();
        g_pending = false;
        const float F = Rnext;
        if (more) {
            if (row_ok && kByBase && h) Rnext = entry_of(p.rtab, column + tstride);
            if (row_ok && !kByBase && (!kMid || h)) Rnext = rcur[tstride];
            // next tiles, straight into the other buffer (free since the last barrier)
            kc.forth();
            kc.issue_here((step + 1) * kKeyBlock, job.len, lds + (buf ^ 1) * 2 * kTile);
            vc.forth();
            vc.issue_here((step + 1) * kKeyBlock, job.len, lds + (buf ^ 1) * 2 * kTile + kTile);
        }
        if (!skip) {
            h16x8 zf[4];
            if constexpr (kWide<D> || kLean) {
                // Register-lean arrangement (two arrays of 32 live instead of four: two waves per SIMD
                // instead of one): scores and dP first, then the chain over both in place.
                float x[32], dp[32];
                score_tiles_ps<D>(x, ktile, lo, qf);
                dp_tiles_o<D>(dp, vtile, lo, dof);
                if (key0 + 63 + strict > q0w) mask_step(x, key0 + 32 * h, qi, strict);
                float gsum;
                float Lend = carried_beta_g(x, dp, F, gsum);
                if constexpr (kMid) {
                    float Llo, Lup;
                    half_values(Lend, Llo, Lup);
                    float carry = h ? 1.0f : Lup;
                    __builtin_amdgcn_sched_barrier(0);
                    asm("" : "+v"(carry));
                    scale_all(dp, carry);
                    __builtin_amdgcn_sched_barrier(0);
                    gsum *= carry;
                    Lend *= carry;
                    Mstore = Lup;
                }
                if (step == 0) {                         // the gradient of rem rides in the prefix, see below (further right: no remainder)
                    float Llo, Lup;
                    half_values(Lend, Llo, Lup);
                    Gc = dr * Llo;                       // what leaves the left half of the leftmost block is rem
                }
                float clo, cup;
                half_values(gsum, clo, cup);
                const float Glane = h ? Gc + clo : Gc;   // the prefix entering this lane's 32 keys: block edge (left half-wave) or middle
                Gc = Gc + clo + cup;
                Gstore = Glane;
                g_pending = true;
                walk_logit_grads_g(x, dp, Glane, zf);
            } else {
                float x[32], beta[32], dp[32];
                float Glane;
                score_tiles_ps<D>(x, ktile, lo, qf);
                if (key0 + 63 + strict > q0w) {
    mask_step(x, key0 + 32 * h, qi, strict);
                }
                // dP does not depend on the weights: its MFMAs go between the segments of the chain,
                // where the chain's exp/rcp overlap them
                const float Lend = carried_weights_and_dp<D>(x, beta, dp, F, vtile, lo, dof);
                // The gradient of rem rides in the prefix: g is formed from the plain dP, and the term
                // -beta_ik * d_rem_i * rem_i that d_rem adds to dz_ik is a constant d_rem_i * rem_i in
                // the running prefix.  What leaves the left half of the leftmost block is the product over
                // all keys, rem_i.
                if (step == 0) {
                    float Llo, Lup;
                    half_values(Lend, Llo, Lup);
                    Gc = dr * Llo;
                }
                logit_grads<false>(x, beta, dp, Gc, lane, &Glane);
                // the prefix entering this lane's 32 keys - the block's edge for the left half-wave, its middle
                // (for the key-owner pass whose waves own 32 keys) for the right one -, stored at the top of the
                // next iteration
                Gstore = Glane;
                g_pending = true;
#pragma unroll
                for (int c = 0; c < 4; ++c) zf[c] = pack8(&dp[8 * c]);
            }
#pragma unroll
            for (int c = 0; c < 4; ++c) {      // (operands of a key group requested together, see score_raw_o)
                h16x8 kt[D / 32];
#pragma unroll
                for (int db = 0; db < D / 32; ++db) kt[db] = fetch_cols_o<D>(ktile, lo, db, c);
                if (kWide<D>) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int db = 0; db < D / 32; ++db) dqacc[db] = mfma(kt[db], zf[c], dqacc[db]);
            }
        }
        if (kByBase) column += tstride;
        else rcur += tstride;
        wait_global_memory();                  // the next tiles have landed
        __syncthreads();
    };
    for (int step = first; step < n_steps; step += 2) {
        do_step(step, std::integral_constant<int, 0>{});
        if (step + 1 < n_steps) do_step(step + 1, std::integral_constant<int, 1>{});
    }
    store_prefixes();
    draw();

    store_query_rows<D>(lds + wave * kRowStage<D>, dqacc, p.scale, p.dq,                 // (the tiles are free)
                        slice_offset(p.dq, job.seq, head, job.tok0), q0w, job.len, lane, p.cols);
}

template <int D, bool kLean = false, bool kMid = false>
__global__ __launch_bounds__(kThreads, (D == 64 && kLean) ? 3 : (D <= 128 ? 2 : 1)) void mfma_bwd_dq_kernel(KParams p) {
    dq_job<D, kLean, kMid, D <= 128 ? kSharedCu : kOnePerCu>(p, blockIdx.x, __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), threadIdx.x & 63, [] {});
}

template <int D, bool kLean, bool kMid>
__global__ __launch_bounds__(kThreads, kLean ? 3 : 2) void mfma_bwd_dq_drawing_kernel(KParams) {
    __shared__ int words[2];
    draw_jobs(words, [&](const KParams& p, int block, int wave, int lane, auto draw) { dq_job<D, kLean, kMid, kDrawn>(p, block, wave, lane, draw); });
}

// ---------------------------------------------------------------- pass 1, two steps per iteration
// Same sweep with 8 waves: wave-group 0 (waves 0-3) and wave-group 1 (waves 4-7) take two
// CONSECUTIVE 64-key steps of the same 128 queries in every iteration (group 1 the right one).
// All the heavy work of a step (scores, weights, dP, g = a*dP and its prefix sums inside the
// step) only needs the step's own keys and the forward's carry table; what couples neighbouring
// steps is one number per query, the sum of g over the step.  The groups swap those totals
// through LDS at a barrier, the right group adds the left group's total to its prefix, and each
// group accumulates its own partial dQ, summed once at the end.  The longest dependent chain
// of a launch (the sweep of the last row-block) is halved, which is what bounds the time when
// the whole problem is only two waves per SIMD.
template <int D>
__global__ __launch_bounds__(2 * kThreads, 2) void mfma_bwd_dq2_kernel(KParams p) {
    constexpr int kTile = 64 * D * 2;
    // tile(buf, grp, kv) = lds + ((buf * 2 + grp) * 2 + kv) * kTile
    __shared__ __attribute__((aligned(16))) char lds[8 * kTile];
    __shared__ float xch[2][kRowBlock];

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int grp = wave >> 2, qs = wave & 3;
    const int n = lane & 31, h = lane >> 5;
    LaneOffsets<D> lo;
    lo.init(lane);
    const int head = head_of_block(p, blockIdx.x);
    const Job job = decode_job(p, order_job(slot_of_block(p, blockIdx.x), p.n_jobs, false));
    const int strict = p.attend_current ? 0 : 1;
    const int m0 = job.rb * kRowBlock;
    const int q0w = m0 + 32 * qs;
    const int qi = q0w + n;
    const bool row_ok = qi < job.len;
    const int64_t qbase = slice_offset(p.q, job.seq, head, job.tok0);
    const int64_t kbase = slice_offset(p.k, job.seq, head, job.tok0);
    const int64_t vbase = slice_offset(p.v, job.seq, head, job.tok0);
    const int64_t dobase = slice_offset(p.d_o, job.seq, head, job.tok0);

    if (blockIdx.x == 0 && wave == 0) clear_words(p, lane);     // as in mfma_bwd_dq_kernel
    h16x8 qf[D / 16], dof[D / 16];
    load_row_frags<D>(qf, p.q, qbase, q0w, n, job.len, lane);
    prescale_frags(qf, p.scale2);          // the score MFMAs then deliver base-2 logits
    load_row_frags<D>(dof, p.d_o, dobase, q0w, n, job.len, lane);

    f32x16 dqacc[D / 32];
#pragma unroll
    for (int db = 0; db < D / 32; ++db) dqacc[db] = f32x16{0};
    float Gc = 0.f;

    const int imax = min(m0 + kRowBlock - 1, job.len - 1);
    const int kmax = imax - strict;
    const int n_steps = kmax >= 0 ? kmax / kKeyBlock + 1 : 0;
    // the sweep's first step (see live_index()), from the even step on: pairs of steps stay the same pairs wherever a sweep begins
    const int live = first_live_block(p, head, job), first = live & ~1;
    const int n_it = (n_steps - first + 1) / 2;
    char* my_tiles = lds + grp * 2 * kTile;          // + buf * 4 * kTile

    // each group copies its own tiles (256 threads per tile pair)
    TileDma<D> kc, vc;
    kc.init(lane, qs, p.k, kbase);
    vc.init(lane, qs, p.v, vbase);
    if (first + grp < n_steps) {
        kc.issue((first + grp) * kKeyBlock, job.len, my_tiles);
        vc.issue((first + grp) * kKeyBlock, job.len, my_tiles + kTile);
    }
    if (wave == 7) close_live_ranges(p, head, job, lane, live);

    // the forward's carry for this group's NEXT step is loaded while this one is computed
    constexpr int64_t tstride = kRowBlock;
    // this lane's cursor into the carry tables and the distance to its prefix entry, see the one-step kernel
    const float* rcur = (h ? p.rtab : p.rmid) + tab_index(p, head, job, job.rb, first) + 32 * qs + n + grp * tstride;
    const int64_t g_from_r = (const char*)p.gtab - (const char*)p.rmid;
    float Rnext = (row_ok && first + grp < n_steps) ? *rcur : 1.0f;
    if (first + grp < live) Rnext = 0.f;             // (no entry)
    float Gstore = 0.f;
    bool g_pending = false;
    // (last of the prologue's loads: its conversion waits for it, and with it for everything requested before)
    float dr = 0.f;
    if (row_ok && p.d_rem.ptr)
        dr = Elem16::load(p.d_rem.ptr, (int64_t)job.seq * p.d_rem.sb + (int64_t)head * p.d_rem.sh + job.tok0 + qi);
    if (first > 0) Gc = dr * 0.f;              // (see the one-step kernel)
    wait_global_memory();
    __syncthreads();
    if (grp == 0) store_scaled_q<D>(p, job, head, qi, lane, qf);      // (placed as in the one-step kernel)
    // Every LDS address of the loop is a sweep-constant register plus an immediate: the lane offsets are made absolute
    // for this group's tiles once, and the loop runs in one copy per tile buffer (see the one-step kernel).
    lo.rebase(my_tiles);
    auto do_iteration = [&](int it, auto buf_c) __attribute__((always_inline)) {
        constexpr int buf = decltype(buf_c)::value;
        constexpr TileAt ktile = {buf * 4 * kTile};
        constexpr TileAt vtile = {buf * 4 * kTile + kTile};
        const int step = first + 2 * it + grp;           // == n_steps: this group idles in the last iteration
        const bool more = step + 2 < n_steps;
        const int key0 = step * kKeyBlock;
        const bool active = step < n_steps && !(key0 + strict > q0w + 31) && q0w < job.len;
        if (g_pending && row_ok) *(float*)((char*)(rcur - 2 * tstride) + g_from_r) = Gstore;
        g_pending = false;
        const float F = Rnext;
        if (more) {
            if (row_ok) Rnext = rcur[2 * tstride];
            // next tiles, straight into the other buffer (free since the last barrier)
            kc.issue((step + 2) * kKeyBlock, job.len, my_tiles + (buf ^ 1) * 4 * kTile);
            vc.issue((step + 2) * kKeyBlock, job.len, my_tiles + (buf ^ 1) * 4 * kTile + kTile);
        }
        // (an active wave's whole step sits in one branch, exchange barrier included: were the step split around the
        // barrier, its 64 weights and gradients would have to hold a value on the idle path too, and the compiler
        // clears half of them at the top of every step)
        if (active) {
            float x[32], beta[32], dp[32];
            float total = 0.f;
            score_tiles_ps<D, true>(x, ktile, lo, qf);
            if (key0 + 63 + strict > q0w) mask_step(x, key0 + 32 * h, qi, strict);
            const float Lend = carried_weights_and_dp<D, true>(x, beta, dp, F, vtile, lo, dof);
            float start = logit_grads_local(x, dp, total, lane);
            // the gradient of rem rides in the prefix as the constant d_rem * rem (see the one-step
            // kernel).  The leftmost block is group 0's first step: the constant joins its total
            // (which carries it to the other group and into Gc) and its own prefix
            if (step == 0) {
                float Llo, Lup;
                half_values(Lend, Llo, Lup);
                const float c0 = dr * Llo;
                total += c0;
                start += c0;
            }
            if (h == 0) xch[grp][32 * qs + n] = total;
            __syncthreads();
            const float other = xch[grp ^ 1][32 * qs + n];
            // group 1 holds the right step of the pair: its prefix also contains group 0's total
            const float Gmy = grp == 0 ? Gc : Gc + other;
            Gc = Gc + total + other;
            const float Glane = Gmy + start;       // the prefix entering this lane's 32 keys: block edge or middle (see the one-step kernel)
            Gstore = Glane;
            g_pending = true;
            logit_grads_apply(beta, dp, Glane);
            h16x8 zf[4];
#pragma unroll
            for (int c = 0; c < 4; ++c) zf[c] = pack8(&dp[8 * c]);
#pragma unroll
            for (int db = 0; db < D / 32; ++db)
#pragma unroll
                for (int c = 0; c < 4; ++c)
                    dqacc[db] = mfma(fetch_cols_o<D>(ktile, lo, db, c), zf[c], dqacc[db]);
        } else {
            if (h == 0) xch[grp][32 * qs + n] = 0.f;
            __syncthreads();
            Gc = Gc + xch[grp ^ 1][32 * qs + n];
        }
        rcur += 2 * tstride;
        wait_global_memory();                  // the next tiles have landed
        __syncthreads();
    };
    for (int it = 0; it < n_it; it += 2) {
        do_iteration(it, std::integral_constant<int, 0>{});
        if (it + 1 < n_it) do_iteration(it + 1, std::integral_constant<int, 1>{});
    }

    if (g_pending && row_ok) *(float*)((char*)(rcur - 2 * tstride) + g_from_r) = Gstore;

    // ---- dQ = dQ(group 0) + dQ(group 1): group 1 parks its accumulators in LDS
    float* park = (float*)lds;                              // [qs][db][r][lane]
    if (grp == 1) {
#pragma unroll
        for (int db = 0; db < D / 32; ++db)
#pragma unroll
            for (int r = 0; r < 16; ++r) park[((qs * (D / 32) + db) * 16 + r) * 64 + lane] = dqacc[db][r];
    }
    __syncthreads();
    if (grp == 0) {
#pragma unroll
        for (int db = 0; db < D / 32; ++db)
#pragma unroll
            for (int r = 0; r < 16; ++r) dqacc[db][r] += park[((qs * (D / 32) + db) * 16 + r) * 64 + lane];
        store_query_rows<D>((char*)(park + qs * (D / 32) * 16 * 64), dqacc, p.scale, p.dq,      // (over what this wave has just read)
                            slice_offset(p.dq, job.seq, head, job.tok0), q0w, job.len, lane, D);
    }
}

// ---------------------------------------------------------------- pass 2: dK, dV
// One workgroup per 64-key block; a step covers 128 queries (32 per wave).  Each wave
// turns its 32 queries into weights (a, dz), writes them as bf16 [query][key] rows into a
// tile shared by the workgroup, and after a barrier reduces ONE [32 keys x 32 d] tile of
// dK and of dV over all 128 queries, so its accumulators are 2 x 16 x D/64 registers and
// two workgroups fit on a CU.  Every Q / dO row is fetched from global memory once, as the
// per-lane row fragments that the score / dP MFMAs need (Q a step ahead, dO at the top of
// the step, hidden behind the weights); the same registers are then stored into the shared
// Q and dO tiles that the reduction reads transposed.  Per-query scalars (carry tables,
// drem) are prefetched one step ahead.
template <int D>
__global__ __launch_bounds__(kThreads, 2) void mfma_bwd_dkv_kernel(KParams p) {
    constexpr int kTile = 64 * D * 2;          // K or V tile (64 keys)
    constexpr int kQTile = 128 * D * 2;        // Q or dO tile (128 queries)
    constexpr int kZTile = 128 * 64 * 2;       // weights of one step, [query][key] bf16
    // the tiles read with the transposing fetch come first so that their offsets fit the
    // 16-bit immediate of the LDS instructions
    __shared__ __attribute__((aligned(1024))) char lds[2 * kTile + 2 * kQTile + 2 * kZTile];
    char* zp = lds;
    char* zd = zp + kZTile;
    char* qtile = zd + kZTile;
    char* dotile = qtile + kQTile;
    char* ktile = dotile + kQTile;
    char* vtile = ktile + kTile;

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int n = lane & 31, h = lane >> 5;
    LaneOffsets<D> lo;
    lo.init(lane);
    LaneOffsets<64> lz;                        // the weight tiles have 64-key rows whatever D is
    lz.init(lane);
    const int head = head_of_block(p, blockIdx.x);
    const int slot = slot_of_block(p, blockIdx.x);   // two 64-key blocks per scheduled 128-row job
    const Job job = decode_key_job(p, slot >> 1);
    const int kb = 2 * job.rb + (slot & 1);
    const int key0 = kb * kKeyBlock;
    if (key0 >= job.len) return;               // uniform over the workgroup
    const int strict = p.attend_current ? 0 : 1;
    const int64_t qbase = slice_offset(p.q, job.seq, head, job.tok0);
    const int64_t kbase = slice_offset(p.k, job.seq, head, job.tok0);
    const int64_t vbase = slice_offset(p.v, job.seq, head, job.tok0);
    const int64_t dobase = slice_offset(p.d_o, job.seq, head, job.tok0);
    const int n_qb = last_live_row_block(p, head, job) + 1;
    const int kh = wave & 1;                   // which 32 keys this wave reduces
    const int dbw = wave >> 1;                 // and which d-blocks: dbw + 2*i
    // lane offsets of this wave's operand columns, picked once (no run-time table indexing)
    const int za0 = pick_nat<64>(lz, 0, kh), za1 = pick_nat<64>(lz, 1, kh);
    int qb0o[D / 64], qb1o[D / 64];
#pragma unroll
    for (int i = 0; i < D / 64; ++i) { qb0o[i] = pick_nat<D>(lo, 0, dbw + 2 * i); qb1o[i] = pick_nat<D>(lo, 1, dbw + 2 * i); }

    {
        TileCopy<D> kc, vc;
        kc.load(p.k, kbase, key0, job.len);
        vc.load(p.v, vbase, key0, job.len);
        kc.scale(p.scale2);                    // K times the logit scale: the score MFMAs deliver base-2 logits
        kc.store(ktile);
        vc.store(vtile);
    }
    f32x16 dkacc[D / 64], dvacc[D / 64];
#pragma unroll
    for (int i = 0; i < D / 64; ++i) { dkacc[i] = f32x16{0}; dvacc[i] = f32x16{0}; }

    const int qb0 = job.rb;
    // prefetched state of the first step
    float Rn = 1.0f, Gn = 0.0f;
    h16x8 qfn[D / 16];
    {
        const int qi0 = qb0 * kRowBlock + 32 * wave + n;
        load_row_frags<D>(qfn, p.q, qbase, qb0 * kRowBlock + 32 * wave, n, job.len, lane);
        if (qi0 < job.len) {
            const int64_t t = tab_index(p, head, job, qb0, kb) + 32 * wave + n;
            Rn = p.rtab[t]; Gn = p.gtab[t];
        }
    }
    __syncthreads();                           // K, V tiles visible

    wait_global_memory();
    for (int qb = qb0; qb < n_qb; ++qb) {
        const int m0 = qb * kRowBlock;
        const int q0w = m0 + 32 * wave;
        const int qi = q0w + n;
        // (1) this lane's Q row fragments were prefetched during the previous step; its dO
        //     fragments are requested now and not needed before the weights are done.  Each
        //     row is fetched from global memory exactly once: the fragments are also what the
        //     shared Q / dO tiles of the reduction are assembled from.
        h16x8 qf[D / 16], dof[D / 16];
#pragma unroll
        for (int ks = 0; ks < D / 16; ++ks) qf[ks] = qfn[ks];
        load_row_frags<D>(dof, p.d_o, dobase, q0w, n, job.len, lane);
        float R = Rn, Gc = Gn;
        if (qb + 1 < n_qb) {
            const int qin = qi + kRowBlock;
            load_row_frags<D>(qfn, p.q, qbase, q0w + kRowBlock, n, job.len, lane);
            Rn = 1.0f; Gn = 0.0f;
            if (qin < job.len) {
                const int64_t t = tab_index(p, head, job, qb + 1, kb) + 32 * wave + n;
                Rn = p.rtab[t]; Gn = p.gtab[t];
            }
        }
        // (2) row 32*wave + n of the shared Q tile (every wave passed the barrier that ends the
        //     previous step's reduction, so the tiles are free)
#pragma unroll
        for (int ks = 0; ks < D / 16; ++ks)
            *(h16x8*)(qtile + tile_offset<D>(32 * wave + n, 2 * ks + h)) = qf[ks];
        // (3) weights of this wave's 32 queries
        float x[32], dp[32];
        const bool skip = key0 + strict > q0w + 31 || q0w >= job.len;
        if (!skip) {
            float beta[32];
            score_tiles_ps<D>(x, ktile, lo, qf);
            if (key0 + 63 + strict > q0w) mask_step(x, key0 + 32 * h, qi, strict);
            stick_weights<true>(x, beta, R, lane);
#pragma unroll
            for (int ks = 0; ks < D / 16; ++ks)
                *(h16x8*)(dotile + tile_offset<D>(32 * wave + n, 2 * ks + h)) = dof[ks];
            dp_tiles_o<D>(dp, vtile, lo, dof);
            logit_grads<true>(x, beta, dp, Gc, lane);
        } else {
#pragma unroll
            for (int ks = 0; ks < D / 16; ++ks)
                *(h16x8*)(dotile + tile_offset<D>(32 * wave + n, 2 * ks + h)) = dof[ks];
#pragma unroll
            for (int idx = 0; idx < 32; ++idx) { x[idx] = 0.f; dp[idx] = 0.f; }
        }
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            *(h16x8*)(zp + tile_offset<64>(32 * wave + n, 4 * h + c)) = pack8(&x[8 * c]);
            *(h16x8*)(zd + tile_offset<64>(32 * wave + n, 4 * h + c)) = pack8(&dp[8 * c]);
        }
        __syncthreads();                       // weights and tiles of all waves visible
        // (4) dK[key][d] += sum_q dz[q][key] Q[q][d];  dV[key][d] += sum_q a[q][key] dO[q][d]
#pragma unroll
        for (int c2 = 0; c2 < 8; ++c2) {
            h16x8 az = fetch_nat_2<64>(zd, za0, za1, 16 * c2);
            h16x8 ap = fetch_nat_2<64>(zp, za0, za1, 16 * c2);
#pragma unroll
            for (int i = 0; i < D / 64; ++i) {
                dkacc[i] = mfma(az, fetch_nat_2<D>(qtile, qb0o[i], qb1o[i], 16 * c2), dkacc[i]);
                dvacc[i] = mfma(ap, fetch_nat_2<D>(dotile, qb0o[i], qb1o[i], 16 * c2), dvacc[i]);
            }
        }
        wait_global_memory();                  // nothing in flight across the back edge
        __syncthreads();                       // reduction done: tiles may be overwritten
    }
    // accumulator rows are keys 32*kh + ..., columns d = 32*(dbw + 2*i) + n (the weight tiles
    // are in natural key order); the last barrier of the loop has freed the weight tiles
    char* stage_k = zp;                        // [64 keys][D] bf16 each: kZTile >= kTile
    char* stage_v = zd;
#pragma unroll
    for (int i = 0; i < D / 64; ++i) {
        stage_acc_tile<D>(stage_k, 32 * kh, 32 * (dbw + 2 * i), dkacc[i], p.scale, lane);
        stage_acc_tile<D>(stage_v, 32 * kh, 32 * (dbw + 2 * i), dvacc[i], 1.0f, lane);
    }
    __syncthreads();
    const int64_t dkbase = slice_offset(p.dk, job.seq, head, job.tok0);
    const int64_t dvbase = slice_offset(p.dv, job.seq, head, job.tok0);
    store_staged_rows<D>(stage_k, p.dk, dkbase, key0, job.len, threadIdx.x, kThreads);
    store_staged_rows<D>(stage_v, p.dv, dvbase, key0, job.len, threadIdx.x, kThreads);
}

// ---------------------------------------------------------------- pass 2, head_dim 64
// dK/dV as ONE resident workgroup per CU that runs its share of the (key block, head) items
// back to back as a single stream of 128-query steps, with the two halves of a step given to
// different waves:
//   waves 0..3 ("producers") turn 32 queries x 64 keys each into weights and logit gradients
//     and leave them, as bf16 [query][key] rows, in one of two LDS buffers;
//   waves 4..7 ("consumers") reduce the buffer of the previous step into dK and dV with
//     MFMAs, and stage what the next step needs (Q / dO tiles, per-query carries, and at an
//     item boundary the next K / V tiles) from global memory into LDS with coalesced loads.
// A SIMD holds one wave of each kind, so matrix and memory work run under the producers'
// vector work, and because the stream never stops at an item boundary nothing of an item's
// set-up (launch, K/V fetch, first tiles) or tear-down (dK/dV store) is exposed.
//
// One iteration s of the stream (workgroup barrier A at its end):
//   producers:  fragments of tile[s&1] -> scores, weights, dP, dz -> Z[s&1]                    | A
//   consumers:  store a staged dK/dV; request step s+1;
//               reduce Z/tile[(s-1)&1]; [B] stage a finished dK/dV into Z[(s-1)&1];
//               deposit step s+1 -> tile[(s+1)&1]                                              | A
// A consumer wave deposits exactly the part of the tiles that its own reduction reads, so the
// refill of buffer (s+1)&1 = (s-1)&1 only has to follow that wave's own reads.  B, needed only
// where a finished dK/dV is staged into the Z buffer that all four consumers have just read, is
// a barrier of the consumer waves alone (a running count in LDS): the producers - the critical
// path - never wait in the middle of a step.  Two rarer hand-overs: a staged dK/dV occupies the Z buffer that the producers write in the next
// iteration, so that iteration has one more workgroup barrier (X) after the consumers' store;
// and the K tile is refilled only after a second LDS count says that every producer holds
// the current item's K fragments.
// An item's accumulators are complete after the reduction that follows its last step; they are
// staged after that iteration's B and written to global memory before the next iteration's B.
// The stream kernel's two internal waits are on counters in LDS that waves of the same
// (resident) workgroup bump, so they end within microseconds.  They are bounded all the same: a
// wave that has slept through kSpinLimit polls stops waiting, raises the launch's error word
// (KParams::gave_up, the last 256 bytes of the backward scratch) and runs on, so that the kernel
// always drains; its results are then meaningless.
constexpr int kSpinLimit = 1 << 22;            // polls of 64+ clocks each: more than 0.1 s
__device__ inline void wait_for_count(int* counter, int target, int* gave_up) {
    for (int i = 0; i < kSpinLimit; ++i) {
        if (__hip_atomic_load(counter, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) >= target) return;
        __builtin_amdgcn_s_sleep(1);
    }
    if (gave_up && (threadIdx.x & 63) == 0) *gave_up = 1;
}

// Weights and logit gradients of ONE [32 keys x 32 queries] tile whose lanes hold 16 consecutive keys
// (the own-keys and paired kernels and the eight-producer stream): the carries enter per 32 keys.
template <class Between>
__device__ inline void own_tile_weights(float (&x)[16], float (&beta)[16], float Rin, int lane, Between&& between) {
    const float L = product_chain_with<true, 16>(x, beta, between);
    float Llo, Lup;
    half_values(L, Llo, Lup);
    scale_clamped<16>(x, (lane >= 32) ? Rin : Rin * Lup);         // upper half-wave: the right 16 keys
}
__device__ inline void own_tile_grads(const float (&a)[16], const float (&beta)[16], float (&dp)[16], float Gin,
                                      int lane) {
    float c = 0.f, pre[16];
#pragma unroll
    for (int idx = 0; idx < 16; ++idx) {
        dp[idx] = a[idx] * dp[idx];     // g
        c += dp[idx];
        pre[idx] = c;
    }
    float clo, cup;
    half_values(c, clo, cup);
    const float F = (lane >= 32) ? Gin + clo : Gin;
#pragma unroll
    for (int idx = 0; idx < 16; ++idx) dp[idx] = __builtin_fmaf(-beta[idx], pre[idx] + F, dp[idx]);
}

struct KeyItem {
    Job job;
    int head, kb, key0, n_steps;
    bool valid;
};

__device__ inline KeyItem decode_item(const KParams& p, int idx) {
    KeyItem r;
    r.valid = idx >= 0;
    if (idx < 0) idx = 0;
    r.head = head_of_block<kStreamItems>(p, idx);
    const int slot = slot_of_block(p, idx);          // two 64-key blocks per scheduled 128-row job
    r.job = decode_key_job(p, slot >> 1);
    r.kb = 2 * r.job.rb + (slot & 1);
    r.key0 = r.kb * kKeyBlock;
    r.n_steps = last_live_row_block(p, r.head, r.job) + 1 - r.job.rb;
    return r;
}

// NP = number of producer waves.  4: producer w does queries 32w.. of the step against all 64 keys
// (one wave per SIMD computes weights).  8: producer w does queries 32(w%4).. against the 32 keys
// 32(w/4).. of the block - two producers per SIMD, which is what lets a SIMD issue their vector
// instructions back to back (one wave alone issues one every 2.2-2.7 ns, two together one every
// 1.1-1.2 ns); the half blocks take the mid-block carries of the dQ pass, like the own-keys kernel.
template <int D, int NP>
__global__ __launch_bounds__((NP + 4) * 64, NP == 4 ? 2 : 3) void mfma_bwd_dkv_stream_kernel(KParams p) {
    constexpr int kTile = 64 * D * 2;          // K or V tile (64 keys)
    constexpr int kQTile = 128 * D * 2;        // Q or dO tile (128 queries)
    constexpr int kZTile = 128 * 64 * 2;       // weights of one step, [query][key] bf16
    constexpr int kBuf = 2 * kZTile + 2 * kQTile;
    constexpr int kCarry = kRowBlock * 16;      // {R, G, R mid-block, G mid-block} per query
    __shared__ __attribute__((aligned(1024))) char lds[3 * kTile + 2 * kCarry + 2 * kBuf];
    __shared__ int consumers_done;             // consumer waves that have finished a reduction, running total
    __shared__ int producers_took_k;           // producer waves that hold an item's K fragments, running total
    char* vtiles = lds;                        // V of item j in vtiles + (j&1)*kTile
    char* ktile = vtiles + 2 * kTile;          // read once per item, into the producers' registers
    char* carry = ktile + kTile;
    char* bufs = carry + 2 * kCarry;           // per buffer: zp, zd, qtile, dotile

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const bool producer = wave < NP;
    const int w4 = wave & 3;
    const int n = lane & 31, h = lane >> 5;
    const int strict = p.attend_current ? 0 : 1;
    const int n_items = 2 * p.n_jobs * p.n_heads;

    // Items are taken in list order (longest sweeps first).  A job's second key block can lie
    // beyond the end of its sequence: such an item runs like any other, its one step finds
    // nothing to do and nothing is stored, which is cheaper than teaching the pipeline to skip.
    const int G = gridDim.x, g = blockIdx.x;
    // items of class c = index % 8 go to the workgroups of XCD c (workgroups are dealt to the
    // XCDs round-robin): with the head count a multiple of 8 a head's K, V, Q, dO and carries
    // then stay in one XCD's L2.  Inside a class the workgroups walk the list boustrophedon,
    // which evens out the sweep lengths (the list is sorted by them).
    const int W = G >> 3, w = g >> 3, c8 = g & 7;
    auto static_item = [&](int r) { const int i = 8 * (r * W + ((r & 1) ? W - 1 - w : w)) + c8; return i < n_items ? i : -1; };
    int cur_idx = static_item(0);
    int nxt_idx = static_item(1);
    KeyItem cur = decode_item(p, cur_idx);
    if (!cur.valid) return;                    // uniform over the workgroup
    KeyItem nxt = decode_item(p, nxt_idx);
    int ring = 2;                              // round of the item after `nxt`
    if (threadIdx.x == 0) { consumers_done = 0; producers_took_k = 0; }

    if (producer) {
        LaneOffsets<D> lo;
        lo.init(lane);
        __syncthreads();                       // first item's tiles and carries visible
        int s = 0;
        bool staged_prev = false;              // the consumers staged a dK/dV in the previous iteration
        // (no logit scale here: the Q tiles hold q times scale * log2 e, see store_scaled_q)
        if constexpr (NP == 8) {
        const int kh = wave >> 2;              // this wave's half of the 64-key block
        for (int item = 0;; ++item) {
            const char* vtile = vtiles + (item & 1) * kTile;
            // rows 32kh.. of the K and V tiles are this wave's keys, in the order that puts 16
            // consecutive keys into a lane's accumulator registers (see request_keys)
            h16x8 kfr[D / 16], vfr[D / 16];
#pragma unroll
            for (int ks = 0; ks < D / 16; ++ks) {
                kfr[ks] = fetch_rows_o<D>(ktile, lo, kh, ks);
                vfr[ks] = fetch_rows_o<D>(vtile, lo, kh, ks);
            }
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
            if (lane == 0) __hip_atomic_fetch_add(&producers_took_k, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
            const int key0 = cur.key0 + 32 * kh;
            const int len = cur.job.len;
            for (int it = 0; it < cur.n_steps; ++it, ++s) {
                const bool x_now = staged_prev;
                staged_prev = it == 0 && item > 0;
                char* zp = bufs + (s & 1) * kBuf;
                char* zd = zp + kZTile;
                const char* qtile = zd + kZTile;
                const char* dotile = qtile + kQTile;
                const int q0w = (cur.job.rb + it) * kRowBlock + 32 * w4;
                const int qi = q0w + n;
                const bool skip = key0 + strict > q0w + 31 || q0w >= len || key0 >= len;
                // (one branch holds the whole step of a wave that has work: split in two around barrier X, the
                // weights would be values that "flow" through the idle path as well, and the compiler then keeps
                // a copy of all of them across the loop)
                if (!skip) {
                    float x[16], beta[16], dp[16];
                    const float4 cv = *(const float4*)(carry + (s & 1) * kCarry + (32 * w4 + n) * 16);
                    // table entries of pairs that no query of the row sees are not written
                    const bool sees = qi < len && qi - strict - key0 + 1 > 0;
                    const float Rt = sees ? (kh ? cv.x : cv.z) : 1.0f;
                    const float Gt = sees ? (kh ? cv.w : cv.y) : 0.0f;
                    h16x8 qf[D / 16], dof[D / 16];
#pragma unroll
                    for (int ks = 0; ks < D / 16; ++ks) {
                        qf[ks] = fetch_rows_o<D>(qtile, lo, w4, ks);
                        dof[ks] = fetch_rows_o<D>(dotile, lo, w4, ks);
                    }
                    f32x16 acc = {0};
#pragma unroll
                    for (int ks = 0; ks < D / 16; ++ks) acc = mfma(kfr[ks], qf[ks], acc);
#pragma unroll
                    for (int r = 0; r < 16; ++r) x[r] = acc[r];
                    if (key0 + 31 + strict > q0w || q0w + 31 >= len) {        // diagonal or ragged tile
                        const int nvis = qi < len ? qi - strict - (key0 + 16 * h) + 1 : 0;
#pragma unroll
                        for (int idx = 0; idx < 16; ++idx)
                            if (idx >= nvis) x[idx] = -INFINITY;
                    }
                    // dP = dO V^T: one MFMA behind each of the chain's four segments
                    static_assert(D == 64, "one dP MFMA per chain segment");
                    f32x16 dacc;
                    own_tile_weights(x, beta, Rt, lane, [&](int seg) {
                        dacc = mfma(vfr[seg], dof[seg], seg == 0 ? f32x16{0} : dacc);
                    });
#pragma unroll
                    for (int r = 0; r < 16; ++r) dp[r] = dacc[r];
                    if (x_now) __syncthreads();    // X
                    own_tile_grads(x, beta, dp, Gt, lane);
#pragma unroll
                    for (int c = 0; c < 2; ++c) {
                        *(h16x8*)(zp + tile_offset<64>(32 * w4 + n, 4 * kh + 2 * h + c)) = pack8(&x[8 * c]);
                        *(h16x8*)(zd + tile_offset<64>(32 * w4 + n, 4 * kh + 2 * h + c)) = pack8(&dp[8 * c]);
                    }
                } else {
                    if (x_now) __syncthreads();    // X
                    const h16x8 none = {0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
                    for (int c = 0; c < 2; ++c) {
                        *(h16x8*)(zp + tile_offset<64>(32 * w4 + n, 4 * kh + 2 * h + c)) = none;
                        *(h16x8*)(zd + tile_offset<64>(32 * w4 + n, 4 * kh + 2 * h + c)) = none;
                    }
                }
                __syncthreads();               // A
            }
            if (!nxt.valid) break;
            cur = nxt;
            nxt = decode_item(p, static_item(ring));
            ++ring;
        }
        } else {
        for (int item = 0;; ++item) {
            const char* vtile = vtiles + (item & 1) * kTile;
            // the key block of an item never changes: its score and dP operands stay in registers
            h16x8 kfr[2][D / 16], vfr[2][D / 16];
#pragma unroll
            for (int t = 0; t < 2; ++t)
#pragma unroll
                for (int ks = 0; ks < D / 16; ++ks) {
                    kfr[t][ks] = fetch_rows_o<D>(ktile, lo, t, ks);
                    vfr[t][ks] = fetch_rows_o<D>(vtile, lo, t, ks);
                }

            // tell the consumers that the K tile may be refilled
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
            if (lane == 0) __hip_atomic_fetch_add(&producers_took_k, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
            const int key0 = cur.key0;
            const int len = cur.job.len;
            for (int it = 0; it < cur.n_steps; ++it, ++s) {
                // A dK/dV staged in the previous iteration sits in the Z buffer this iteration
                // writes: wait (barrier X) until the consumers have stored it.
                const bool x_now = staged_prev;
                staged_prev = it == 0 && item > 0;
                char* zp = bufs + (s & 1) * kBuf;
                char* zd = zp + kZTile;
                const char* qtile = zd + kZTile;
                const char* dotile = qtile + kQTile;
                const int q0w = (cur.job.rb + it) * kRowBlock + 32 * w4;
                const int qi = q0w + n;
                const bool skip = key0 + strict > q0w + 31 || q0w >= len;
                // (one branch for the whole step, see above)
                if (!skip) {
                    float x[32], beta[32], dp[32];
                    // Both carries that enter this LANE's 32 keys come from the tables: the right half-wave
                    // takes the forward's block-edge product and the mid-block prefix, the left one the
                    // mid-block product and the block-edge prefix - no exchange between the halves, and the
                    // prefix sums run in one pass.  Entries of (query, half block) pairs that the query does not
                    // see are not written: their weights are zero whatever the carry.  Rows past the end of
                    // the sequence hold copies of its last row: a zero carry makes their weights and
                    // gradients exactly zero.
                    const float4 cv = *(const float4*)(carry + (s & 1) * kCarry + (32 * w4 + n) * 16);
                    const bool sees = qi < len && qi - strict - (key0 + 32 * h) + 1 > 0;
                    const float R = sees ? (h ? cv.x : cv.z) : (qi < len ? 1.0f : 0.0f);
                    const float Gc = sees ? (h ? cv.w : cv.y) : 0.0f;
                    h16x8 qf[D / 16], dof[D / 16];
#pragma unroll
                    for (int ks = 0; ks < D / 16; ++ks) {
                        qf[ks] = fetch_rows_o<D>(qtile, lo, w4, ks);
                        dof[ks] = fetch_rows_o<D>(dotile, lo, w4, ks);
                    }
                    f32x16 raw[2];
#pragma unroll
                    for (int t = 0; t < 2; ++t) {
                        f32x16 acc = {0};
#pragma unroll
                        for (int ks = 0; ks < D / 16; ++ks) acc = mfma(kfr[t][ks], qf[ks], acc);
                        raw[t] = acc;
                    }
#pragma unroll
                    for (int t = 0; t < 2; ++t)
#pragma unroll
                        for (int r = 0; r < 16; ++r) x[16 * t + r] = raw[t][r];
                    if (key0 + 63 + strict > q0w) mask_step(x, key0 + 32 * h, qi, strict);
                    // dP = dO V^T does not depend on the weights: its eight MFMAs go between the
                    // segments of the chain, where the chain's exp/rcp overlap them
                    static_assert(D == 64, "one dP MFMA per chain segment");
                    f32x16 dacc[2];
                    carried_chain_with<true, 32>(x, beta, R, [&](int seg) {      // finished weights: no scaling pass
                        const int t = seg & 1, ks = seg >> 1;
                        dacc[t] = mfma(vfr[t][ks], dof[ks], ks == 0 ? f32x16{0} : dacc[t]);
                    });
#pragma unroll
                    for (int t = 0; t < 2; ++t)
#pragma unroll
                        for (int r = 0; r < 16; ++r) dp[16 * t + r] = dacc[t][r];
                    if (x_now) __syncthreads();    // X
                    logit_grads_from<32>(x, beta, dp, Gc);
#pragma unroll
                    for (int c = 0; c < 4; ++c) {
                        *(h16x8*)(zp + tile_offset<64>(32 * w4 + n, 4 * h + c)) = pack8(&x[8 * c]);
                        *(h16x8*)(zd + tile_offset<64>(32 * w4 + n, 4 * h + c)) = pack8(&dp[8 * c]);
                    }
                } else {
                    if (x_now) __syncthreads();    // X
                    const h16x8 none = {0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
                    for (int c = 0; c < 4; ++c) {
                        *(h16x8*)(zp + tile_offset<64>(32 * w4 + n, 4 * h + c)) = none;
                        *(h16x8*)(zd + tile_offset<64>(32 * w4 + n, 4 * h + c)) = none;
                    }
                }
                __syncthreads();               // A
            }
            if (!nxt.valid) break;
            cur = nxt;
            nxt = decode_item(p, static_item(ring));
            ++ring;
        }
        }
        __syncthreads();                       // A of the draining iteration
    } else {
        LaneOffsets<D> lo;
        lo.init(lane);
        LaneOffsets<64> lz;                    // the weight tiles have 64-key rows whatever D is
        lz.init(lane);
        const int ct = threadIdx.x & (kThreads - 1);
        // Wave w4 reduces ONE of the two outputs (even: dK from dz and Q, odd: dV from a and dO),
        // all 64 keys of it and one 32-wide d-block: the two key halves share the Q / dO operand,
        // three operand fetches per two MFMAs instead of four.
        static_assert(D == 64, "the consumers' tiling assumes two 32-wide d-blocks");
        const bool is_dv = w4 & 1;
        const int dbw = w4 >> 1;
        int za[2][2];
#pragma unroll
        for (int kh = 0; kh < 2; ++kh) { za[kh][0] = pick_nat<64>(lz, 0, kh); za[kh][1] = pick_nat<64>(lz, 1, kh); }
        const int qb0o = pick_nat<D>(lo, 0, dbw), qb1o = pick_nat<D>(lo, 1, dbw);
        f32x16 acc[2];                         // key halves
        acc[0] = f32x16{0}; acc[1] = f32x16{0};

        // Staging registers of one step.  A consumer wave stages exactly the part of the step's
        // tiles that its own reduction reads - the 32-wide d-block `dbw` of Q (dK waves) or of dO
        // (dV waves), all 128 rows: lane l holds the 16-byte chunk l%4 of rows l/4 + 16*part - so
        // refilling a tile buffer needs no barrier among the consumers (the producers, who read
        // whole rows, are kept apart from it by A).  Threads ct < 128 also stage the carries of
        // query ct.  Every request is unconditional, with rows clamped to the sequence, and every
        // iteration consumes what it requested: no register is "perhaps still being loaded" on
        // some path, so the compiler's wait-count bookkeeping stays exact.
        u32x4 tx[8];
        float cR, cG, cRm = 1.f, cGm = 0.f;
        // Four lanes fill the 64 bytes of a row that this wave reduces; an LDS write cycle takes eight
        // lanes, i.e. two rows, whose swizzles must differ in the bit that selects the other half of the
        // row's banks: rows r and r + 2 do (r and r + 1 would collide), hence the order 0 2 1 3 ...
        const int crow4 = lane >> 2;
        const int crow = (crow4 & ~3) | ((crow4 & 1) << 1) | ((crow4 >> 1) & 1), cch = 4 * dbw + (lane & 3);
        // Per-item base pointers, worked out once per item and held in VECTOR registers (which
        // the consumers have to spare): a step's requests then cost a few vector instructions.
        // Left to itself the compiler keeps such uniform values in scalar registers, runs out
        // of them, and re-derives the pointers from the kernel arguments in every iteration
        // (a wave issues one instruction every four or five cycles, scalar ones included, and
        // the consumers' share of a step is short).
        struct ItemPtrs {
            const char* x;                     // Q or dO: row 0 of the sequence, this head, this thread's chunk
            const float *rt, *gt;              // carries of this (head, key block): row block 0, query 0
            const float *rm, *gm;              // the mid-block carries
            int row0, len;                     // first query of the item's sweep; sequence length
        };
        auto item_ptrs = [&](const KeyItem& t) {
            ItemPtrs r;
            const TensorArg& xt = is_dv ? p.d_o : p.q_scaled;      // Q as the dQ pass left it: times scale * log2 e
            r.x = xt.ptr + 2 * ((int64_t)t.job.seq * xt.sb + (int64_t)t.head * xt.sh + (int64_t)t.job.tok0 * xt.st) + cch * 16;
            const int64_t tk = tab_index(p, t.head, t.job, 0, t.kb);
            r.rt = p.rtab + tk;
            r.gt = p.gtab + tk;
            r.rm = p.rmid + tk;
            r.gm = p.gmid + tk;
            r.row0 = t.job.rb * kRowBlock;
            r.len = t.job.len;
            asm volatile("" : "+v"(r.x), "+v"(r.rt), "+v"(r.gt));
            asm volatile("" : "+v"(r.rm), "+v"(r.gm));
            return r;
        };
        const uint32_t x_st2 = 2u * (uint32_t)(is_dv ? p.d_o.st : p.q_scaled.st);
        auto request_step = [&](const ItemPtrs& t, int row0) {
            const int qi = min(row0 + (ct & (kRowBlock - 1)), t.len - 1);
            const int qb = qi >> 7;            // row block of the query: its slab starts qb*(qb+1) columns in
            const int64_t ix = (int64_t)qb * (qb + 1) * kRowBlock + (qi & (kRowBlock - 1));
            // (The pointers went through registers that the compiler cannot see into, see item_ptrs: it no longer knows
            // that they point to global memory, and plain loads would become FLAT instructions, which also count as LDS
            // traffic - every wait for an LDS read in the reduction would wait for these loads too.)
            auto gl = [](const float* q) { return *(const __attribute__((address_space(1))) float*)q; };
            cR = gl(t.rt + ix); cG = gl(t.gt + ix);
            cRm = gl(t.rm + ix); cGm = gl(t.gm + ix);
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const uint32_t row = (uint32_t)min(row0 + crow + 16 * i, t.len - 1);
                tx[i] = *(const __attribute__((address_space(1))) u32x4*)(t.x + (size_t)row * x_st2);
            }
        };
        constexpr int kLoadsPerStep = 8 + 4;        // per lane: what request_step issues
        // K and V tiles of an item go straight from global memory into LDS (no registers, and
        // nothing for the wait-count bookkeeping to track): every instruction moves 64 x 16 bytes
        // into 1 KB of consecutive LDS, the lane picks the global chunk that belongs at its LDS
        // position (rows in MFMA order, chunks swizzled).  Rows past the end are clamped: those
        // keys are masked for every valid query and their dK/dV rows are not stored.
        auto request_keys = [&](const KeyItem& t, char* vdst) {
            const int64_t kbase = (int64_t)t.job.seq * p.k.sb + (int64_t)t.head * p.k.sh + (int64_t)t.job.tok0 * p.k.st;
            const int64_t vbase = (int64_t)t.job.seq * p.v.sb + (int64_t)t.head * p.v.sh + (int64_t)t.job.tok0 * p.v.st;
#pragma unroll
            for (int i2 = 0; i2 < 2; ++i2) {
                const int inst = w4 + 4 * i2;              // 8 instructions per tile over 4 waves
                const int pos = inst * 64 + lane;          // LDS chunk position
                const int r = pos / (D / 8), pc = pos % (D / 8);
                const int c = pc ^ swz<D>(r);
                // NP = 4: the accumulator registers of a producer lane are 32 consecutive keys over its two
                // tiles; NP = 8: 16 consecutive keys of the one tile (rows 32kh..) of producer half kh
                const int kl = NP == 4 ? (((r >> 2) & 1) << 5) | (((r >> 5) & 1) << 4) | (((r >> 3) & 3) << 2) | (r & 3)
                                       : (((r >> 5) & 1) << 5) | (((r >> 2) & 1) << 4) | (((r >> 3) & 3) << 2) | (r & 3);
                const int row = min(t.key0 + kl, t.job.len - 1);
                // (the copy as inline assembly, see TileDma: through the builtin, the first LDS fetch of EVERY iteration's
                // reduction waited for all vector-memory traffic, the tiles just requested for step s + 2 included)
                dma16(p.k.ptr + 2 * kbase, 2u * (uint32_t)(row * (int)p.k.st + c * 8), lds_address(ktile + inst * 1024));
                dma16(p.v.ptr + 2 * vbase, 2u * (uint32_t)(row * (int)p.v.st + c * 8), lds_address(vdst + inst * 1024));
            }
        };
        auto deposit = [&](int s) {
            char* xtile = bufs + (s & 1) * kBuf + 2 * kZTile + (is_dv ? kQTile : 0);
#pragma unroll
            for (int i = 0; i < 8; ++i) *(u32x4*)(xtile + tile_offset<D>(crow + 16 * i, cch)) = tx[i];
            if (ct < kRowBlock) {
                *(float4*)(carry + (s & 1) * kCarry + ct * 16) = float4{cR, cG, cRm, cGm};
            }
        };
        auto store_staged = [&](int idx, const char* staging) {
            const KeyItem t = decode_item(p, idx);
            const int64_t dkbase = (int64_t)t.job.seq * p.dk.sb + (int64_t)t.head * p.dk.sh + (int64_t)t.job.tok0 * p.dk.st;
            const int64_t dvbase = (int64_t)t.job.seq * p.dv.sb + (int64_t)t.head * p.dv.sh + (int64_t)t.job.tok0 * p.dv.st;
            store_staged_rows<D>(staging, p.dk, dkbase, t.key0, t.job.len, ct, kThreads);
            store_staged_rows<D>(staging + kTile, p.dv, dvbase, t.key0, t.job.len, ct, kThreads);
        };
        auto stage = [&](char* staging) {
#pragma unroll
            for (int kh = 0; kh < 2; ++kh) {
                // the Q rows carried scale * log2 e: dK = scale * dZ^T Q = (scale / scale2) * the sum
                stage_acc_tile<D>(staging + (is_dv ? kTile : 0), 32 * kh, 32 * dbw, acc[kh], is_dv ? 1.0f : p.scale / p.scale2, lane);
                acc[kh] = f32x16{0};
            }
        };
        // dK[key][d] += sum_q dz[q][key] Q[q][d]  or  dV[key][d] += sum_q a[q][key] dO[q][d].
        // The operands of four 16-query groups are fetched as one batch, so that the MFMAs wait
        // for LDS once per batch rather than once each; `between(b)` (the tile requests) goes
        // behind the fetches of batch b.
        auto reduce = [&](int s_done) {
            const char* zt = bufs + (s_done & 1) * kBuf + (is_dv ? 0 : kZTile);            // a or dz
            const char* xt = bufs + (s_done & 1) * kBuf + 2 * kZTile + (is_dv ? kQTile : 0); // dO or Q
            constexpr int kBatch = NP == 8 ? 2 : 4;        // NP = 8: three waves per SIMD, fewer registers
#pragma unroll
            for (int b = 0; b < 8 / kBatch; ++b) {
                h16x8 aw[kBatch][2], bx[kBatch];
#pragma unroll
                for (int j = 0; j < kBatch; ++j) {
                    const int c2 = kBatch * b + j;
                    aw[j][0] = fetch_nat_2<64>(zt, za[0][0], za[0][1], 16 * c2);
                    aw[j][1] = fetch_nat_2<64>(zt, za[1][0], za[1][1], 16 * c2);
                    bx[j] = fetch_nat_2<D>(xt, qb0o, qb1o, 16 * c2);
                }
#pragma unroll
                for (int j = 0; j < kBatch; ++j) {
                    acc[0] = mfma(aw[j][0], bx[j], acc[0]);
                    acc[1] = mfma(aw[j][1], bx[j], acc[1]);
                }
                if (NP == 8) __builtin_amdgcn_sched_barrier(0);
            }
        };

        // A step's tiles and carries are requested right after the previous step's have been
        // deposited, almost a whole iteration before their own deposit (an iteration is shorter than
        // a round trip to memory plus the reduction: requested at the start of the iteration that
        // deposits them, as an earlier version did, they were waited for).  `front` is the position of
        // the next request in the stream of (item, step) pairs; past the end of the stream it stays on
        // the last step (a harmless repeat).
        struct Front {
            ItemPtrs ptrs;
            int it, n_steps, ring;
            bool done;
        } front;
        front.ptrs = item_ptrs(cur);
        front.it = 0; front.n_steps = cur.n_steps; front.ring = 1; front.done = false;
        auto request_front = [&]() {
            request_step(front.ptrs, front.ptrs.row0 + front.it * kRowBlock);
            if (front.done) return;
            if (front.it + 1 < front.n_steps) { ++front.it; return; }
            const int idx = static_item(front.ring);
            if (idx < 0) { front.done = true; return; }
            const KeyItem t = decode_item(p, idx);
            front.ptrs = item_ptrs(t);
            front.it = 0; front.n_steps = t.n_steps; ++front.ring;
        };
        // Memory operations complete in order: with one step's requests in flight, everything issued
        // before them (a deposited step, K / V tiles, stores) has landed.
        static_assert(kLoadsPerStep < 16, "wait-count immediate");
        auto wait_all_but_requests = [&]() { __builtin_amdgcn_s_waitcnt(0x0F70 | kLoadsPerStep); };
        request_keys(cur, vtiles);
        request_front();
        deposit(0);
        request_front();
        wait_all_but_requests();
        __syncthreads();                       // first item's tiles and carries visible

        int s = 0;
        bool finish_after_reduce = false;      // the step about to be reduced is its item's last
        bool store_pending = false;            // a staged dK/dV waits in Z[s&1] to be stored
        int fin_stage = cur_idx, fin_store = cur_idx;
        // B, a barrier of the four consumer waves only (the producers have no part in what it
        // protects and must not be held up by it): a running count in LDS, bumped by each wave,
        // and a short, bounded spin (all four waves are resident).
        int sync_target = 0;
        auto consumer_sync = [&]() {
            sync_target += 4;
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
            if (lane == 0) __hip_atomic_fetch_add(&consumers_done, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
            wait_for_count(&consumers_done, sync_target, p.gave_up);
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
        };
        // One iteration of the stream: the producers work on step s meanwhile.
        auto iteration = [&](bool last, bool keys_now, int item) {
            if (store_pending) {               // staged in the previous iteration
                store_staged(fin_store, bufs + (s & 1) * kBuf);
                store_pending = false;
                __syncthreads();               // X: the producers may overwrite the staging
            }
            if (keys_now) {
                // the K tile is free once every producer holds this item's fragments; V goes to the
                // tile of the other parity
                wait_for_count(&producers_took_k, NP * (item + 1), p.gave_up);
                __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
                request_keys(decode_item(p, nxt_idx), vtiles + ((item + 1) & 1) * kTile);
            }
            if (s > 0) reduce(s - 1);
            // B, only where a finished dK/dV is staged into the Z buffer just reduced: every
            // consumer must be through with it
            if (finish_after_reduce) {
                consumer_sync();
                stage(bufs + ((s - 1) & 1) * kBuf);
                fin_store = fin_stage;
                store_pending = true;
            }
            deposit(s + 1);                    // requested at the end of the previous iteration
            finish_after_reduce = last;
            if (last) fin_stage = cur_idx;
            __builtin_amdgcn_sched_barrier(0);
            request_front();                   // step s + 2
            wait_all_but_requests();
            __syncthreads();                   // A
            ++s;
        };
        for (int item = 0;; ++item) {
            // The next item's K and V are requested in the second-to-last step
            const int n_steps = cur.n_steps;
            const bool has_next = nxt.valid;
            const int keys_at = n_steps >= 2 ? n_steps - 2 : 0;
            for (int it = 0; it < n_steps; ++it) iteration(it + 1 == n_steps, has_next && it == keys_at, item);
            if (!has_next) break;
            cur_idx = nxt_idx;
            cur = nxt;
            nxt_idx = static_item(ring);
            nxt = decode_item(p, nxt_idx);
            ++ring;
        }
        // draining iteration: the last step of the last item
        if (store_pending) store_staged(fin_store, bufs + (s & 1) * kBuf);
        reduce(s - 1);
        consumer_sync();                       // B
        stage(bufs + ((s - 1) & 1) * kBuf);
        __syncthreads();                       // A (consumers only need each other's staging)
        store_staged(fin_stage, bufs + ((s - 1) & 1) * kBuf);
    }
}

// ---------------------------------------------------------------- pass 2, every wave on its own keys
// One workgroup per (128-key block, head); wave w owns the 32 keys 32w..32w+31 of the block for
// the whole sweep, K and V fragments in registers, and accumulates its [32 keys x D] slices of
// dK and dV itself: nothing is exchanged between waves, and the only workgroup barrier is the
// one that publishes the next 64-query Q / dO tiles (global -> LDS DMA, double-buffered).
// A step covers 64 queries as two [32 keys x 32 queries] score tiles; lane (n, h) holds the 16
// consecutive keys 16h..16h+15 of one query per tile.  The carries that enter the wave's 32 keys
// come from the tables of the forward and of the dQ pass: the block-edge ones for the half of
// a 64-key block that touches the edge, the mid-block ones for the other half.  Weights and
// logit gradients go as bf16 [query][32 a | 32 dz] rows into a tile private to the wave and
// come back transposed as the A operands of  dV += A^T dO  and  dK += dZ^T Q.
// At head_dim 256; at 128 behind the paired kernel and there to test it against.  (At 64, where the paired kernel has replaced it, it took 97 us on a
// pack of 8192 tokens and 745 on one of 65536 (H=16) that the paired kernel takes 89 and 732 on.)
// kSplit: at head_dim 256 the [32 keys x 256] accumulators of dK and dV alone are 256 registers a lane, on top of 128
// for the K and V fragments.  There the grid has kSplit = 2 workgroups per (key block, head), blockIdx.y = 0, 1, and
// workgroup `part` accumulates and stores columns 128 * part .. 128 * part + 127 of dK and dV only; scores, weights and
// logit gradients are formed in both.
template <int D, int kSplit = 1>
__global__ __launch_bounds__(kThreads, 1) void mfma_bwd_dkv_own_kernel(KParams p) {
    constexpr int kNB = D / 32 / kSplit;         // 32-wide column blocks of dK / dV accumulated here
    const int part = kSplit > 1 ? (int)blockIdx.y : 0;
    static_assert(32 * (D / kSplit) * 2 <= 64 * 64 * 2, "a wave stages its [32 keys x columns] outputs in its weight tile");
    constexpr int kQTile = 64 * D * 2;           // Q or dO tile of one step (64 queries)
    constexpr int kZTile = 64 * 64 * 2;          // per wave: [64 queries][32 a | 32 dz] bf16
    constexpr int kStep = 64;
    // At head_dim 128 a SIMD holds one wave, so nothing but the wave itself can keep the matrix cores
    // busy during its exp/rcp: there the reduction over a step's second tile waits for the NEXT step
    // and goes between the segments of that step's first chain.  The Q / dO tiles of a step then
    // have to outlive it by one step: three tile buffers instead of two.
    constexpr bool kDefer = D == 128;
    constexpr int kNBuf = kDefer ? 3 : 2;
    __shared__ __attribute__((aligned(16))) char lds[2 * kNBuf * kQTile + 4 * kZTile];   // Q, dO per buffer | one Z tile per wave

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int n = lane & 31, h = lane >> 5;
    LaneOffsets<D> lo;
    lo.init(lane);
    LaneOffsets<64> lz;
    lz.init(lane);
    const int head = head_of_block(p, blockIdx.x);
    const Job job = decode_key_job(p, slot_of_block(p, blockIdx.x));
    const int strict = p.attend_current ? 0 : 1;
    const int q_begin = job.rb * kRowBlock;            // first key of the block = first query that may see it
    const int kb0 = q_begin + 32 * wave;               // first key of this wave
    char* ztile = lds + 2 * kNBuf * kQTile + wave * kZTile;

    const int64_t qbase = slice_offset(p.q, job.seq, head, job.tok0);
    const int64_t kbase = slice_offset(p.k, job.seq, head, job.tok0);
    const int64_t vbase = slice_offset(p.v, job.seq, head, job.tok0);
    const int64_t dobase = slice_offset(p.d_o, job.seq, head, job.tok0);

    // A operands of the score tiles: MFMA row m holds key 16*((m>>2)&1) + 4*(m>>3) + (m&3) of
    // the wave, so that the accumulator registers of a lane are 16 consecutive keys
    h16x8 kfr[D / 16], vfr[D / 16];
    {
        const int m = lane & 31;
        const int key = 16 * ((m >> 2) & 1) + 4 * (m >> 3) + (m & 3);
        load_row_frags<D>(kfr, p.k, kbase, kb0, key, job.len, lane);
        load_row_frags<D>(vfr, p.v, vbase, kb0, key, job.len, lane);
        prescale_frags(kfr, p.scale2);         // K times the logit scale: the score MFMAs deliver base-2 logits
    }

    f32x16 dkacc[kNB], dvacc[kNB];
#pragma unroll
    for (int db = 0; db < kNB; ++db) { dkacc[db] = f32x16{0}; dvacc[db] = f32x16{0}; }

    const int n_steps = min((job.len - q_begin + kStep - 1) / kStep, 2 * (last_live_row_block(p, head, job) + 1 - job.rb));

    TileDma<D, true> qc, dc;
    qc.init(lane, wave, p.q, qbase);
    dc.init(lane, wave, p.d_o, dobase);
    if (n_steps > 0) {
        qc.issue(q_begin, job.len, lds);
        dc.issue(q_begin, job.len, lds + kQTile);
    }

    // carries of a (query, this wave's 32 keys) pair: the right half of a 64-key block takes the
    // forward's block-edge carry and the mid-block prefix, the left half the other two
    const int kb64 = (q_begin + 32 * wave) / kKeyBlock;      // 2*rb or 2*rb + 1: a column of every row block's slab from rb on
    const float* rsrc = ((wave & 1) ? p.rtab : p.rmid) + tab_index(p, head, job, 0, kb64) + n;
    const float* gsrc = ((wave & 1) ? p.gmid : p.gtab) + tab_index(p, head, job, 0, kb64) + n;
    float Rn[2] = {1.f, 1.f}, Gn[2] = {0.f, 0.f};
    // A step's 64 queries lie inside one 128-row block: the table index is a uniform base plus the lane's row.
    // Rows past the end of the sequence are read too (the tables are allocated in whole row blocks) and not used.
    auto request_carries = [&](int q0) {
        const int qb = q0 >> 7;
        const int64_t ix = (int64_t)qb * (qb + 1) * kRowBlock + (q0 & (kRowBlock - 1));      // uniform
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            Rn[t] = rsrc[ix + 32 * t];
            Gn[t] = gsrc[ix + 32 * t];
        }
    };
    if (n_steps > 0) request_carries(q_begin);
    wait_global_memory();
    __syncthreads();

    // Every LDS address of the loop is "a register that is fixed for the whole sweep + a constant": the lane offsets are
    // made absolute once (Q / dO tiles from the start of the array, the weight tile from this wave's tile), and the loop
    // runs in one copy per tile buffer, so that buffer and row offsets are compile-time numbers in the offset fields of
    // the fetches (with the tile address in a scalar register each fetch or pinned sum costs a vector add with a scalar
    // operand: 25 of them per step here).
    if (kSplit > 1) {
        // this workgroup's column blocks: kNB blocks are 4 * kNB sixteen-byte chunks, a multiple of 16, and the swizzle
        // only touches chunk bits 0..3, so block b + part * kNB lies part * kNB * 64 bytes further along the same row
        static_assert(kSplit == 1 || kNB % 4 == 0, "the shift must not meet the swizzled chunk bits");
#pragma unroll
        for (int a = 0; a < 2; ++a)
#pragma unroll
            for (int b = 0; b < kNB; ++b) lo.nat[a][b] += part * (kNB * 64);
    }
    lo.rebase(lds);
    lz.rebase(ztile);
    constexpr TileAt zt{0};
    uint32_t zst[4];              // this lane's row of the weight tile: chunks 2h, 2h + 1 (a) and 4 + 2h, 4 + 2h + 1 (dz)
#pragma unroll
    for (int c = 0; c < 4; ++c) zst[c] = lds_lane_base(ztile, tile_offset<64>(n, (c >> 1) * 4 + 2 * h + (c & 1)));
    auto put_z = [&](int c, int t, h16x8 v) __attribute__((always_inline)) {
        *(__attribute__((address_space(3))) h16x8*)((__attribute__((address_space(3))) char*)(uintptr_t)zst[c] + t * 32 * 64 * 2) = v;
    };

    auto second_tile_reduction = [&](auto qt, auto dot) __attribute__((always_inline)) {
#pragma unroll
        for (int kk = 2; kk < 4; ++kk) {
            const h16x8 af = fetch_nat_o<64>(zt, lz, 16 * kk, 0);
            const h16x8 zf = fetch_nat_o<64>(zt, lz, 16 * kk, 1);
#pragma unroll
            for (int db = 0; db < kNB; ++db) {
                dvacc[db] = mfma(af, fetch_nat_o<D>(dot, lo, 16 * kk, db), dvacc[db]);
                dkacc[db] = mfma(zf, fetch_nat_o<D>(qt, lo, 16 * kk, db), dkacc[db]);
            }
        }
    };
    bool pending = false;                      // the previous step left its second tile's reduction to this one
    auto do_step = [&](int step, auto buf_c) __attribute__((always_inline)) {
        constexpr int buf = decltype(buf_c)::value;
        constexpr int nbuf = buf + 1 == kNBuf ? 0 : buf + 1;
        constexpr int pbuf = buf == 0 ? kNBuf - 1 : buf - 1;
        constexpr TileAt qtile{buf * 2 * kQTile}, dotile{buf * 2 * kQTile + kQTile};
        constexpr TileAt pqtile{pbuf * 2 * kQTile}, pdotile{pbuf * 2 * kQTile + kQTile};      // the previous step's tiles (kDefer)
        const int q0 = q_begin + step * kStep;
        const bool more = step + 1 < n_steps;
        float Rin[2], Gin[2];
#pragma unroll
        for (int t = 0; t < 2; ++t) { Rin[t] = Rn[t]; Gin[t] = Gn[t]; }
        if (more) {       // next tiles, straight into the next buffer (nobody reads it since the last barrier)
            qc.issue(q0 + kStep, job.len, lds + nbuf * 2 * kQTile);
            dc.issue(q0 + kStep, job.len, lds + nbuf * 2 * kQTile + kQTile);
            request_carries(q0 + kStep);
        }
        // whole step left of this wave's first key: nothing visible
        const bool skip = kb0 + strict > q0 + kStep - 1 || kb0 >= job.len;
        if (!skip) {
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                const int qt0 = q0 + 32 * t;
                const int qi = qt0 + n;
                // visible keys among this lane's 16 (queries past the end see none)
                const int nvis = qi < job.len ? qi - strict - (kb0 + 16 * h) + 1 : 0;
                const bool sees_wave = qi < job.len && qi - strict - kb0 + 1 > 0;
                const float Rt = sees_wave ? Rin[t] : 1.0f;      // table entries of invisible pairs are not written
                const float Gt = sees_wave ? Gin[t] : 0.0f;
                float x[16], beta[16], dp[16];
                {
                    // with one wave on the SIMD (d = 128) nothing hides an LDS round trip in front of
                    // each MFMA: all operands of the tile are requested first
                    h16x8 bq[D / 16];
#pragma unroll
                    for (int ks = 0; ks < D / 16; ++ks) bq[ks] = fetch_rows_o<D>(qtile, lo, t, ks);
                    if (D == 128) __builtin_amdgcn_sched_barrier(0);
                    f32x16 acc = {0};
#pragma unroll
                    for (int ks = 0; ks < D / 16; ++ks) acc = mfma(kfr[ks], bq[ks], acc);
#pragma unroll
                    for (int r = 0; r < 16; ++r) x[r] = acc[r];
                }
                if (kb0 + 31 + strict > qt0 || qt0 + 31 >= job.len) {     // diagonal or ragged tile
#pragma unroll
                    for (int idx = 0; idx < 16; ++idx)
                        if (idx >= nvis) x[idx] = -INFINITY;
                }
                if (t == 0 && kDefer && pending) {
                    // the previous step's second tile: rows 32.. of the wave's weight tile (not yet
                    // overwritten: this step's second tile comes later) and of the previous Q / dO tiles
                    auto red_a = [&](int seg) { return fetch_nat_o<64>(zt, lz, 32 + 16 * (seg >> 1), seg & 1); };
                    auto red_b = [&](int seg, int db) {
                        return (seg & 1) ? fetch_nat_o<D>(pqtile, lo, 32 + 16 * (seg >> 1), db) : fetch_nat_o<D>(pdotile, lo, 32 + 16 * (seg >> 1), db);
                    };
                    h16x8 na = red_a(0), nb[kNB];
#pragma unroll
                    for (int db = 0; db < kNB; ++db) nb[db] = red_b(0, db);
                    own_tile_weights(x, beta, Rt, lane, [&](int seg) {
                        const h16x8 ca = na;
                        h16x8 cb[kNB];
#pragma unroll
                        for (int db = 0; db < kNB; ++db) cb[db] = nb[db];
                        if (seg < 3) {
                            na = red_a(seg + 1);
#pragma unroll
                            for (int db = 0; db < kNB; ++db) nb[db] = red_b(seg + 1, db);
                        }
#pragma unroll
                        for (int db = 0; db < kNB; ++db) {
                            if (seg & 1) dkacc[db] = mfma(ca, cb[db], dkacc[db]);
                            else dvacc[db] = mfma(ca, cb[db], dvacc[db]);
                        }
                    });
                } else if (t == 0) {
                    own_tile_weights(x, beta, Rt, lane, [](int) {});
                } else {
                    // The reduction over the first tile's 32 queries only needs that tile's weights, which
                    // this wave wrote above: its MFMAs go between the segments of the second tile's chain,
                    // whose exp/rcp overlap them.  Segment 2kk: dV += A^T dO, segment 2kk + 1: dK += dZ^T Q.
                    auto red_a = [&](int seg) { return fetch_nat_o<64>(zt, lz, 16 * (seg >> 1), seg & 1); };
                    auto red_b = [&](int seg, int db) {
                        return (seg & 1) ? fetch_nat_o<D>(qtile, lo, 16 * (seg >> 1), db) : fetch_nat_o<D>(dotile, lo, 16 * (seg >> 1), db);
                    };
                    h16x8 na = red_a(0), nb[kNB];
#pragma unroll
                    for (int db = 0; db < kNB; ++db) nb[db] = red_b(0, db);
                    own_tile_weights(x, beta, Rt, lane, [&](int seg) {
                        const h16x8 ca = na;
                        h16x8 cb[kNB];
#pragma unroll
                        for (int db = 0; db < kNB; ++db) cb[db] = nb[db];
                        if (seg < 3) {
                            na = red_a(seg + 1);
#pragma unroll
                            for (int db = 0; db < kNB; ++db) nb[db] = red_b(seg + 1, db);
                        }
#pragma unroll
                        for (int db = 0; db < kNB; ++db) {
                            if (seg & 1) dkacc[db] = mfma(ca, cb[db], dkacc[db]);
                            else dvacc[db] = mfma(ca, cb[db], dvacc[db]);
                        }
                    });
                }
                {
                    h16x8 bd[D / 16];
#pragma unroll
                    for (int ks = 0; ks < D / 16; ++ks) bd[ks] = fetch_rows_o<D>(dotile, lo, t, ks);
                    if (D == 128) __builtin_amdgcn_sched_barrier(0);
                    f32x16 acc = {0};
#pragma unroll
                    for (int ks = 0; ks < D / 16; ++ks) acc = mfma(vfr[ks], bd[ks], acc);
#pragma unroll
                    for (int r = 0; r < 16; ++r) dp[r] = acc[r];
                }
                // a -> columns 16h.. of row (32t + n), dz -> columns 32 + 16h..
                put_z(0, t, pack8(&x[0]));
                put_z(1, t, pack8(&x[8]));
                own_tile_grads(x, beta, dp, Gt, lane);
                put_z(2, t, pack8(&dp[0]));
                put_z(3, t, pack8(&dp[8]));
            }
            // dV += A^T dO, dK += dZ^T Q over the second tile's queries (the first tile's went with the
            // second chain): now, or with the next step's first chain
            if (!kDefer) second_tile_reduction(qtile, dotile);
            pending = kDefer;
        }
        wait_global_memory();                  // the next tiles and carries have landed
        __syncthreads();
    };
    // one copy of the step per tile buffer
    int last_buf = 0;
    for (int step = 0; step < n_steps; step += kNBuf) {
        do_step(step, std::integral_constant<int, 0>{});
        last_buf = 0;
        if (step + 1 < n_steps) { do_step(step + 1, std::integral_constant<int, 1>{}); last_buf = 1; }
        if (kNBuf == 3 && step + 2 < n_steps) { do_step(step + 2, std::integral_constant<int, kNBuf - 1>{}); last_buf = 2; }
    }
    if (kDefer && pending) {
        if (last_buf == 0) second_tile_reduction(TileAt{0}, TileAt{kQTile});
        else if (last_buf == 1) second_tile_reduction(TileAt{2 * kQTile}, TileAt{3 * kQTile});
        else second_tile_reduction(TileAt{(kNBuf - 1) * 2 * kQTile}, TileAt{(kNBuf - 1) * 2 * kQTile + kQTile});
    }

    // ---- rows kb0.. of dK (scaled) and dV, through the wave's own tile as coalesced 16-byte stores
#pragma unroll
    for (int which = 0; which < 2; ++which) {
        const TensorArg& out = which == 0 ? p.dk : p.dv;
        const int64_t ob = slice_offset(out, job.seq, head, job.tok0);
        constexpr int kCols = D / kSplit;          // columns part * kCols .. of the rows
#pragma unroll
        for (int db = 0; db < kNB; ++db)
            stage_acc_tile<kCols>(ztile, 0, 32 * db, which == 0 ? dkacc[db] : dvacc[db], which == 0 ? p.scale : 1.0f, lane);
        for (int c = lane; c < 32 * kCols / 8; c += 64) {
            const int row = c / (kCols / 8), cc = c % (kCols / 8);
            if (kb0 + row < job.len)
                *(u32x4*)(out.ptr + 2 * (ob + (int64_t)(kb0 + row) * out.st + part * kCols + cc * 8)) = *(const u32x4*)(ztile + row * (kCols * 2) + cc * 16);
        }
    }
}


// ---------------------------------------------------------------- short sequences: the whole backward in one kernel
// A sequence of at most 32 * W tokens fits one workgroup of W waves: its queries (Q and dO) stay in LDS and, as row fragments, in
// registers, and its key blocks pass by from left to right as in the dQ pass.  Every score is evaluated ONCE: the step's
// weights and logit gradients go to LDS as 16-bit [query][64 keys] rows, and after a barrier the waves reduce them over all
// queries into the finished dK and dV rows of the key block (nobody else contributes to them).  Its weights for dK and dV are the
// dQ pass's, from Q scaled and rounded to 16 bits as in the forward (the own-keys and paired kernels round scaled K instead).  q, k, v, dO are read once
// where the two passes read them twice, no prefix table is written or read, and it is one launch.
// What bounds it is memory (seven tensors' bytes): two workgroups of four waves (80 KB of LDS) or four of two waves (sequences
// of at most 64 tokens) share a CU at head_dim 64, so that one's loads and stores run under the other's arithmetic; the next key
// block's K and V are requested into the tile just used.  On 65536 tokens in documents of 16 .. 128 (H=16, d=64) it takes 257 us and executes
// 800 vector and 410 scalar instructions a wave, 144 us of issue at the measured rates.  (When it took 268 us, its copies and stores alone
// took 200 and the whole of it, on rows that the caches held, 241.  Two documents in turn per workgroup, the next one's rows requested into registers meanwhile, are
// behind at every size: 64 registers and the second document's scalars spill, and the loads were not what was waited for.)
template <int D, int W>
__global__ __launch_bounds__(W * 64, D == 64 ? 2 : 1) void mfma_bwd_short_kernel(KParams p) {
    constexpr int kRows = W * 32;
    constexpr int kTile = 64 * kPitch<D> * 2;
    constexpr int kQ = 0, kDO = kRows * kPitch<D> * 2, kK = 2 * kDO, kV = kK + kTile, kA = kV + kTile, kZ = kA + kRows * 128;
    constexpr int kNB = D / 32;                // 32-column blocks of dK or dV that a wave reduces, for
    constexpr int kKH = W == 2 ? 2 : 1;        // one 32-key half of the block or both
    static_assert(W * kKH * kRowStage<D> <= 2 * kRows * 128, "the waves stage their outputs in the weight tiles");
    __shared__ __attribute__((aligned(1024))) char lds[kZ + kRows * 128];

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int n = lane & 31, h = lane >> 5;
    const int head = head_of_block(p, blockIdx.x);
    const Job job = decode_job(p, slot_of_block(p, blockIdx.x));
    if (blockIdx.x == 0 && threadIdx.x == 0 && p.gave_up) *p.gave_up = 0;
    LaneOffsets<D> lo;
    lo.init(lane);
    lo.rebase(lds);
    LaneOffsets<64> lz;
    lz.init(lane);
    lz.rebase(lds);
    const int strict = p.attend_current ? 0 : 1;
    const int q0w = 32 * wave, qi = q0w + n;
    const bool row_ok = qi < job.len;
    auto base_of = [&](const TensorArg& t) { return slice_offset(t, job.seq, head, job.tok0); };
    const int64_t qbase = base_of(p.q), kbase = base_of(p.k), vbase = base_of(p.v), dobase = base_of(p.d_o);

    // a tile is four waves' copies: two each where there are only two
    auto copy = [&](auto natural, const TensorArg& t, int64_t base, int row0, char* tile, bool fresh) {
#pragma unroll
        for (int w4 = 0; w4 < 4; w4 += W) {
            TileDma<D, decltype(natural)::value> c;
            c.init(lane, wave + w4, t, base, p.cols);
            if (fresh) c.clear(tile);
            c.issue(row0, job.len, tile);
        }
    };
    constexpr std::true_type kNaturalRows{};
    constexpr std::false_type kMfmaRows{};
    copy(kMfmaRows, p.k, kbase, 0, lds + kK, true);
    copy(kMfmaRows, p.v, vbase, 0, lds + kV, true);
    for (int r = 0; r < job.len; r += 64) {
        copy(kNaturalRows, p.q, qbase, r, lds + kQ + r * kPitch<D> * 2, true);
        copy(kNaturalRows, p.d_o, dobase, r, lds + kDO + r * kPitch<D> * 2, true);
    }
    // the carry that enters this lane's 32 keys of a block; 0 for rows past the end, whose weights are then exactly 0
    // (and for a block that holds nothing but the invisible last token: the forward has no entry for it)
    constexpr int kBlocks = W / 2;
    const int n_kb = (job.len + kKeyBlock - 1) / kKeyBlock;
    const float* rcur = (h ? p.rtab : p.rmid) + tab_index(p, head, job, 0, 0) + q0w + n;
    float F[kBlocks];
#pragma unroll
    for (int kb = 0; kb < kBlocks; ++kb) F[kb] = row_ok && 64 * kb + strict <= min(q0w + 31, job.len - 1) ? rcur[kb * kRowBlock] : 0.f;
    float dr = 0.f;
    if (row_ok && p.d_rem.ptr)
        dr = Elem16::load(p.d_rem.ptr, (int64_t)job.seq * p.d_rem.sb + (int64_t)head * p.d_rem.sh + job.tok0 + qi);
    wait_global_memory();
    __syncthreads();
    // row fragments from the tiles that the reduction needs anyway (as loads of their own they are 64 cache lines an instruction);
    // rows past the end repeat the last one, and their weights are zeros
    h16x8 qf[D / 16], dof[D / 16];
#pragma unroll
    for (int ks = 0; ks < D / 16; ++ks) {
        qf[ks] = *(const h16x8*)(lds + kQ + tile_offset<D>(qi, 2 * ks + h));
        dof[ks] = *(const h16x8*)(lds + kDO + tile_offset<D>(qi, 2 * ks + h));
    }
    prescale_frags(qf, p.scale2);

    f32x16 dqacc[D / 32];                      // (started by the first block, which every wave with rows sees)
    float Gc = 0.f;
    constexpr TileAt ktile{kK}, vtile{kV};
    const int which = W == 2 ? wave : wave >> 1, kh0 = W == 2 ? 0 : wave & 1;

#pragma unroll
    for (int kb = 0; kb < kBlocks; ++kb) {
        if (kb >= n_kb && kb > 0) break;
        const int key0 = kb * kKeyBlock;
        // a wave whose queries see nothing of the block has no rows in the reduction below, which starts at the block's first token
        if (q0w < job.len && key0 + strict <= q0w + 31) {
            float x[32], beta[32], dp[32];
            score_tiles_ps<D>(x, ktile, lo, qf);
            if (key0 + 63 + strict > q0w) mask_step(x, key0 + 32 * h, qi, strict);
            const float Lend = carried_weights_and_dp<D>(x, beta, dp, F[kb], vtile, lo, dof);
            if (kb == 0) {
                float Llo, Lup;
                half_values(Lend, Llo, Lup);
                Gc = dr * Llo;                 // what leaves the left half of the leftmost block is rem (see the dQ pass)
            }
#pragma unroll
            for (int c = 0; c < 4; ++c) *(h16x8*)(lds + kA + tile_offset<64>(qi, 4 * h + c)) = pack8(&x[8 * c]);
            logit_grads<false>(x, beta, dp, Gc, lane);
            h16x8 zf[4];
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                zf[c] = pack8(&dp[8 * c]);
                *(h16x8*)(lds + kZ + tile_offset<64>(qi, 4 * h + c)) = zf[c];
            }
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                h16x8 kt[D / 32];
#pragma unroll
                for (int db = 0; db < D / 32; ++db) kt[db] = fetch_cols_o<D>(ktile, lo, db, c);
#pragma unroll
                for (int db = 0; db < D / 32; ++db) dqacc[db] = mfma(kt[db], zf[c], kb == 0 && c == 0 ? f32x16{0} : dqacc[db]);
            }
        } else if (kb == 0) {
#pragma unroll
            for (int db = 0; db < D / 32; ++db) dqacc[db] = f32x16{0};
        }
        __syncthreads();                       // weights complete, K and V free
        if (kb + 1 < n_kb) {
            copy(kMfmaRows, p.k, kbase, key0 + kKeyBlock, lds + kK, false);
            copy(kMfmaRows, p.v, vbase, key0 + kKeyBlock, lds + kV, false);
        }
        // [32 keys x D] of dV (which = 0) or dK: keys 32 kh .. of the block, over the queries from the block on; transposed tiles
        // (lane = key), which leave as rows the way dQ does
        f32x16 acc[kKH][kNB];
        {
            const int offw = which ? kZ : kA, offb = which ? kQ : kDO;
            auto fetch = [&](int x0, int x1, int add) {
                union { s16x4 v[2]; h16x8 b; } u;
                u.v[0] = lds_read_tr_at((uint32_t)(x0 + add), 0);
                u.v[1] = lds_read_tr_at((uint32_t)(x1 + add), 0);
                return u.b;
            };
            // 32 queries at a time, all their operands requested before the first product (a wave writes whole 32-row tiles of
            // weights, zeros past the end); the first ones start the sums
            auto reduce = [&](int r, auto first) {
                h16x8 w[2][kKH], b[2][kNB];
#pragma unroll
                for (int half = 0; half < 2; ++half) {
#pragma unroll
                    for (int i = 0; i < kKH; ++i)
                        w[half][i] = fetch(kh0 + i ? lz.nat[0][1] : lz.nat[0][0], kh0 + i ? lz.nat[1][1] : lz.nat[1][0], offw + (r + 16 * half) * 128);
#pragma unroll
                    for (int db = 0; db < kNB; ++db) b[half][db] = fetch(lo.nat[0][db], lo.nat[1][db], offb + (r + 16 * half) * kPitch<D> * 2);
                }
#pragma unroll
                for (int half = 0; half < 2; ++half)
#pragma unroll
                    for (int db = 0; db < kNB; ++db)
#pragma unroll
                        for (int i = 0; i < kKH; ++i)
                            acc[i][db] = mfma(b[half][db], w[half][i], decltype(first)::value && half == 0 ? f32x16{0} : acc[i][db]);
            };
            reduce(key0, std::true_type{});
            for (int r = key0 + 32; r < job.len; r += 32) reduce(r, std::false_type{});
        }
        if (which) {
#pragma unroll
            for (int i = 0; i < kKH; ++i)
#pragma unroll
                for (int db = 0; db < kNB; ++db)
#pragma unroll
                    for (int e = 0; e < 16; ++e) acc[i][db][e] *= p.scale;
        }
        __syncthreads();                       // weight tiles free
        {
            const TensorArg& out = which ? p.dk : p.dv;
#pragma unroll
            for (int i = 0; i < kKH; ++i)
                store_query_rows<D>(lds + kA + (wave * kKH + i) * kRowStage<D>, acc[i], 1.0f, out, base_of(out), key0 + 32 * (kh0 + i),
                                    job.len, lane, p.cols);
        }
        if (kb + 1 < n_kb) {
            wait_global_memory();              // the next K and V have landed
            __syncthreads();
        }
    }

    // (the wave's own Q rows: nobody reads them any more)
    store_query_rows<D>(lds + kQ + q0w * kPitch<D> * 2, dqacc, p.scale, p.dq, base_of(p.dq), q0w, job.len, lane, p.cols);
}

// ---------------------------------------------------------------- pass 2, two waves per 32 keys
// What a wave of the own-keys kernel holds for its 32 keys at head_dim 128 - K and V fragments and the
// [32 keys x 128] accumulators of dK and dV - is 190 registers: one wave per SIMD.  Here TWO waves share
// 32 keys.  Both hold the K and V fragments; wave r of the pair turns query tile r of the step (32 of
// its 64 queries) into weights and logit gradients and writes them to the pair's tile in LDS; after a
// barrier wave 0 reduces the weights of ALL 64 queries with dO into dV, wave 1 the logit gradients with Q into
// dK, so each accumulates [32 keys x D] of one output.  (A split of both outputs' columns fetches both kinds of
// weights in both waves - six operands a 16 queries instead of five - and leaves head_dim 96 with two column blocks in one wave and
// one in the other: 12 heads, 20011 tokens, d = 80 222 -> 213 us.)  Two workgroup barriers per step (weights complete; tiles handed over).
// What bounds it is instruction issue (MFMA and vector instructions keep a SIMD busy 84 to 94 % of the time in which its CU has
// work) and the waits of waves that run in step.  kPairs = 2: a workgroup is 64 keys, four waves and exactly half of a CU's LDS, so
// that two of them share a CU and one's barriers and round trips pass under the other's work, and the diagonal and the end of a
// sequence are cut off by 64 keys.  Against one workgroup of kPairs = 4 a CU (128 keys, eight waves, half the tile copies):
// B=4 H=16 T=2047 d=128 181 -> 163 us, B=1 H=16 T=16384 1690 -> 1530, d = 80 as above 249 -> 213.
// At head_dim 64 a wave holds one output's [32 keys x 64] and needs 165 registers, three waves to a SIMD, and a workgroup 48 KB of LDS, three to a
// CU.  A sweep's step is two tiles in a row there in the own-keys kernel, one in each wave here, which the longest sweeps of a launch gain most from
// (H=16 T=4096: 97 us, the resident stream 114).  With three workgroups to fill each other's gaps the pacing of a workgroup's own waves costs more than
// it gives: without it T=4096 109 -> 97 us, 65536 packed tokens 746 -> 732; at head dims 96 and 128 it makes no difference.
// kScaledQ (head_dim 64): which operand of the scores is scaled and rounded.  Without it K, in registers; with it the tiles are the scaled copy of q that the
// dQ pass leaves behind, for the scores and for dK, as in the stream: the weights are those behind the forward's carries, but q is rounded twice where dK is formed.
// Errors of dK / dV against 64 bits (2-norms, 1e-3, bf16, H=4 T=2048), K and scaled q, the latter the stream's to four digits:  all heads' mean logits at -6
// 2.93 / 2.92 and 3.08 / 2.65, logits of standard deviation 3 3.41 / 2.62 and 3.79 / 2.63, mean logits 0 .. -6 over the heads 2.44 / 2.42 and 2.90 / 2.41.
template <int D, int kPairs, bool kScaledQ, Sharing kSharing, class Draw>
__device__ __forceinline__ void paired_keys_job(const KParams& p, const int block, const int wave, const int lane, Draw draw, char* const lds) {
    constexpr int kQTile = 64 * kPitch<D> * 2;           // Q or dO tile of one step (64 queries)
    constexpr int kZTile = 64 * 64 * 2;          // per pair: [64 queries][32 a | 32 dz] bf16
    constexpr int kStep = 64;
    constexpr int kBlocks = D / 32;              // 32-wide column blocks of dK or dV
    constexpr bool kPaced = D != 64;
    static_assert(2 * kPairs * 32 * D * 2 <= 4 * kQTile, "every wave stages its [32 keys x D] output in the tiles");

    const int grp = wave >> 1, r = wave & 1;
    const int n = lane & 31, h = lane >> 5;
    LaneOffsets<D> lo;
    lo.init(lane);
    LaneOffsets<64> lz;
    lz.init(lane);
    constexpr int kParts = 4 / kPairs;                 // workgroups of a scheduled 128-row job
    const int slot = slot_of_block(p, block);
    const int head = head_of_block<kSharing>(p, block);
    const Job job = decode_key_job(p, slot / kParts);
    const int strict = p.attend_current ? 0 : 1;
    const int first_kb = 2 * job.rb + slot % kParts;   // first 64-key block of the workgroup's keys
    const int q_begin = first_kb * kKeyBlock;          // first key = first query that may see it
    if (q_begin >= job.len) {
        draw();
        return;
    }
    const int kb0 = q_begin + 32 * grp;                // first key of this pair
    char* ztile = lds + 4 * kQTile + grp * kZTile;

    const TensorArg& q = kScaledQ ? p.q_scaled : p.q;
    const int64_t qbase = slice_offset(q, job.seq, head, job.tok0);
    const int64_t kbase = slice_offset(p.k, job.seq, head, job.tok0);
    const int64_t vbase = slice_offset(p.v, job.seq, head, job.tok0);
    const int64_t dobase = slice_offset(p.d_o, job.seq, head, job.tok0);

    // A operands of the score tile: MFMA row m holds key 16*((m>>2)&1) + 4*(m>>3) + (m&3) of the pair,
    // so that the accumulator registers of a lane are 16 consecutive keys (as in the own-keys kernel)
    h16x8 kfr[D / 16], vfr[D / 16];
    {
        const int m = lane & 31;
        const int key = 16 * ((m >> 2) & 1) + 4 * (m >> 3) + (m & 3);
        load_row_frags<D>(kfr, p.k, kbase, kb0, key, job.len, lane, p.cols);
        load_row_frags<D>(vfr, p.v, vbase, kb0, key, job.len, lane, p.cols);
        if (!kScaledQ) prescale_frags(kfr, p.scale2);
    }
    f32x16 acc[kBlocks];         // r = 0: dV, r = 1: dK
#pragma unroll
    for (int j = 0; j < kBlocks; ++j) acc[j] = f32x16{0};

    const int n_steps = min((job.len - q_begin + kStep - 1) / kStep, 2 * (last_live_row_block(p, head, job) + 1) - first_kb);

    // copies of a step's Q and dO tiles: with eight waves the first four take Q and the others dO, four waves take both
    const bool q_first = kPairs == 2 || wave < 4;
    TileDma<D, true> tc, tc2;
    tc.init(lane, wave & 3, q_first ? q : p.d_o, q_first ? qbase : dobase, p.cols);
    if (kPairs == 2) tc2.init(lane, wave, p.d_o, dobase, p.cols);
    const int my_tile = q_first ? 0 : kQTile;
#pragma unroll
    for (int b = 0; b < 2; ++b) {
        tc.clear(lds + b * 2 * kQTile + my_tile);
        if (kPairs == 2) tc2.clear(lds + b * 2 * kQTile + kQTile);
    }
    auto issue_tiles = [&](int row0, char* tiles) __attribute__((always_inline)) {
        tc.issue(row0, job.len, tiles + my_tile);
        if (kPairs == 2) tc2.issue(row0, job.len, tiles + kQTile);
    };
    if (n_steps > 0) issue_tiles(q_begin, lds);

    // carries of a (query, this pair's 32 keys) pair, see the own-keys kernel
    const int kb64 = kb0 / kKeyBlock;
    const float* rsrc = ((grp & 1) ? p.rtab : p.rmid) + tab_index(p, head, job, 0, kb64);
    const float* gsrc = ((grp & 1) ? p.gmid : p.gtab) + tab_index(p, head, job, 0, kb64);
    float Rn = 1.f, Gn = 0.f;
    // A step's 64 queries lie inside one 128-row block: the table index is a uniform base plus the lane's
    // row.  Rows past the end of the sequence are read too (the tables are allocated in whole row blocks)
    // and not used.
    const int my_row = 32 * r + n;
    auto request_carries = [&](int q0) __attribute__((always_inline)) {
        const int qb = q0 >> 7;
        const int64_t ix = (int64_t)qb * (qb + 1) * kRowBlock + (q0 & (kRowBlock - 1));      // uniform
        Rn = rsrc[ix + my_row];
        Gn = gsrc[ix + my_row];
    };
    if (n_steps > 0) request_carries(q_begin);
    wait_global_memory();
    __syncthreads();

    // Every LDS address of the loop is "a register that is fixed for the whole sweep + a constant": the sums of
    // LDS base, lane offset and this wave's share (query tile r, the Q or the dO tiles, the pair's weight tile) are
    // made once, and the loop runs in two copies, one per tile buffer, so that buffer and row offsets are compile-time
    // numbers that go into the offset fields of the fetches.  (With the tile address in a scalar register each
    // fetch costs one or two vector adds with a scalar operand, 1.8 ns each: 40 of them per step.)
    uint32_t row_at[D / 16], nat_at[2][kBlocks], z_at[2];
#pragma unroll
    for (int ks = 0; ks < D / 16; ++ks) row_at[ks] = lds_lane_base(lds + r * 32 * kPitch<D> * 2, lo.rows[ks]);
#pragma unroll
    for (int a2 = 0; a2 < 2; ++a2) {
#pragma unroll
        for (int j = 0; j < kBlocks; ++j) nat_at[a2][j] = lds_lane_base(lds + (r ? 0 : kQTile), lo.nat[a2][j]);
        z_at[a2] = lds_lane_base(ztile, r ? lz.nat[a2][1] : lz.nat[a2][0]);
    }
    auto rows_at = [&](uint32_t base, int imm) __attribute__((always_inline)) {
        return *(const __attribute__((address_space(3))) h16x8*)((__attribute__((address_space(3))) char*)(uintptr_t)base + imm);
    };
    auto transposed = [&](uint32_t at0, uint32_t at1, int imm) __attribute__((always_inline)) {
        union { s16x4 v[2]; h16x8 b; } u;
        u.v[0] = lds_read_tr_at(at0, imm);
        u.v[1] = lds_read_tr_at(at1, imm);
        return u.b;
    };

    auto do_step = [&](int step, auto buf_c) __attribute__((always_inline)) {
        constexpr int buf = decltype(buf_c)::value;
        constexpr int kQ = buf * 2 * kQTile;             // byte offsets of this step's Q and dO tiles
        constexpr int kDO = kQ + kQTile;
        const int q0 = q_begin + step * kStep;
        const float Rin = Rn, Gin = Gn;
        // the score operands are requested first: their LDS round trip passes under the scalar work of the tile requests
        h16x8 bq[D / 16];
#pragma unroll
        for (int ks = 0; ks < D / 16; ++ks) bq[ks] = rows_at(row_at[ks], kQ);
        __builtin_amdgcn_sched_barrier(0);
        if (step + 1 < n_steps) {     // next tiles, straight into the other buffer (nobody reads it since the last barrier)
            issue_tiles(q0 + kStep, lds + (buf ^ 1) * 2 * kQTile);
            request_carries(q0 + kStep);
        }
        __builtin_amdgcn_sched_barrier(0);
        // whole step left of this pair's first key: nothing visible (the same for both waves of the pair)
        const bool skip = kb0 + strict > q0 + kStep - 1 || kb0 >= job.len;
        if (!skip) {
            const int qt0 = q0 + 32 * r;
            const int qi = qt0 + n;
            if (kb0 + strict > qt0 + 31) {             // this wave's query tile sees none of the keys (the other one does)
                const h16x8 none = {0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
                for (int c = 0; c < 4; ++c) *(h16x8*)(ztile + tile_offset<64>(32 * r + n, 2 * c + h)) = none;
            } else {
                float x[16], dp[16];
                const int nvis = qi < job.len ? qi - strict - (kb0 + 16 * h) + 1 : 0;
                const bool sees = qi < job.len && qi - strict - kb0 + 1 > 0;
                const float Rt = sees ? Rin : 1.0f;      // table entries of invisible pairs are not written
                const float Gt = sees ? Gin : 0.0f;
                float beta[16];
                if (kPaced) __builtin_amdgcn_s_setprio(3);     // paced like the two-step dQ kernel's chain: the wave behind goes first
                {
                    f32x16 sacc = {0};
#pragma unroll
                    for (int ks = 0; ks < D / 16; ++ks) sacc = mfma(kfr[ks], bq[ks], sacc);
#pragma unroll
                    for (int i = 0; i < 16; ++i) x[i] = sacc[i];
                }
                if (kb0 + 31 + strict > qt0 || qt0 + 31 >= job.len) {     // diagonal or ragged tile
#pragma unroll
                    for (int idx = 0; idx < 16; ++idx)
                        if (idx >= nvis) x[idx] = -INFINITY;
                }
                // dP = dO V^T between the segments of the chain, its operands fetched one segment ahead
                constexpr int kPer = (D / 16 + 3) / 4;
                h16x8 nx[kPer];
#pragma unroll
                for (int i = 0; i < kPer; ++i) nx[i] = rows_at(row_at[i], kDO);
                f32x16 dacc;
                own_tile_weights(x, beta, Rt, lane, [&](int seg) {
                    h16x8 cur[kPer];
#pragma unroll
                    for (int i = 0; i < kPer; ++i) cur[i] = nx[i];
                    if (seg < 3) {
#pragma unroll
                        for (int i = 0; i < kPer; ++i)
                            if (kPer * (seg + 1) + i < D / 16) nx[i] = rows_at(row_at[kPer * (seg + 1) + i], kDO);
                    }
#pragma unroll
                    for (int i = 0; i < kPer; ++i) {
                        const int ks = kPer * seg + i;
                        if (ks < D / 16) dacc = mfma(vfr[ks], cur[i], ks == 0 ? f32x16{0} : dacc);
                    }
                    if (kPaced && seg == 1) __builtin_amdgcn_s_setprio(2);
                });
                if (kPaced) __builtin_amdgcn_s_setprio(1);
#pragma unroll
                for (int i = 0; i < 16; ++i) dp[i] = dacc[i];
                // a -> columns 16h.. of row (32r + n) now, dz -> columns 32 + 16h.. below
                *(h16x8*)(ztile + tile_offset<64>(32 * r + n, 2 * h)) = pack8(&x[0]);
                *(h16x8*)(ztile + tile_offset<64>(32 * r + n, 2 * h + 1)) = pack8(&x[8]);
                own_tile_grads(x, beta, dp, Gt, lane);
                *(h16x8*)(ztile + tile_offset<64>(32 * r + n, 4 + 2 * h)) = pack8(&dp[0]);
                *(h16x8*)(ztile + tile_offset<64>(32 * r + n, 4 + 2 * h + 1)) = pack8(&dp[8]);
                if (kPaced) __builtin_amdgcn_s_setprio(0);
            }
        }
        __syncthreads();                       // the pair's weights are complete
        if (!skip) {
            // dV += A^T dO (r = 0) or dK += dZ^T Q (r = 1) over the step's 64 queries.  The operands of 16 queries are
            // requested while the MFMAs of the 16 before them run (left to itself the compiler requests them right before
            // their MFMA, which then waits for the LDS round trip).
            h16x8 w[2], o[2][kBlocks];
            auto fetch_kk = [&](int kk, h16x8& ww, h16x8 (&oo)[kBlocks]) __attribute__((always_inline)) {
                ww = transposed(z_at[0], z_at[1], 16 * kk * 64 * 2);
#pragma unroll
                for (int j = 0; j < kBlocks; ++j) oo[j] = transposed(nat_at[0][j], nat_at[1][j], kQ + 16 * kk * kPitch<D> * 2);
            };
            fetch_kk(0, w[0], o[0]);
#pragma unroll
            for (int kk = 0; kk < 4; ++kk) {
                if (kk < 3) fetch_kk(kk + 1, w[(kk + 1) & 1], o[(kk + 1) & 1]);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int j = 0; j < kBlocks; ++j) acc[j] = mfma(w[kk & 1], o[kk & 1][j], acc[j]);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        wait_global_memory();                  // the next tiles and carries have landed
        __syncthreads();                       // ... and everybody is through with this step's tiles
    };
    for (int step = 0; step < n_steps; step += 2) {
        do_step(step, std::integral_constant<int, 0>{});
        if (step + 1 < n_steps) do_step(step + 1, std::integral_constant<int, 1>{});
    }

    draw();
    // ---- this wave's output, rows kb0.. of dV or of dK (scaled), staged in its share of the tiles and stored as coalesced
    // 16-byte chunks
    const TensorArg& out = r ? p.dk : p.dv;
    const int64_t ob = slice_offset(out, job.seq, head, job.tok0);
    char* const stage = lds + wave * (32 * D * 2);
    const float dk_scale = kScaledQ ? p.scale / p.scale2 : p.scale;
#pragma unroll
    for (int j = 0; j < kBlocks; ++j) stage_acc_tile<D>(stage, 0, 32 * j, acc[j], r ? dk_scale : 1.0f, lane);
    for (int c = lane; c < 32 * D / 8; c += 64) {
        const int row = c / (D / 8), cc = c % (D / 8);
        if (kb0 + row < job.len && (D != 96 || cc * 8 < p.cols))
            *(u32x4*)(out.ptr + 2 * (ob + (int64_t)(kb0 + row) * out.st + cc * 8)) = *(const u32x4*)(stage + row * (D * 2) + cc * 16);
    }
}

template <int D, int kPairs, bool kScaledQ = false>
__global__ __launch_bounds__(128 * kPairs, D == 64 ? 3 : 2) void mfma_bwd_dkv_pair_kernel(KParams p) {
    constexpr int kQTile = 64 * kPitch<D> * 2, kZTile = 64 * 64 * 2;
    __shared__ __attribute__((aligned(16))) char lds[4 * kQTile + kPairs * kZTile];   // (Q, dO) x 2 buffers | one Z tile per pair
    paired_keys_job<D, kPairs, kScaledQ, kPairs == 4 ? kOnePerCu : kSharedCu>(p, blockIdx.x, __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), threadIdx.x & 63, [] {}, lds);
}

template <int D>
__global__ __launch_bounds__(256, D == 64 ? 3 : 2) void mfma_bwd_dkv_pair_drawing_kernel(KParams) {
    constexpr int kQTile = 64 * kPitch<D> * 2, kZTile = 64 * 64 * 2;
    __shared__ __attribute__((aligned(16))) char lds[4 * kQTile + 2 * kZTile];   // (Q, dO) x 2 buffers | one Z tile per pair
    draw_jobs((int*)(lds + 4 * kQTile), [&](const KParams& p, int block, int wave, int lane, auto draw) { paired_keys_job<D, 2, false, kDrawn>(p, block, wave, lane, draw, lds); });
}

}  // inline namespace SBA_ELEM_NS
}  // namespace sba

#ifndef SBA_ELEM_F16
bool sba_mfma_bwd_available() { return true; }
#endif

// SBA_DKV_KERNEL overrides the choice between the key-owner kernels (tests run them on the same inputs).  =pair, =other, =plain and =stream8 are explained where
// the choice is made; =own is the own-keys kernel at head_dim 128 and the paired one at 64 to 96, =pair4 has four pairs from 72 on and two at 64.
static bool own_keys_kernel(const char* e, bool by_size) {
    if (e && (!strcmp(e, "own") || !strncmp(e, "pair", 4))) return true;
    if (e && !strcmp(e, "other")) return false;
    return by_size;
}

// Whether the paired kernel at head_dim 64 takes the dQ pass's scaled copy of q (kScaledQ): for launches that hang on their longest sweeps, which the stream had
// before it and still has where they are small, so that neither gradient is further off for the change of kernel.  The others round K, as the kernel did that
// they had before.  (For them the copy would be a write of q in the dQ pass and a larger error of dK: forward + backward of packs of 65536 tokens 1.007 / 1.024 / 1.009,
// B=4 T=8192 1.006 / 1.013 / 1.004 of the time, T=4096 0.997 / 0.998 / 1.003: the heads' mean logits 0 .. -6 in order / in a random one / all at -6.)
// SBA_DKV_KERNEL=pairq / =pair picks one.
static bool paired_scaled_q(const char* e, const sba::KParams& kp, unsigned grid) {
    if (e && (!strcmp(e, "own") || !strncmp(e, "pair", 4))) return !strcmp(e, "pairq");
    if (kp.seq_len <= 8 * sba::kRowBlock && grid >= 2u * (unsigned)sba_cu_count()) return false;
    return sba_tail_ratio(kp, grid) > (kp.seq_len <= 32 * sba::kRowBlock ? 3.35 : kp.n_heads <= 8 && !kp.cu_seqlens ? 2.2 : 2.75);
}

// SBA_DQ_KERNEL=lean / =plain overrides the choice between the two arrangements of the one-step dQ kernel at
// head_dim 64 (tests run both on the same inputs).
static bool lean_dq_kernel(bool by_size) {
    const char* e = getenv("SBA_DQ_KERNEL");
    if (e && !strcmp(e, "lean")) return true;
    if (e && !strcmp(e, "plain")) return false;
    return by_size;
}

#ifdef SBA_ELEM_F16
int sba_launch_mfma_f16_bwd(const sba::KParams& kp_in, int phases, hipStream_t s) {
#else
int sba_launch_mfma_bwd(const sba::KParams& kp_in, int phases, hipStream_t s) {
#endif
    using namespace sba;
    KParams kp = kp_in;
    dim3 grid((unsigned)kp.n_jobs * kp.n_heads);
    const bool p1 = phases != 2, p2 = phases != 1;
    kp.queue_stride = sba_queue_stride(kp);
    // the dQ kernels reach a lane's prefix entry from its carry entry by one uniform distance (see there)
    if (!kp.rtab || !kp.rmid || !kp.gtab || !kp.gmid) return SBA_ERR_WORKSPACE;
    if (!kp.makes_mid && (const char*)kp.gmid - (const char*)kp.rtab != (const char*)kp.gtab - (const char*)kp.rmid) return SBA_ERR_WORKSPACE;
    // Key-owner pass.  head_dim 64: the paired kernel, but for fewer than one and a half row blocks a CU (all heads), where three workgroups a CU do not
    // come together, and for launches that hang on few long sweeps, whose steps are longer in it; there the resident producer/consumer stream is ahead.  Forward +
    // backward with the paired kernel (scaled q) over the same with the stream, by workgroups of the row-owner passes and tail ratio, mean logits 0 .. -6
    // over the heads in order / in a random one / all at -6:
    //     fewer than 384 (K rounded)  192 (H=16 T=1500) 1.11 / 1.08 / 1.085    256 (H=16 T=2048) 1.07 / 1.07 / 1.08, (H=4 T=8192) 1.15 / 1.16 / 1.15    320 (H=16 T=2500) 1.02 /
    //         1.015 / 1.01, (H=8 T=5000) 1.05 / 1.05 / 1.05, packs of 2000 tokens 1.02 / 1.02 / 1.02    376 (H=8 T=6000) 1.04 / 1.02 / 1.03
    //     longest sequence up to 4096 tokens  384 (H=12 T=4096, 5.2) 0.99 / 0.99 / 0.99, (H=16 T=3072, 5.1) 0.98 / 0.975 / 1.00, (B=6 H=4 T=2048, 5.0) 0.95 / 0.96 / 0.96    408 (H=24 T=2176,
    //         4.7) 0.97 / 0.97 / 0.97    512 (H=16 T=4096, 3.9) 0.955 / 0.95 / 0.96, (B=4 H=4 T=4096) 0.93 / 0.94 / 0.97, (B=16 H=2 T=2048, 3.8) 0.96 / 0.96 / 0.97, (H=32 T=2048) 0.94 / 0.95 /
    //         0.95;  packs  4096 + 2048 H=8 (384, 6.2) 1.02 / 1.02 / 1.03, 4096 to 400 H=4 (500, 5.7) 1.02 / 1.01 / 1.02, 4096 to 1000 H=8 (544, 5.3) 0.98 / 0.97 / 0.98, 2048 to 400
    //         H=16 (512, 5.3) 0.94 / 0.96 / 0.965;  one document among short ones  4096 and 100s H=4 (528, 13) 1.04 / 1.05 / 1.05, 4096 and 300s H=2 (664, 14.5) 1.03, H=4 (848, 9.2) 0.98,
    //         4096 and 200s H=8 (896, 6.3) 1.01, 3500 and 300s H=8 (944, 6.1) 0.98, 3000 and 128s H=8 (512, 9.0) 1.05, 2500 and 128s H=8 (480, 10.2) 1.07, 2048 and 100s (424, 18) 1.04, (448,
    //         11.6) 1.045, 2048 and 300s H=4 (784, 8.3) 0.88, 2048 and 256s H=8 (928, 7.2) 0.91, 2048 and 128s H=16 (896, 5.8) 0.93, 4096 and 128s H=16 (1472, 3.5) 0.89 / 0.89 / 0.90
    //     longer  384 (H=4 T=12288, 5.3) 1.06 / 1.06 / 1.04, (H=8 T=6144) 1.03 / 1.01 / 1.03, (H=6 T=8192) 1.015 / 1.00 / 1.03, (B=2 H=2 T=12288) 1.00 / 1.00 / 1.02    440 (H=4 T=14000, 4.6) 1.045 / 1.045 /
    //         1.03    480 (H=12 T=5120, 4.2) 0.97 / 0.975 / 0.98    512 (3.9 to 4.0) (H=4 T=16384) 1.03 / 1.03 / 1.00, (H=2 T=32768) 0.94 / 0.94 / 1.01, heads at 0 and -6 1.07 / 1.08 / 0.99,
    //         (H=8 T=8192) 0.96 / 0.96 / 0.98, (B=2 H=2 T=16384) 0.94 / 0.94 / 1.01, (B=2 H=4 T=8192) 0.94 / 0.945 / 0.99    628 (H=4 T=20000, 3.2) 0.97 / 0.97 / 1.02    640 (H=16 T=5000, 3.1)
    //         0.935 / 0.91 / 1.00    784 (H=4 T=25000, 2.6) 0.95 / 0.95 / 1.00, (B=2 H=2 T=25000) 0.83 / 0.83 / 0.98;  packs  8192 + 4096 + 2048 H=4 (448, 6.0) 1.04 / 1.05 / 1.05, 16384 + 8192
    //         H=2 (384, 6.3) 1.11 / 1.11 / 1.07, 11000 and short ones H=4 (436, 5.8) 1.04 / 1.05 / 1.05, 6000 and 300s H=4 (908, 8.1) 1.04, 8192 and 512s H=8 (1152, 3.6) 0.89 / 0.925 / 0.95
    // and over the kernel whose waves own 32 keys each (two waves per SIMD at 215 registers), which was there before for launches that do not hang on their longest
    // sweeps: 1024 (H=32 T=4096) 0.95 / 0.94 / 0.935, (H=16 T=8192) 0.96 / 0.94 / 0.93, (B=8 T=2048) 0.935 / 0.94 / 0.98, (B=4 T=1024) 0.97 / 0.95 / 0.97,
    // packs of 8192 tokens 0.95 / 0.93 / 0.93, 16384 0.93 / 0.95 / 0.93, 65536 0.98 / 0.97 / 0.98, documents up to 1024 0.96 / 0.96 / 0.95, up to 256 0.98 / 0.975 / 0.97.
    // head_dim 72 to 128: the paired kernel at every size (B=1, H=16, T=512 ... 2048: with four pairs 27 / 44 / 62 / 81 us where the
    // kernel with one workgroup per 64-key block takes 33 / 55 / 73 / 103).  SBA_DKV_KERNEL=pair / =pairq (see paired_scaled_q()) / =other (the stream at
    // head_dim 64) picks one.
    const char* which = getenv("SBA_DKV_KERNEL");
    const unsigned cus = (unsigned)sba_cu_count();
    const bool scaled_q = kp.head_dim == 64 && paired_scaled_q(which, kp, grid.x);
    const double paired_up_to = kp.seq_len > 32 * kRowBlock ? (kp.n_heads <= 4 && kp.n_seq == 1 ? 3.5 : 4.5) : grid.x >= 3 * cus ? 9.5 : 5.5;
    const bool own = own_keys_kernel(which, kp.head_dim == 64 ? 2 * grid.x >= 3 * cus && (!scaled_q || sba_tail_ratio(kp, grid.x) <= paired_up_to) : true);
    const bool plain = which && !strcmp(which, "plain");
    // the stream with eight half-block producers (12 waves): behind the one with four full-block producers
    // (107 against 99.5 us at B=1 H=16 T=4096), which stays the default
    const bool stream8 = which && !strcmp(which, "stream8");
    // the scaled copy of q is for the stream and for the paired kernel in its place: nobody else reads it, so the dQ pass skips it
    const bool stream = kp.head_dim == 64 && !plain && !own;
    // Paired kernel: workgroups of two pairs, two a CU, but for launches of short sweeps that do not fill the chip with them, where the
    // prologue counts.  Forward + backward with two pairs over the same with four, d=128 / 96:  T=300 B=16 1.04 / 1.03,
    // T=512 B=2 1.06 / 1.00, B=4 1.04 / 0.99, B=8 (512 row blocks) 1.05 / 1.05, B=16 (1024) 1.00 / 1.00;  T=640 B=4 1.00 / 0.98;
    // T=768 B=2 0.93 / 0.945;  T=1024 B=1 0.88, B=2 0.95 / 0.95, B=8 0.98 / 1.00;  T=4096 0.97;  packs of documents of at most 512 tokens 0.95
    // (65536 tokens), 256 0.98 (16384).
    const bool four_pairs = which && !strncmp(which, "pair", 4) ? !strcmp(which, "pair4") : kp.seq_len <= 4 * kRowBlock && grid.x < 4u * cus;
    const bool needs_scaled_q = stream || (own && scaled_q);
    if (needs_scaled_q && !kp.q_scaled.ptr) return SBA_ERR_WORKSPACE;
    if (!needs_scaled_q) kp.q_scaled.ptr = nullptr;
    // Sequences of at most 128 tokens: one kernel for both passes (it all runs in phase 1).  A kernel asked for by name is one of
    // the two-pass ones.
    if (kp.seq_len <= kRowBlock && kp.head_dim <= 128 && !which && !getenv("SBA_DQ_KERNEL") && sba_two_step_env() < 0) {
        if (!p1) return SBA_OK;
        if (kp.head_dim == 96) {
            hipLaunchKernelGGL((mfma_bwd_short_kernel<96, 4>), grid, dim3(256), 0, s, kp);
        } else if (kp.head_dim == 128) {
            hipLaunchKernelGGL((mfma_bwd_short_kernel<128, 4>), grid, dim3(256), 0, s, kp);
        } else {
            if (kp.seq_len <= 64) hipLaunchKernelGGL((mfma_bwd_short_kernel<64, 2>), grid, dim3(128), 0, s, kp);
            else hipLaunchKernelGGL((mfma_bwd_short_kernel<64, 4>), grid, dim3(256), 0, s, kp);
        }
        return hipGetLastError() == hipSuccess ? SBA_OK : SBA_ERR_LAUNCH;
    }
    if (kp.head_dim == 64) {
        // Small grids that last as long as their longest sweep (tail ratio from 3.7: B=1, H=16 up to T=4096) take the
        // variant that halves it; batches of short sequences on the same number of workgroups do not (B=8, T=512:
        // 23.8 us with one step per iteration against 27.4, B=4, T=1024 36.0 against 37.7).
        const bool two_steps = sba_two_step_env() >= 0 ? grid.x <= (unsigned)sba_two_step_env()
                                                       : grid.x <= kTwoStepDqMaxGrid && sba_tail_ratio(kp, grid.x) >= 3.7;
        if (p1 && kp.makes_mid) sba_launch_drawing((mfma_bwd_dq_kernel<64, true, true>), (mfma_bwd_dq_drawing_kernel<64, true, true>), grid.x, kThreads, 3, sba_turning(kp, 3), kp.gtab, kDqQueue, false, s);
        else if (p1 && two_steps) hipLaunchKernelGGL((mfma_bwd_dq2_kernel<64>), grid, dim3(2 * kThreads), 0, s, kp);
        // The register-lean arrangement (three waves per SIMD) from five workgroups per CU on, unless the launch hangs on
        // one long sweep (tail ratio above 2.5: there the plain arrangement's shorter step is ahead, e.g. 111 against 118 us
        // on an 8192-token pack with a 4096-token document); from eight workgroups per CU on always.  On 1280-3232
        // workgroups of 15 dense shapes it takes 0.98-1.00 of the plain one's forward + backward where all heads look far and 0.98-1.02 where
        // they differ, but for single sequences of 10000 tokens and more (1.00-1.07: B=1 H=12 T=16384 1690 against 1580 us, H=16 T=10240 898
        // and 865; from T=14000 on 0.99-1.02); on packs 0.96-1.00.  At four workgroups per CU (six shapes of 1024 workgroups) the
        // plain one is ahead by 1-3 %.
        else if (p1 && lean_dq_kernel(grid.x >= 8u * cus || (grid.x >= 5u * cus && sba_tail_ratio(kp, grid.x) <= 2.5)))
            sba_launch_drawing((mfma_bwd_dq_kernel<64, true>), (mfma_bwd_dq_drawing_kernel<64, true, false>), grid.x, kThreads, 3, sba_turning(kp, 3), kp.gtab, kDqQueue, false, s);
        else if (p1) hipLaunchKernelGGL((mfma_bwd_dq_kernel<64>), grid, dim3(kThreads), 0, s, sba_turning(kp, 2));
        if (p2 && plain) {
            hipLaunchKernelGGL((mfma_bwd_dkv_kernel<64>), dim3(2 * grid.x), dim3(kThreads), 0, s, kp);
        } else if (p2 && own && scaled_q) {        // (has no drawing form: a launch that hangs on its longest sweeps has not the work that pays)
            hipLaunchKernelGGL((mfma_bwd_dkv_pair_kernel<64, 2, true>), dim3(2 * grid.x), dim3(256), 0, s, kp);
        } else if (p2 && own) {
            sba_launch_drawing((mfma_bwd_dkv_pair_kernel<64, 2>), (mfma_bwd_dkv_pair_drawing_kernel<64>), 2 * grid.x, kThreads, 3, kp, kp.gtab, kKeyQueue, p1, s);
        } else if (p2) {
            // one resident workgroup per CU, in whole rounds of the 8 XCDs (surplus workgroups
            // find no item)
            const unsigned n_items = 2 * grid.x;
            unsigned n_wg = n_items < cus ? n_items : cus;
            n_wg = (n_wg + 7) & ~7u;
            if (stream8) hipLaunchKernelGGL((mfma_bwd_dkv_stream_kernel<64, 8>), dim3(n_wg), dim3(12 * 64), 0, s, kp);
            else hipLaunchKernelGGL((mfma_bwd_dkv_stream_kernel<64, 4>), dim3(n_wg), dim3(8 * 64), 0, s, kp);
        }
    } else if (kp.head_dim == 96) {
        if (p1 && kp.makes_mid) sba_launch_drawing((mfma_bwd_dq_kernel<96, false, true>), (mfma_bwd_dq_drawing_kernel<96, false, true>), grid.x, kThreads, 2, kp, kp.gtab, kDqQueue, false, s);
        else if (p1) sba_launch_drawing((mfma_bwd_dq_kernel<96>), (mfma_bwd_dq_drawing_kernel<96, false, false>), grid.x, kThreads, 2, kp, kp.gtab, kDqQueue, false, s);
        if (p2 && four_pairs) hipLaunchKernelGGL((mfma_bwd_dkv_pair_kernel<96, 4>), grid, dim3(2 * kThreads), 0, s, kp);
        else if (p2) sba_launch_drawing((mfma_bwd_dkv_pair_kernel<96, 2>), (mfma_bwd_dkv_pair_drawing_kernel<96>), 2 * grid.x, kThreads, 2, kp, kp.gtab, kKeyQueue, p1, s);
    } else if (kp.head_dim == 256) {
        // one wave per SIMD in both passes; every wave of the key-owner pass on its own 32 keys, two workgroups per
        // key block that each accumulate one half of the columns of dK and dV - the other key-owner kernels do not
        // fit the CU here
        if (p1) hipLaunchKernelGGL((mfma_bwd_dq_kernel<256>), grid, dim3(kThreads), 0, s, kp);
        if (p2) {
            hipLaunchKernelGGL((mfma_bwd_dkv_own_kernel<256, 2>), dim3(grid.x, 2), dim3(kThreads), 0, s, kp);
        }
    } else {
        if (p1 && kp.makes_mid) sba_launch_drawing((mfma_bwd_dq_kernel<128, false, true>), (mfma_bwd_dq_drawing_kernel<128, false, true>), grid.x, kThreads, 2, kp, kp.gtab, kDqQueue, false, s);
        else if (p1) sba_launch_drawing((mfma_bwd_dq_kernel<128>), (mfma_bwd_dq_drawing_kernel<128, false, false>), grid.x, kThreads, 2, kp, kp.gtab, kDqQueue, false, s);
        // key owners at head_dim 128: two waves per 32 keys (6-9 % faster than one wave per 32 keys,
        // which SBA_DKV_KERNEL=own still selects)
        const bool pair = !(which && !strcmp(which, "own"));
        if (p2 && own && pair && four_pairs) hipLaunchKernelGGL((mfma_bwd_dkv_pair_kernel<128, 4>), grid, dim3(2 * kThreads), 0, s, kp);
        else if (p2 && own && pair) sba_launch_drawing((mfma_bwd_dkv_pair_kernel<128, 2>), (mfma_bwd_dkv_pair_drawing_kernel<128>), 2 * grid.x, kThreads, 2, kp, kp.gtab, kKeyQueue, p1, s);
        else if (p2 && own) hipLaunchKernelGGL((mfma_bwd_dkv_own_kernel<128>), grid, dim3(kThreads), 0, s, kp);
        else if (p2) hipLaunchKernelGGL((mfma_bwd_dkv_kernel<128>), dim3(2 * grid.x), dim3(kThreads), 0, s, kp);
    }
    return hipGetLastError() == hipSuccess ? SBA_OK : SBA_ERR_LAUNCH;
}
