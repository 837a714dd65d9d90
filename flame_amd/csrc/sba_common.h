// Shared device/host helpers for the stick-breaking attention kernels (gfx950).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <stdlib.h>
#include <atomic>
#include "../../include/sba_mi355x.h"

namespace sba {

constexpr int kRowBlock = 128;   // query rows per scheduled job (one workgroup)
constexpr int kMaxHeadDim = 256; // bf16: matrix-core kernels at 64, 128 and 256; every other size and type up to here: generic kernels
constexpr int kKeyBlock = 64;    // keys per sweep step of the MFMA kernels / carry-table column

// Generic (fp32 / any head dim) kernels only: logits above this (in base-2 units) are clamped;
// sigmoid(z) differs from 1 by < 2^-30 there, so outputs move by < 1e-9, and exp2 of the clamped
// value cannot overflow.  The matrix-core kernels do not clamp: their product chains let
// 1 + e^z overflow to +inf (see sba_mfma.h).
constexpr float kMaxLogit2 = 30.0f;
constexpr float kLog2e = 1.4426950408889634f;

struct TensorArg { char* ptr; int64_t sb, sh, st; };
struct VectorArg { char* ptr; int64_t sb, sh; };

// Division by a number that the host knows, in three scalar instructions where the compiler's takes twenty and two transfers to
// the vector unit: n / d = n * ceil(2^(31 + l) / d) >> (31 + l) with 2^l >= d, exact for 0 <= n < 2^31 (the product exceeds n / d by
// less than n 2^l / (d 2^(31 + l)) < 1 / d).  The multiplier is at most 2^32 - 1 from d = 2 on; 2^31 at d = 1.
struct Divisor {
    uint32_t mul;
    int shift;
};
inline Divisor divisor(int d) {
    int l = 0;
    while ((INT64_C(1) << l) < d) ++l;
    return Divisor{(uint32_t)(((UINT64_C(1) << (31 + l)) + d - 1) / d), 31 + l};
}
__device__ inline int divided(int n, const Divisor& d) { return (int)(((uint64_t)(uint32_t)n * d.mul) >> d.shift); }

// Kernel-side copy of SbaParams (by value in the launch).
struct KParams {
    int n_seq, n_heads, seq_len, total_tokens, head_dim, attend_current, save, n_jobs;
    int cols;                      // columns of q, k, v, o, dO, dq, dk, dv that exist: head_dim, or less at head_dim 96
    int carry_only;                // forward kernels: write the carry table and nothing else (no P*V, no o / rem)
    float scale2;                  // scale * log2(e): logits in base-2 units
    float scale;                   // natural-unit scale (for dq/dk)
    const int32_t* cu_seqlens;
    const int32_t* schedule;
    TensorArg q, k, v, o, d_o, dq, dk, dv;
    VectorArg rem, d_rem;
    float* rtab;                   // forward carry table (layout: tab_index() below): the product of (1 - beta) over all keys
                                   //   right of a 64-key block, i.e. the carry entering its RIGHT 32 keys
    float* gtab;                   // backward prefix table, same shape: sum of g over all keys left of the block
    float* rmid;                   // the carry entering the block's LEFT 32 keys (bf16: written by the forward)
    float* gmid;                   // the prefix entering the block's RIGHT 32 keys (written by the dQ pass, like gtab);
                                   //   the bf16 dQ kernels rely on gmid - rtab == gtab - rmid
    TensorArg q_scaled;            // bf16 head_dim 64 backward: q times scale2, rounded to bf16, written by the dQ pass for
                                   //   the key-owner stream and paired kernels (ptr NULL: not wanted)
    float* dkv32;                  // generic path: fp32 dk|dv accumulators
    float* halves;                 // fp32 key-owner pass: sums of two workgroups that share a key block (null: none does)
    float* weights;                // sba_attention_weights(): the attention weights, fp32 (debug output)
    Divisor heads, seqs, cus;      // n_heads, n_seq and n_cus, for the way from a workgroup's index to its job
    int n_cus;
    int spread;                    // heads change their place from round to round of the CUs, see head_of_block()
    int turn;                      // jobs after which the order of a dense launch turns round (0: never), see turned()
    int makes_mid;                 // dQ pass: rmid is not there yet (SBA_SAVE_ONE_TABLE)
    int early_end;                 // forward sweeps end once nothing is left of any of their rows' sticks
    int* gave_up;                  // backward error word (set if a kernel abandoned a bounded internal wait)
    int* queue;                    // where the launch's workgroups draw their jobs, see draw_jobs(): queue i's counter lies i strides further
    int64_t queue_stride;
    int queue_blocks;              // jobs of such a launch
    int64_t tab_head_stride;       // floats per head in each carry table
    int64_t tab_tokens;            // tokens per head in dkv32 and halves (n_seq*T dense, sumT packed)
};

// tab0: first carry-table column of the job's sequence
struct Job { int tok0, len, rb, seq, tab0; };

// Workgroup -> (job, head).  A slot of n_heads consecutive workgroups (which the dispatcher deals round-robin to the 8 XCDs) is
// one job of every head.  Which head comes first moves on by one from slot to slot in the dense layout and every eighth slot
// in the packed one.  A head that stays on one XCD is best for the XCD's L2 if all sweeps are equally long; heads that differ in how far
// their sweeps reach make one XCD the last to finish, and the others wait for it, since workgroups are dealt in order.  Neither
// turn is ahead everywhere; forward + backward in us, every slot / every eighth / fixed heads:
//     mean logits 0 .. -6 over the heads      B=2 H=8 T=16384 d=128 3604 / 3314 / 5497     B=1 H=16 T=8192 d=128 1029 / 1170 / 1207
//         B=4 H=16 T=4096 d=64 644 / 698 / 758     B=1 H=16 T=8192 d=64 726 / 700 / 756     B=1 H=32 T=4096 d=128 635 / 624 / 627
//         packs d=64: 65536 tokens, documents up to 16384 1548 / 1502 / 1554     131072 tokens H=8 1567 / 1417 / 1561     32768 tokens
//         659 / 661 / 657     8192 tokens 212 / 214 / 221     d=128 32768 tokens 1178 / 1193 / 1187
//     all heads at -6 (sweeps nearly full)     B=2 H=8 T=16384 d=128 6053 / 5968 / 5680     B=1 H=16 T=8192 d=128 1429 / 1355 / 1348
//         packs d=64: 65536 tokens 1800 / 1740 / 1716     131072 tokens 1775 / 1706 / 1685
// So turning wins up to 40 % where heads differ and costs up to 7 % where they do not, which no launch can know beforehand (an
// order by the lengths that the forward leaves behind would be a criterion for the backward); packs, whose documents mix the lengths of
// a slot already, turn rarely.  Jobs are sorted by decreasing sweep
// length (longest first); `longest_last` walks the list from its other end (the key-owner
// pass, whose work grows as the row-block index falls).
//
// kSharedCu: kernels of which a CU holds several workgroups.  The CU that gets a round's i-th workgroup gets the next round's i-th, too, so
// by the turn above a head's longest sweeps meet on the same CUs where a round is a multiple of the heads' cycle (2 ... 16 heads on 256
// CUs).  With KParams::spread the heads of round r start the binary fractions' bit-reversed r-th on instead (0, 1/2, 1/4, 3/4, ... of
// them).  Forward + backward against the plain turn, mean logits 0 .. -6 over the heads, in this order / two random ones / all at -6:
//     B=2 H=4 T=16384 d=64 0.87 / 0.88 0.87 / 1.01, d=128 0.88 / 0.88 0.87 / 1.01     B=4 H=4 T=8192 d=64 0.90 / 0.91 0.90 / 1.00
//     B=1 H=8 T=16384 d=128 0.96 / 0.96 0.98 / 1.00     B=1 H=16 T=8192 d=64 0.91 / 0.99 0.99 / 1.00, d=128 0.94 / 1.00 1.01 / 1.01
//     B=1 H=32 T=4096 d=64 0.89 / 0.99 1.00 / 0.99     B=1 H=16 T=16384 d=128 1.00 / 1.01 1.00 / 1.00
// so it pays in any order of up to eight heads, where few heads make a cycle, and costs at most 1 % with more of them in no order; packs
// of 30000 to 65536 tokens, seven of them, 0.93 ... 1.00 in this order and 0.96 ... 1.01 in random ones.  Up to 3000 tokens, whose sweeps end near their starts in no head, and on packs of fewer rounds
// 0.98 ... 1.02: not there.  Kernels with one workgroup a CU lose by it (key owners at d=128 223 -> 237 us, 566 -> 617).
// (A turn of several heads a slot, so that those that follow each other on an XCD are no neighbours: ahead where the neighbours reach
// equally far - over ten shapes 0.99 of the time in the order above, 1.004 in random ones.  Heads have no such order in general.)
//
// The stream's items, two slots to a job and dealt out beforehand, turn by one head in 16 slots, for the sake of the XCD's L2, against one
// a slot in the same orders:  H=16 T=4096 0.99 / 0.98 0.99 / 0.97     H=16 T=5000 0.98 / 0.97 1.00 / 0.99     H=8 T=7000 0.98 / 1.01 1.00 / 0.97
//     H=32 T=1800 1.00 / 1.00 0.99 / 0.97     H=12 T=3000, H=16 T=3500 1.00 / 1.00 / 1.00, 0.99
// With fewer than eight heads they turn every slot (H=4 T=12000 would be 1.04).
// Launches that draw their jobs (draw_jobs()) turn by one head in eight slots: an XCD that is through early takes jobs of the others, and
// the turn by slots costs the L2 more than the unequal heads do.  Forward + backward, turn by slots / by eighths / fixed heads over the launch that
// does not draw, heads in order / in a random one / all at -6:  H=16 T=16384 d=128 0.959 0.933 0.952 / 0.957 0.930 0.981 / 0.992 0.964 0.964
//     T=8192 0.987 1.010 1.044 / 0.994 1.003 1.011 / 0.987 0.946 0.935     packs of 65536 tokens d=80 0.964 0.959 0.984 / 0.963 0.986 0.979 / 0.983 0.979 0.971
enum Sharing { kOnePerCu, kSharedCu, kStreamItems, kDrawn };
template <Sharing kSharing = kOnePerCu>
__device__ inline int head_of_block(const KParams& p, int block) {
    const int slot = divided(block, p.heads);
    int turn = slot;
    if (p.cu_seqlens || kSharing == kDrawn) turn = slot >> 3;
    else if (kSharing == kStreamItems && p.n_heads >= 8) turn = slot >> 4;
    if (kSharing == kSharedCu && p.spread) {
        const int round = divided(slot * p.n_heads, p.cus), of_round = slot - divided(round * p.n_cus + p.n_heads - 1, p.heads);
        turn = (p.cu_seqlens ? of_round >> 3 : of_round) + (int)__umulhi(__builtin_bitreverse32((uint32_t)round), (uint32_t)p.n_heads);
    }
    const int i = block - slot * p.n_heads + turn;
    return i - divided(i, p.heads) * p.n_heads;
}
__device__ inline int slot_of_block(const KParams& p, int block) { return divided(block, p.heads); }
// offset of a (sequence, head)'s first row in a tensor, in elements (products of non-negative indices: their high halves need no
// sign correction)
__device__ inline int64_t slice_offset(const TensorArg& t, int seq, int head, int tok0) {
    return (int64_t)((uint64_t)(uint32_t)seq * (uint64_t)t.sb + (uint64_t)(uint32_t)head * (uint64_t)t.sh + (uint64_t)(uint32_t)tok0 * (uint64_t)t.st);
}
__device__ inline int order_job(int slot, int n_jobs, bool longest_last) {
    return longest_last ? n_jobs - 1 - slot : slot;
}

// Dense jobs are generated arithmetically (row-blocks in decreasing order); packed jobs
// come from the host-built schedule, which has the same order.  Row i of the schedule:
// {first_token, doc_len, row_block, first table column of the document} of the i-th job, then
// the same four of the job that comes i-th for the key-owner kernels.
constexpr int kScheduleInts = 8;

// The schedule is read-only for the kernels and indexed with wave-uniform values: read it
// through the constant address space, so that the loads are scalar (one per wave, and no wait
// for the vector-memory traffic in flight).
typedef const __attribute__((address_space(4))) int32_t* ScheduleRow;
__device__ inline ScheduleRow schedule_row(const KParams& p, int i, int offset) {
    return (ScheduleRow)(uintptr_t)(p.schedule + kScheduleInts * (int64_t)i + offset);
}

// The order of a launch whose workgroups are all resident at once (KParams::turn jobs to a round of the CUs, 0: as they come): the
// list, longest sweeps first, is walked forwards and backwards in turn, so that the CUs with the longest sweep of one round get
// the shortest of the next.  Only the kernels that are launched with it ask for it (kTurns): the division and what it keeps in scalar
// registers cost the resident stream 1.4 %.
__device__ inline int turned(const KParams& p, int i) {
    if (p.turn == 0) return i;
    const int round = i / p.turn;
    return round & 1 ? (2 * round + 1) * p.turn - 1 - i : i;
}

__device__ inline Job dense_job(const KParams& p, int job) {
    Job j;
    int n_rb = (p.seq_len + kRowBlock - 1) / kRowBlock;
    const int from_end = divided(job, p.seqs);
    j.rb = n_rb - 1 - from_end;
    j.seq = job - from_end * p.n_seq;
    j.tok0 = 0;
    j.len = p.seq_len;
    j.tab0 = j.seq * n_rb * (n_rb + 1);
    return j;
}

template <bool kTurns = false>
__device__ inline Job decode_job(const KParams& p, int job) {
    if (p.cu_seqlens == nullptr) return dense_job(p, kTurns ? turned(p, job) : job);
    const ScheduleRow s = schedule_row(p, job, 0);
    Job j;
    j.tok0 = s[0]; j.len = s[1]; j.rb = s[2]; j.seq = 0; j.tab0 = s[3];
    return j;
}

// The key-owner (dK/dV) kernels sweep from a job's row-block to the END of its sequence:
// their longest sweeps are the FIRST row-blocks of the longest sequences.  i-th job in that
// order: arithmetic for the dense layout, the second half of row i of the host-built schedule
// for the packed.
__device__ inline Job decode_key_job(const KParams& p, int i) {
    if (p.cu_seqlens == nullptr) return dense_job(p, p.n_jobs - 1 - i);
    const ScheduleRow s = schedule_row(p, i, 4);
    Job j;
    j.tok0 = s[0]; j.len = s[1]; j.rb = s[2]; j.seq = 0; j.tab0 = s[3];
    return j;
}

// Token index inside dkv32 and halves.
__device__ inline int64_t tab_token(const KParams& p, const Job& j, int local) {
    return (p.cu_seqlens == nullptr) ? (int64_t)j.seq * p.seq_len + local : (int64_t)j.tok0 + local;
}

// Carry tables, compact layout: every sequence has one slab per 128-query row block qb that
// holds exactly the 2*qb + 2 key blocks (64 keys each) that row block can see, as
// [key block][128 queries] fp32.  The slabs of a sequence follow each other (row block qb
// starts qb*(qb+1) columns into the sequence's part, a column being 128 floats), the sequences
// follow each other (Job::tab0), heads are outermost.  A sequence of n row blocks takes
// n*(n+1) columns: half of a full [key blocks][tokens] rectangle.
// Returns the index of (row block qb, key block kb, query 0 of the row block).
__device__ inline int64_t tab_index(const KParams& p, int head, const Job& j, int qb, int kb) {
    return (int64_t)head * p.tab_head_stride + ((int64_t)j.tab0 + qb * (qb + 1) + kb) * kRowBlock;
}

// Where a sweep ends.  A row whose product of (1 - beta) has become exactly 0 gives every key further left the weight 0, the
// logit gradient 0 and leaves no remainder, so a sweep in which that holds for all of its rows ends there: nothing that
// follows could change a bit of any result.  The forward records the leftmost key block it reached per row block
// ("first live block"); the dQ pass starts its sweep there, and leaves for every row block of keys the last row block of
// queries whose sweep reached it ("last live row block"), where the key-owner sweeps end.  Table entries left of a row block's
// first live block exist only where a key-owner sweep passes over them, as zeros that the dQ pass fills in.
// Both numbers live in the tables: the first 64 rows of a row block never see its last key block, so that column's first
// entry belongs to nobody, in rtab as in gtab.
typedef const __attribute__((address_space(4))) int32_t* UniformInts;       // read-only in the kernel: scalar loads
__device__ inline int64_t live_index(const KParams& p, int head, const Job& j, int rb) { return tab_index(p, head, j, rb, 2 * rb + 1); }
__device__ inline void set_first_live(const KParams& p, int head, const Job& j, int kb) {
    ((int32_t*)p.rtab)[live_index(p, head, j, j.rb)] = kb;
}
__device__ inline int first_live_block(const KParams& p, int head, const Job& j) {
    return ((UniformInts)(uintptr_t)p.rtab)[live_index(p, head, j, j.rb)];
}
__device__ inline int last_live_row_block(const KParams& p, int head, const Job& j) {
    return ((UniformInts)(uintptr_t)p.gtab)[live_index(p, head, j, j.rb)];
}
// What one wave of a dQ workgroup does for its row block, whose own sweep starts at key block s0: the last live row block of
// the keys of the same number, and zeros in the entries that key-owner sweeps read although this row block's sweep did not
// reach them (those of later row blocks reach further left: between the lowest of their first blocks and s0).
__device__ inline void close_live_ranges(const KParams& p, int head, const Job& j, int lane, int s0) {
    const int n_rb = (j.len + kRowBlock - 1) / kRowBlock;
    int lowest = s0, last = j.rb;
    for (int at = j.rb + 1; at < n_rb; at += 64) {
        const int f = at + lane < n_rb ? ((const int32_t*)p.rtab)[live_index(p, head, j, at + lane)] : INT32_MAX;
        lowest = min(lowest, f);
        const uint64_t reach = __builtin_amdgcn_ballot_w64((f >> 1) <= j.rb);
        if (reach) last = at + 63 - __builtin_clzll(reach);
    }
    if (lane == 0) ((int32_t*)p.gtab)[live_index(p, head, j, j.rb)] = last;
    if (s0 == 0) return;
    for (int d = 32; d; d >>= 1) lowest = min(lowest, __shfl_xor(lowest, d));
    const int64_t at = tab_index(p, head, j, j.rb, 0);
    for (int i = (lowest & ~1) * kRowBlock + lane; i < s0 * kRowBlock; i += 64) {       // (pairs of key blocks end their sweeps together)
        p.rtab[at + i] = 0.f;
        p.gtab[at + i] = 0.f;
        if (p.rmid) { p.rmid[at + i] = 0.f; p.gmid[at + i] = 0.f; }
    }
}

// Workgroups that draw their jobs.  The dispatcher deals workgroups to the XCDs in turn and in order: where one XCD has no room for its
// next one, all others wait.  With sweeps of unequal lengths a fifth of the chip's slots is empty from the first round to the last.  So a
// launch of many rounds has as many workgroups as the chip holds, which draw their jobs: job i belongs to queue i % 8 and workgroups draw from
// the queue of their own XCD, whose L2 holds the heads of its jobs, and, once that is empty, from the next one that is not.
// A queue is a counter of the jobs taken beyond the first round, which are dealt out by index.  The counters lie in the tables, behind the words
// of live_index() of eight row blocks: the forward's in rtab, the two backward passes' in gtab.
constexpr int kQueues = 8, kForwardQueue = 32, kDqQueue = 32, kKeyQueue = 48;       // entries of live_index()'s column
__device__ inline int queued_block(int queue, int ticket) { return queue + kQueues * (ticket + (int)gridDim.x / kQueues); }
__device__ inline int* queue_counter(const KParams& p, int queue) { return p.queue + queue * p.queue_stride; }
__device__ inline int take_ticket(const KParams& p, int queue) {
    return __hip_atomic_fetch_add(queue_counter(p, queue), 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ inline int lane_index() { return __builtin_amdgcn_mbcnt_hi(-1, __builtin_amdgcn_mbcnt_lo(-1, 0)); }
// (first wave) the job of the ticket that lane 0 took from its home queue, or one from another queue that has some left, or -1.  Counters
// only grow, so the search ends.
__device__ inline int drawn_block(const KParams& p, int home, int ticket, int lane) {
    int block = queued_block(home, __builtin_amdgcn_readfirstlane(ticket));
    while (block >= p.queue_blocks) {
        const int queue = (home + lane) & (kQueues - 1);
        const int next = queued_block(queue, __hip_atomic_load(queue_counter(p, queue), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
        const uint64_t left = __builtin_amdgcn_ballot_w64(lane < kQueues && next < p.queue_blocks);
        if (!left) return -1;
        const int other = (home + __builtin_ctzll(left)) & (kQueues - 1);
        block = queued_block(other, __builtin_amdgcn_readfirstlane(lane == 0 ? take_ticket(p, other) : 0));
    }
    return block;
}
// Runs run(parameters, block, wave, lane, draw) for the workgroup's jobs.  Parameters and lane are given as if they were others each time, so
// that nothing computed from them stays in registers from job to job (without this the forward at head_dim 128 takes 253 registers in place of 214, the dQ pass
// there spills 48 and the key owners 17).  A job calls draw() behind its last step: the ticket is on its way while the results are stored.  (Asked for before the job, it
// would be bound to the end of a long sweep while others find no work: 8192-token packs 1.15 of the time.)
// words: two ints of LDS that a job does not use behind its last barrier.
template <class Run>
__device__ __forceinline__ void draw_jobs(int* words, Run&& run) {
    typedef const __attribute__((address_space(4))) KParams* Arguments;
    int block = blockIdx.x;
    const int home = block & (kQueues - 1);
    int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    for (int parity = 0;; parity ^= 1) {
        Arguments args = (Arguments)__builtin_amdgcn_kernarg_segment_ptr();
        int lane = lane_index();
        asm volatile("" : "+s"(args), "+v"(lane), "+s"(wave));
        __builtin_assume(lane >= 0 && lane < 64);
        const KParams& p = *(const KParams*)args;
        int ticket = 0;
        run(p, block, wave, lane, [&]() __attribute__((always_inline)) {
            if (wave == 0 && lane_index() == 0) ticket = take_ticket(p, home);
        });
        if (wave == 0) {
            const int l = lane_index();
            const int next = drawn_block(p, home, ticket, l);
            if (l == 0) words[parity] = next;
        }
        __syncthreads();                       // (everybody is through with this job's LDS, too)
        block = __builtin_amdgcn_readfirstlane(words[parity]);
        if (block < 0) return;
    }
}
// In front of a dQ pass that draws its jobs, or of a key-owner pass by itself: the dQ pass clears the key owners' queues.
__global__ static void clear_queues_kernel(int* queue, int64_t stride) { queue[threadIdx.x * stride] = 0; }
__device__ inline void clear_words(const KParams& p, int lane) {
    if (lane == 0 && p.gave_up) *p.gave_up = 0;
    if (lane < kQueues && p.queue_stride) ((int*)p.gtab)[kRowBlock + kKeyQueue + lane * p.queue_stride] = 0;
}

__device__ inline float bf16_to_f32(uint16_t b) { return __uint_as_float(((uint32_t)b) << 16); }
__device__ inline uint16_t f32_to_bf16(float f) {   // round to nearest even
    uint32_t u = __float_as_uint(f);
    if ((u & 0x7fffffffu) > 0x7f800000u) return (uint16_t)((u >> 16) | 0x40);
    u += 0x7fffu + ((u >> 16) & 1u);
    return (uint16_t)(u >> 16);
}

template <typename T> struct Elem;
template <> struct Elem<float> {
    __device__ static float load(const char* p, int64_t i) { return ((const float*)p)[i]; }
    __device__ static void store(char* p, int64_t i, float v) { ((float*)p)[i] = v; }
};
template <> struct Elem<_Float16> {
    __device__ static float load(const char* p, int64_t i) { return (float)((const _Float16*)p)[i]; }
    __device__ static void store(char* p, int64_t i, float v) { ((_Float16*)p)[i] = (_Float16)v; }
};
template <> struct Elem<uint16_t> {   // bf16 bits
    __device__ static float load(const char* p, int64_t i) { return bf16_to_f32(((const uint16_t*)p)[i]); }
    __device__ static void store(char* p, int64_t i, float v) { ((uint16_t*)p)[i] = f32_to_bf16(v); }
};

}  // namespace sba

// SBA_TWO_STEP_MAX_GRID (experiments and tests; read once per process): grids of at most this many workgroups take
// the kernels that split a sweep inside the workgroup (head_dim 64), larger ones do not.  -1: not set.
inline int sba_two_step_env() {
    static const int v = [] {
        const char* e = getenv("SBA_TWO_STEP_MAX_GRID");
        return e ? atoi(e) : -1;
    }();
    return v;
}
// The two-steps-per-iteration dQ kernel up to 544 workgroups (measured at H = 16: 103.9 us against the one-step
// kernel's 106.4 at 528 workgroups, 122.0 against 120.6 at 576).  The forward's rule is in sba_launch_mfma_fwd().
constexpr unsigned kTwoStepDqMaxGrid = 544;

// compute units of the current device (asked once per device)
inline int sba_cu_count() {
    static std::atomic<int> cached[64];       // zero-initialised; threads that race here store the same value
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) dev = 0;
    int n = cached[dev].load(std::memory_order_relaxed);
    if (n == 0) {
        if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) n = 256;
        cached[dev].store(n, std::memory_order_relaxed);
    }
    return n;
}

// How long a launch's longest sweep is against the work of an average workgroup slot when every workgroup runs
// one sweep and a CU holds four of them:  r = longest sweep x (4 x CUs) / all sweep steps of the launch  (steps of
// 64 keys; a sequence of n row blocks has n (n + 1) of them per head, which is also its number of carry-table
// columns).  A launch cannot end before its longest sweep has; for r well above 1 most of the chip idles behind
// it, and the kernels that cut a sweep into pieces pay.  seq_len is the longest sequence of the launch, columns its carry-table
// columns per head.
inline double sba_tail_ratio(int seq_len, int64_t columns, int n_heads, unsigned grid) {
    const double longest = 2.0 * ((seq_len + sba::kRowBlock - 1) / sba::kRowBlock);
    double steps = (double)columns * n_heads;
    if (steps <= 0) steps = (double)grid * (longest / 2 + 1);          // (no table size given: every sweep half the longest)
    return longest * 4.0 * sba_cu_count() / steps;
}
inline double sba_tail_ratio(const sba::KParams& kp, unsigned grid) {
    return sba_tail_ratio(kp.seq_len, kp.tab_head_stride / sba::kRowBlock, kp.n_heads, grid);
}

// The same launch with KParams::turn set, for a kernel of which a CU holds `resident` workgroups and that takes `per_job` of them for
// each (job, head).  Only for dense batches in whole rounds of the CUs, several row blocks to a round.  Time against the plain order:
// 16-bit forward at head_dim 64 0.99 ... 0.91 on 512 and 768 workgroups of 9 shapes (1.08 where a round is one row block of every
// sequence: the turn only parts the row blocks of a sequence that meet on a CU), the dQ pass of its backward 0.995 ... 1.005 (forward + backward, nine
// shapes of 512; the key owners, whose launch gained from it, have a kernel that is not turned), float32 0.91 ... 1.00 on 512 workgroups of 9.  On 384 ... 640 workgroups that are no whole rounds
// 1.00 ... 1.03, and at head_dim 96 and 128 in 16 bits 0.98 ... 1.02: left as they come.
inline sba::KParams sba_turning(const sba::KParams& kp, int resident, int per_job = 1) {
    sba::KParams r = kp;
    const int64_t cus = sba_cu_count(), per = (int64_t)kp.n_heads * per_job, grid = kp.n_jobs * per, round = cus / per;
    if (!kp.cu_seqlens && grid > cus && grid <= resident * cus && round > kp.n_seq && kp.n_jobs % round == 0) r.turn = (int)round;
    return r;
}

// Distance of the eight queues' counters: they are in eight heads' or eight sequences' first row blocks (0: there are not so many).
inline int64_t sba_queue_stride(const sba::KParams& kp) {
    if (kp.n_heads >= sba::kQueues) return kp.tab_head_stride;
    return !kp.cu_seqlens && kp.n_seq >= sba::kQueues ? kp.tab_head_stride / kp.n_seq : 0;
}
// Whether a pass of a 16-bit launch draws its jobs.  Forward + backward over the same with a workgroup per job, mean logits 0 .. -6 over the heads in
// order / in a random one / all at -6; work = carry-table columns (64-key steps of all sweeps) x heads:
//     head dims 72 to 128, all three passes   H=16 d=128 T=16384 (work 264000) 0.91 / 0.93 / 0.94, T=12000 0.92 / 0.92 / 0.93, T=8192 (67000) 0.98 / 0.97 / 0.92,
//         H=32 T=8192 0.90 / 0.93 / 0.93, B=2 H=8 T=16384 0.925 / 0.81 / 0.97, B=4 T=4096 (68000) 0.97 / 0.99 / 1.01, B=16 T=4096 0.96 / 0.97 / 0.97;
//         d=80 T=16384 0.93 / 0.94 / 0.94, B=8 H=12 T=4096 0.965 / 0.98 / 1.00;  packs  65536 tokens d=128 0.96 / 0.97 / 0.99, d=80 0.96 / 0.97 / 0.99, documents up
//         to 16384 0.915 / 0.94 / 0.98, up to 1024 d=96 0.99 / 0.98 / 0.97, 32768 tokens 1.00 / 0.98 / 1.01;  below the line B=8 T=2048 (35000) 1.01 / 1.03 / 1.015
//     head_dim 64, the backward's two passes (the forward, of which a CU holds four, gains nothing)   packs  65536 tokens 0.99 / 0.98 / 1.00, H=32 0.96 / 0.95 / 0.99,
//         131072 tokens 0.97 / 0.96 / 0.98, documents up to 16384 0.97 / 0.95 / 0.98;  B=16 H=16 T=4096 0.97 / 0.98 / 0.97, B=4 T=16384 0.98 / 0.98 / 0.99;  below the
//         lines packs of documents up to 1024 1.005 / 1.01 / 1.01, 32768 tokens 1.01 / - / 1.02, B=4 T=4096 (2048 workgroups) 1.01 / - / 1.02
// Short sweeps lose by it: documents up to 300 tokens 1.14.
// SBA_DRAW=1 / =0 (experiments and tests): wherever there are more jobs than the chip holds workgroups, or nowhere.
inline bool sba_draws(const sba::KParams& kp, unsigned blocks, unsigned slots) {
    if (!kp.queue_stride || slots == 0 || blocks <= slots) return false;
    const char* e = getenv("SBA_DRAW");
    if (e && (e[0] == '0' || e[0] == '1')) return e[0] == '1';
    const int64_t grid = (int64_t)kp.n_jobs * kp.n_heads, columns = kp.tab_head_stride / sba::kRowBlock, mean_sweep = columns / kp.n_jobs;
    return kp.head_dim == 64 ? grid >= SBA_DOC_MAJOR_GRID && mean_sweep >= 12 : columns * kp.n_heads >= 60000 && mean_sweep >= 4;
}
// Launches `drawing` with `resident` workgroups a CU where that pays, else `plain` with a workgroup per job.  table, entry: where its queues lie
// (null: nowhere).
template <class Kernel>
inline void sba_launch_drawing(Kernel plain, Kernel drawing, unsigned blocks, int threads, int resident, const sba::KParams& kp, float* table, int entry,
                               bool cleared, hipStream_t s) {
    const unsigned slots = (unsigned)(resident * kp.n_cus) & ~(unsigned)(sba::kQueues - 1);
    if (!table || !sba_draws(kp, blocks, slots)) {
        hipLaunchKernelGGL(plain, dim3(blocks), dim3(threads), 0, s, kp);
        return;
    }
    sba::KParams r = kp;
    r.queue = (int*)table + sba::kRowBlock + entry;
    r.queue_blocks = (int)blocks;
    r.turn = 0;
    if (!cleared) hipLaunchKernelGGL(sba::clear_queues_kernel, dim3(1), dim3(sba::kQueues), 0, s, r.queue, r.queue_stride);
    hipLaunchKernelGGL(drawing, dim3(slots), dim3(threads), 0, s, r);
}

// Launchers implemented in the kernel translation units.
int sba_generic_padded_dim(int D);
int sba_launch_generic_fwd(const sba::KParams& kp, int dtype, hipStream_t s);
int sba_launch_generic_bwd(const sba::KParams& kp, int dtype, hipStream_t s);
int sba_launch_generic_weights(const sba::KParams& kp, int dtype, hipStream_t s);
int sba_launch_mfma_fwd(const sba::KParams& kp, hipStream_t s);
int sba_launch_mfma_bwd(const sba::KParams& kp, int phases, hipStream_t s);
int sba_launch_mfma_f16_fwd(const sba::KParams& kp, hipStream_t s);       // the same kernels compiled for float16 elements
int sba_launch_mfma_f16_bwd(const sba::KParams& kp, int phases, hipStream_t s);
int sba_launch_mfma_f32_fwd(const sba::KParams& kp, hipStream_t s);
int sba_launch_mfma_f32_bwd(const sba::KParams& kp, int phases, hipStream_t s);
bool sba_f32_halves_keys(int seq_len, int64_t columns, int n_heads);        // whether the fp32 key-owner pass cuts sweeps in two
bool sba_mfma_bwd_available();
