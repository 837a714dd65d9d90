// fp32 matrix-core kernels (head_dim 64 and 128): the same sweeps, carry tables and per-step arithmetic
// as the bf16 kernels, with every product on v_mfma_f32_32x32x2_f32.  The reference runs fp32
// inputs through its one tiled kernel as well (stickbreaking_attention/utils.py:8 ALLOW_TF32,
// sb_attn/sb_fwd.py:139-253); here fp32 stays fp32 end to end (the 1e-4 tolerance class), the
// backward is bit-reproducible.
//
// What bounds them is the matrix pipe, which runs fp32 at 1/16 of its bf16 rate: a 32 x 64 tile of scores and its product
// with V keep one SIMD busy for 8192 cycles.  So fp32 runs, which are small, need their work spread over all SIMDs, and
// everything else hides behind the MFMAs:
//   * a workgroup of the forward and of the dQ pass owns 32 query rows, its four waves take four consecutive 64-key steps
//     per iteration and exchange one number per query (product of 1 - beta, sum of g) at the iteration's one barrier;
//   * no tiles in LDS: a wave's operands come straight from global memory (through L1 and L2) into registers, in chunks of
//     16 MFMAs (1024 cycles) of which the next is always on its way;
//   * a workgroup of the key-owner pass owns 64 keys and has eight waves, 256 queries per step.
// B=2, H=8, T=1024, d=64, forward / dQ / dK,dV in us: 85 / 120 / 103 with 128 rows per workgroup, one step at a time and
// tiles through LDS; now 31 / 49 / 87 (the MFMAs alone, evenly spread over the chip: 14 / 20 / 27).
//
// Geometry as in sba_mfma.h: a step covers 64 keys, score tiles are computed transposed (S^T = K Q^T), and MFMA row M of
// tile t holds key
//     key_local = 32*((M>>2)&1) + 16*t + 4*(M>>3) + (M&3)
// so that lane (n, h) has the 32 consecutive keys 32*h + idx of query n in registers
// (idx = 16*t + r): the product chains and prefix sums of sba_mfma.h apply unchanged.
// The 32x32x2 MFMA takes one float per lane for A (row = lane%32, k = lane/32) and for B
// (column = lane%32, k = lane/32).  The contraction index is spread so that a lane fetches four
// consecutive floats at a time: head-dim products use d = 8*j + 4*(lane/32) + i in MFMA 4*j + i;
// key products (P*V, dQ) use key 32*(lane/32) + idx in MFMA idx, which is exactly the register
// the weight of that key sits in.
#include "sba_mfma.h"

namespace sba {
namespace f32 {

constexpr int SK = 64 + 4;                 // row stride of the weight tiles [query][64 keys]
typedef float f32x4 __attribute__((ext_vector_type(4)));

__device__ inline f32x16 mfma32(float a, float b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0);
}
__device__ inline int key_of_row(int t, int M) { return 32 * ((M >> 2) & 1) + 16 * t + 4 * (M >> 3) + (M & 3); }

// One (sequence, head) slice of a tensor: uniform origin and row stride in bytes.
struct Slice {
    const char* origin;
    uint32_t st;
    __device__ inline Slice(const TensorArg& t, const Job& job, int head)
        : origin(t.ptr + 4 * (slice_offset(t, job.seq, head, job.tok0))), st(4u * (uint32_t)t.st) {}
    __device__ inline const char* row(int r) const { return origin + (uint64_t)(uint32_t)r * st; }
};

// 16 of a lane's floats of one row for the head-dim products (chunk c: d = 32*c + 8*j + 4*h + i)
struct Chunk { f32x4 v[4]; };
// `rows`: uniform address of a row; `off`: the lane's row relative to it, in bytes, plus 16*h
__device__ inline Chunk load_chunk(const char* rows, uint32_t off, int c) {
    Chunk r;
#pragma unroll
    for (int j = 0; j < 4; ++j) r.v[j] = *(const f32x4*)(rows + 128 * c + 32 * j + (size_t)off);
    return r;
}
__device__ inline f32x16 chunk_product(const Chunk& a, const float* b, f32x16 acc) {
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int i = 0; i < 4; ++i) acc = mfma32(a.v[j][i], b[4 * j + i], acc);
    return acc;
}
// 16 keys of one 32-wide column block for the key products: keys 32*h + 16*half + e, column 32*db + m
struct Column { float v[16]; };

// The rows (K or V) of one 64-key step as a wave's lanes address them; rows past the end are clamped to the last one
// (their keys are masked for every valid query).
struct StepRows {
    const char* rows;
    uint32_t st, share[2], column, limit;     // lane offsets: row shares of the two tiles; the lane's column in its first key and in the last row
    __device__ inline StepRows(const Slice& s, int key0, int len, int lane) {
        const int m = lane & 31, h = lane >> 5;
        const int last = min(len - 1 - key0, 63);
        rows = s.row(key0);
        st = s.st;
#pragma unroll
        for (int t = 0; t < 2; ++t) share[t] = (uint32_t)min(key_of_row(t, m), last) * st + 16u * h;
        column = 32u * h * st + 4u * m;
        limit = (uint32_t)last * st + 4u * m;
    }
    __device__ inline Chunk chunk(int t, int c) const { return load_chunk(rows, share[t], c); }
    __device__ inline Column keys(int db, int half) const {
        Column r;
        uint32_t off = column + (uint32_t)(16 * half) * st;
        asm volatile("" : "+v"(off));        // (sixteen offsets worked out here each time, not kept in registers through the sweep)
#pragma unroll
        for (int e = 0; e < 16; ++e) {
            r.v[e] = *(const float*)(rows + 128 * db + (size_t)min(off, limit));
            off += st;
        }
        return r;
    }
};

// this lane's share of row `row` for the head-dim products: f[4*j + i] = x[row][8*j + 4*h + i] * s
template <int D>
__device__ inline void load_row_share(float (&f)[D / 2], const Slice& t, int row, int len, int h, float s) {
    const char* ptr = t.row(min(row, len - 1)) + 16 * h;
#pragma unroll
    for (int j = 0; j < D / 8; ++j) {
        const f32x4 x = *(const f32x4*)(ptr + 32 * j);
#pragma unroll
        for (int i = 0; i < 4; ++i) f[4 * j + i] = x[i] * s;
    }
}

// x[16*t + r] = sum_d rows[key(t, row)][d] * f[d-share]: S^T (rows of K, f = scaled Q) or dP^T (rows of V, f = dO).
// `cur` is the first chunk (tile 1), requested by the caller; `after` requests what comes behind the last.
template <int D, class After>
__device__ inline void head_dim_product(float (&x)[32], const StepRows& k, const float (&f)[D / 2], Chunk cur, After&& after) {
    constexpr int kC = D / 32;
    f32x16 acc;
#pragma unroll
    for (int i = 0; i < 2 * kC; ++i) {
        Chunk next = cur;
        if (i + 1 < 2 * kC) next = k.chunk(i + 1 < kC ? 1 : 0, (i + 1) % kC);
        else after();
        __builtin_amdgcn_sched_barrier(0);
        acc = chunk_product(cur, &f[16 * (i % kC)], i % kC == 0 ? f32x16{0} : acc);
        __builtin_amdgcn_sched_barrier(0);
        if (i % kC == kC - 1) {
#pragma unroll
            for (int r = 0; r < 16; ++r) x[16 * (i < kC ? 1 : 0) + r] = acc[r];
        }
        cur = next;
    }
}
// acc[db] (rows d = 32*db + .., column = query) += sum_keys rows[key][d] * w[key]: O^T += V^T P^T, dQ^T += K^T dZ^T.
// `cur` is the first column chunk; `after` as above.
template <int D, class After>
__device__ inline void key_product(f32x16 (&acc)[D / 32], const StepRows& k, const float (&w)[32], Column cur, After&& after) {
#pragma unroll
    for (int i = 0; i < D / 16; ++i) {
        Column next = cur;
        if (i + 1 < D / 16) next = k.keys((i + 1) >> 1, (i + 1) & 1);
        else after();
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[i >> 1] = mfma32(cur.v[e], w[16 * (i & 1) + e], acc[i >> 1]);
        __builtin_amdgcn_sched_barrier(0);
        cur = next;
    }
}

// The accumulators of the four waves (S = 4) added up and stored as rows of a [tokens, D] tensor: every wave stores a quarter of
// them (registers D/8 * wave ..: rows d = 32*db + 8*g + 4*h + 0..3, column = query).
template <int D, int S>
__device__ inline void merge_query_rows(float* park, const f32x16 (&acc)[D / 32], const Slice& t, int row, bool row_ok, int lane, int wave, float s) {
    if (S == 1) {
        if (!row_ok) return;
        char* ptr = const_cast<char*>(t.row(row)) + 16 * (lane >> 5);
#pragma unroll
        for (int g = 0; g < D / 8; ++g) {
            const int db = g >> 2, r = 4 * (g & 3);
            *(f32x4*)(ptr + 32 * g) = f32x4{acc[db][r] * s, acc[db][r + 1] * s, acc[db][r + 2] * s, acc[db][r + 3] * s};
        }
        return;
    }
    float* mine = park + wave * (D / 2) * 64 + lane;
#pragma unroll
    for (int db = 0; db < D / 32; ++db)
#pragma unroll
        for (int r = 0; r < 16; ++r) mine[(16 * db + r) * 64] = acc[db][r];
    __syncthreads();
    if (!row_ok) return;
    char* ptr = const_cast<char*>(t.row(row)) + 16 * (lane >> 5);
#pragma unroll
    for (int i = 0; i < D / 32; ++i) {
        const int g = D / 32 * wave + i;               // registers 4*g .. 4*g + 3
        f32x4 x;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            float sum = 0.f;
#pragma unroll
            for (int w = 0; w < 4; ++w) sum += park[w * (D / 2) * 64 + (4 * g + r) * 64 + lane];
            x[r] = sum * s;
        }
        *(f32x4*)(ptr + 32 * g) = x;
    }
}

// The 32 rows of a wave.  S = 4: the four waves of a workgroup share them and take four consecutive steps of their sweep, and
// a job has four workgroups, longest sweep first.  S = 1: every wave sweeps over its own rows (sequences of one row block,
// whose sweeps have no four steps).
template <int S> struct RowGroup {
    Job job;
    int head, sub, q0, lane_of_sweep;
    __device__ inline RowGroup(const KParams& p, int wave) {
        const int slot = slot_of_block(p, blockIdx.x);
        head = blockIdx.x - slot * p.n_heads + slot / S;
        head -= divided(head, p.heads) * p.n_heads;
        job = decode_job<true>(p, slot / S);
        sub = S == 4 ? 3 - (slot & 3) : wave;
        lane_of_sweep = S == 4 ? wave : 0;
        q0 = job.rb * kRowBlock + 32 * sub;
    }
};
// first live blocks, one per 32-row group (entries 0 .. 3 of the column that live_index() names)
__device__ inline int first_live_of(const KParams& p, int head, const Job& j, int rb) {
    const int32_t* e = (const int32_t*)p.rtab + live_index(p, head, j, rb);
    const int4 v = *(const int4*)e;
    return min(min(v.x, v.y), min(v.z, v.w));
}
// close_live_ranges() for one 32-row group
template <int S>
__device__ inline void close_group_ranges(const KParams& p, const RowGroup<S>& w, int lane, int s0) {
    const Job& j = w.job;
    const int n_rb = (j.len + kRowBlock - 1) / kRowBlock;
    int lowest = first_live_of(p, w.head, j, j.rb), last = j.rb;
    for (int at = j.rb + 1; at < n_rb; at += 64) {
        const int f = at + lane < n_rb ? first_live_of(p, w.head, j, at + lane) : INT32_MAX;
        lowest = min(lowest, f);
        const uint64_t reach = __builtin_amdgcn_ballot_w64((f >> 1) <= j.rb);
        if (reach) last = at + 63 - __builtin_clzll(reach);
    }
    if (lane == 0 && w.sub == 0) ((int32_t*)p.gtab)[live_index(p, w.head, j, j.rb)] = last;
    for (int d = 32; d; d >>= 1) lowest = min(lowest, __shfl_xor(lowest, d));
    const int64_t at = tab_index(p, w.head, j, j.rb, lowest & ~1) + 32 * w.sub + (lane & 31);
    for (int kb = (lowest & ~1) + (lane >> 5); kb < s0; kb += 2) {
        const int64_t e = at + (int64_t)(kb - (lowest & ~1)) * kRowBlock;
        p.rtab[e] = 0.f;
        p.gtab[e] = 0.f;
    }
}

// ---------------------------------------------------------------- forward
template <int D, bool kCarryOnly, int S>
__global__ __launch_bounds__(kThreads, D == 64 ? 3 : 2) void fwd_kernel(KParams p) {
    __shared__ float xch[2][4][32];                        // [parity of the iteration][wave][query]
    __shared__ float park[kCarryOnly || S == 1 ? 1 : 4 * (D / 2) * 64];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int n = lane & 31, h = lane >> 5;
    const RowGroup<S> grp(p, wave);
    const Job& job = grp.job;
    int32_t* const my_first = (int32_t*)p.rtab + live_index(p, grp.head, job, job.rb) + grp.sub;
    if (grp.q0 >= job.len) {                               // (S = 4: the whole workgroup)
        if (p.save && (S == 1 ? lane : (int)threadIdx.x) == 0) *my_first = INT32_MAX;
        return;
    }
    const int strict = p.attend_current ? 0 : 1;
    const int qi = grp.q0 + n;
    const bool row_ok = qi < job.len;
    const Slice q(p.q, job, grp.head), k(p.k, job, grp.head), v(p.v, job, grp.head);
    float qf[D / 2];
    load_row_share<D>(qf, q, qi, job.len, h, p.scale2);
    f32x16 oacc[D / 32];
#pragma unroll
    for (int db = 0; db < D / 32; ++db) oacc[db] = f32x16{0};
    float R = row_ok ? 1.0f : 0.0f;
    const float nothing = p.early_end ? 0.f : -1.f;        // carries of a sweep that has ended, see live_index()
    const int kmax = min(grp.q0 + 31, job.len - 1) - strict;
    const int n_steps = kmax >= 0 ? kmax / kKeyBlock + 1 : 0;
    const int64_t tabq = tab_index(p, grp.head, job, job.rb, 0) + 32 * grp.sub + n;

    Chunk kc{};
    if (n_steps - 1 - grp.lane_of_sweep >= 0) kc = StepRows(k, (n_steps - 1 - grp.lane_of_sweep) * kKeyBlock, job.len, lane).chunk(1, 0);
    int it = 0, iterations = (n_steps + S - 1) / S;
    for (; it < iterations; ++it) {
        const int step = n_steps - 1 - S * it - grp.lane_of_sweep;
        float (*const x4)[32] = xch[it & 1];
        float t[S];
        auto exchange = [&](float total) {
            if (S == 1) { t[0] = total; return; }
            if (h == 0) x4[wave][n] = total;
            __syncthreads();
#pragma unroll
            for (int w = 0; w < S; ++w) t[w] = x4[w][n];
        };
        if (step >= 0) {
            const int key0 = step * kKeyBlock;
            const StepRows kr(k, key0, job.len, lane), vr(v, key0, job.len, lane);
            float x[32], dummy[1], total;
            Column vc{};
            head_dim_product<D>(x, kr, qf, kc, [&]() { if (!kCarryOnly) vc = vr.keys(0, 0); });
            if (key0 + 63 + strict > grp.q0) mask_step(x, key0 + 32 * h, qi, strict);
            const float factor = stick_weights_local<false>(x, dummy, total, lane);
            exchange(total);
            float mine = R;
#pragma unroll
            for (int w = 0; w < S - 1; ++w)
                if (w < wave) mine *= t[w];
            if (p.save && h == 0 && row_ok) p.rtab[tabq + (int64_t)step * kRowBlock] = mine;
            auto next_keys = [&]() { kc = StepRows(k, max(step - S, 0) * kKeyBlock, job.len, lane).chunk(1, 0); };
            if (!kCarryOnly) {
                scale_clamped<32>(x, mine * factor);
                key_product<D>(oacc, vr, x, vc, next_keys);
            } else {
                next_keys();
            }
        } else {
            exchange(1.0f);
        }
#pragma unroll
        for (int w = 0; w < S; ++w) R *= t[w];
        if (__builtin_amdgcn_ballot_w64(R != nothing) == 0) {      // the same numbers in all four waves
            int here = it + 1;
            asm("" : "+s"(here));
            iterations = here;
        }
    }
    if (p.save && (S == 1 ? lane : (int)threadIdx.x) == 0) *my_first = max(n_steps - S * iterations, 0);
    if (!kCarryOnly) {
        merge_query_rows<D, S>(park, oacc, Slice(p.o, job, grp.head), qi, row_ok, lane, wave, 1.0f);
        if (row_ok && h == 0 && grp.lane_of_sweep == 0)
            ((float*)p.rem.ptr)[(int64_t)job.seq * p.rem.sb + (int64_t)grp.head * p.rem.sh + job.tok0 + qi] = R;
    }
}

// queries of the first half of the steps of the job's key blocks (W = 8)
__device__ inline int first_half(const Job& job) {
    return ((job.len - job.rb * kRowBlock + 511) >> 9) << 8;
}
// end of the queries that the job's keys have weights in
__device__ inline int live_end(const KParams& p, int head, const Job& job) {
    return min(job.len, (last_live_row_block(p, head, job) + 1) * kRowBlock);
}
// a key's row of the sums that workgroup `part` of two leaves of dK or dV
template <int D>
__device__ inline float* half_row(const KParams& p, int part, bool is_dk, const Job& job, int head, int key) {
    return p.halves + (((2 * part + is_dk) * (int64_t)p.n_heads + head) * p.tab_tokens + tab_token(p, job, key)) * D;
}

// ---------------------------------------------------------------- backward pass 1: dQ + prefix table
template <int D, int S>
__global__ __launch_bounds__(kThreads, D == 64 ? 2 : 1) void bwd_dq_kernel(KParams p) {
    __shared__ float xch[2][4][32];
    __shared__ float park[S == 1 ? 1 : 4 * (D / 2) * 64];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int n = lane & 31, h = lane >> 5;
    const RowGroup<S> grp(p, wave);
    const Job& job = grp.job;
    if (grp.q0 >= job.len) return;                         // (S = 4: the whole workgroup)
    const int strict = p.attend_current ? 0 : 1;
    const int qi = grp.q0 + n;
    const bool row_ok = qi < job.len;
    const Slice q(p.q, job, grp.head), k(p.k, job, grp.head), v(p.v, job, grp.head), d_o(p.d_o, job, grp.head);
    float qf[D / 2], dof[D / 2];
    load_row_share<D>(qf, q, qi, job.len, h, p.scale2);
    load_row_share<D>(dof, d_o, qi, job.len, h, 1.0f);
    float dr = 0.f;
    if (row_ok && p.d_rem.ptr)
        dr = ((const float*)p.d_rem.ptr)[(int64_t)job.seq * p.d_rem.sb + (int64_t)grp.head * p.d_rem.sh + job.tok0 + qi];
    f32x16 dqacc[D / 32];
#pragma unroll
    for (int db = 0; db < D / 32; ++db) dqacc[db] = f32x16{0};
    float Gc = 0.f;
    const int kmax = min(grp.q0 + 31, job.len - 1) - strict;
    const int n_steps = kmax >= 0 ? kmax / kKeyBlock + 1 : 0;
    const int64_t tabq = tab_index(p, grp.head, job, job.rb, 0) + 32 * grp.sub + n;
    const int first = __builtin_amdgcn_readfirstlane(((const int32_t*)p.rtab)[live_index(p, grp.head, job, job.rb) + grp.sub]);
    if (first > 0) Gc = dr * 0.f;                          // (see the bf16 dQ kernel)
    if (S == 1 || wave == 3) close_group_ranges(p, grp, lane, first);

    // (whole fours of steps: every wave keeps its share of them wherever a sweep begins)
    const int base = first & ~(S - 1), iterations = (n_steps - base + S - 1) / S;
    Chunk kc{};
    if (base + grp.lane_of_sweep < n_steps) kc = StepRows(k, (base + grp.lane_of_sweep) * kKeyBlock, job.len, lane).chunk(1, 0);
    for (int it = 0; it < iterations; ++it) {
        const int step = base + S * it + grp.lane_of_sweep;
        float (*const x4)[32] = xch[it & 1];
        float t[S];
        auto exchange = [&](float total) {
            if (S == 1) { t[0] = total; return; }
            if (h == 0) x4[wave][n] = total;
            __syncthreads();
#pragma unroll
            for (int w = 0; w < S; ++w) t[w] = x4[w][n];
        };
        if (step >= first && step < n_steps) {
            const int key0 = step * kKeyBlock;
            const StepRows kr(k, key0, job.len, lane), vr(v, key0, job.len, lane);
            float R = row_ok ? p.rtab[tabq + (int64_t)step * kRowBlock] : 0.0f;     // (rows past the end: weights and gradients exactly 0)
            float x[32], beta[32], dp[32], total;
            Chunk vc{};
            head_dim_product<D>(x, kr, qf, kc, [&]() { vc = vr.chunk(1, 0); });
            if (key0 + 63 + strict > grp.q0) mask_step(x, key0 + 32 * h, qi, strict);
            head_dim_product<D>(dp, vr, dof, vc, []() {});
            stick_weights<true>(x, beta, R, lane);
            float start = logit_grads_local(x, dp, total, lane);
            // the gradient of rem rides in the prefix as the constant d_rem * rem (see the bf16 dQ kernel): with the
            // leftmost block it joins that step's total and its own prefix
            const float c0 = step == 0 ? dr * R : 0.f;
            const Column kcol = kr.keys(0, 0);
            exchange(total + c0);
            float mine = Gc;
#pragma unroll
            for (int w = 0; w < S - 1; ++w)
                if (w < wave) mine += t[w];
            mine += c0;
            if (row_ok && h == 0) p.gtab[tabq + (int64_t)step * kRowBlock] = mine;
            logit_grads_apply(beta, dp, mine + start);
            key_product<D>(dqacc, kr, dp, kcol, [&]() { kc = StepRows(k, min(step + S, n_steps - 1) * kKeyBlock, job.len, lane).chunk(1, 0); });
        } else {
            exchange(0.0f);
            kc = StepRows(k, min(step + S, n_steps - 1) * kKeyBlock, job.len, lane).chunk(1, 0);
        }
#pragma unroll
        for (int w = 0; w < S; ++w) Gc += t[w];
    }
    // the scaled Q share carries scale * log2(e): dq = scale * dZ K
    merge_query_rows<D, S>(park, dqacc, Slice(p.dq, job, grp.head), qi, row_ok, lane, wave, p.scale);
}

// ---------------------------------------------------------------- backward pass 2: dK, dV
// One workgroup of W = 8 or 4 waves per (64-key block, head); a step covers 32 queries per wave.  Each wave turns its queries into
// weights and logit gradients (carries from the two tables) and leaves them in LDS as [query][key] rows; after a barrier
// it reduces [32 keys x 32 d] tiles of dV (W = 8: waves 0-3) and dK (waves 4-7) over all queries of the step: key half
// w & 1, column blocks (w >> 1 & 1) + 2*j.
// kCut: two workgroups per (64-key block, head), one for each half of its steps, which leave their sums in KParams::halves for
// add_halves_kernel (where the second half has steps at all; otherwise the first stores the rows).  The cut lies at a step that the
// sequence's length alone decides.  B=2, H=8, T=1024, d=64, both passes and the forward: 168 us with one workgroup a key block, 159 so; 164
// if the second workgroup to finish adds the sums itself (their round trips through memory), 246 with fences around that, which empty
// the L2; 155 with float atomics on cleared rows of dK and dV, which are not defined on every memory that a gradient may lie in.
template <int D, int W, bool kCut = false>
__global__ __launch_bounds__(W * 64, 2) void bwd_dkv_kernel(KParams p) {
    constexpr int kMine = D / 64;              // output tiles per wave and tensor
    constexpr int kBoth = 8 / W;               // tensors per wave
    constexpr int kStep = 32 * W;
    __shared__ __attribute__((aligned(16))) float ztile[2][kStep * SK];      // a | dz: [query][key]
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int n = lane & 31, h = lane >> 5;
    const int head = head_of_block(p, blockIdx.x);
    const int unit = slot_of_block(p, blockIdx.x);
    const int slot = kCut ? unit >> 1 : unit;  // two 64-key blocks per scheduled 128-row job
    const int part = kCut ? unit & 1 : 0;
    const Job job = decode_key_job(p, slot >> 1);
    const int kb = 2 * job.rb + (slot & 1);
    const int key0 = kb * kKeyBlock;
    if (key0 >= job.len) return;               // uniform over the workgroup
    const int strict = p.attend_current ? 0 : 1;
    const Slice q(p.q, job, head), k(p.k, job, head), v(p.v, job, head), d_o(p.d_o, job, head);
    const StepRows kr(k, key0, job.len, lane), vr(v, key0, job.len, lane);
    const int kh = wave & 1, dbw = (wave >> 1) & 1;
    f32x16 acc[kBoth][kMine];
#pragma unroll
    for (int t = 0; t < kBoth; ++t)
#pragma unroll
        for (int j = 0; j < kMine; ++j) acc[t][j] = f32x16{0};
    const int q_live = live_end(p, head, job);
    const int cut = kCut ? first_half(job) : 0;
    const int q_start = job.rb * kRowBlock + part * cut, q_end = kCut && part == 0 ? min(q_live, q_start + cut) : q_live;
    if (kCut && part == 1 && q_start >= q_end) return;         // uniform over the workgroup
    // the step's Q and dO rows, for head_dim 64 requested as soon as the step before has used its own
    constexpr bool kAhead = D == 64;
    float qf[D / 2], dof[D / 2];
    if (kAhead) {
        const int qi0 = q_start + 32 * wave + n;
        load_row_share<D>(qf, q, qi0, job.len, h, p.scale2);
        load_row_share<D>(dof, d_o, qi0, job.len, h, 1.0f);
    }
    for (int q_begin = q_start; q_begin < q_end; q_begin += kStep) {
        const int q0w = q_begin + 32 * wave, qi = q0w + n;
        {
            float x[32], dp[32];
            if (key0 + strict <= q0w + 31 && q0w < q_end) {
                float R = 0.f, Gc = 0.f;           // rows past the end: zero carries make weights and gradients exactly zero
                if (qi < job.len) {
                    const int64_t t = tab_index(p, head, job, q0w / kRowBlock, kb) + (q0w % kRowBlock) + n;
                    R = p.rtab[t]; Gc = p.gtab[t];
                }
                float beta[32];
                if (!kAhead) load_row_share<D>(qf, q, qi, job.len, h, p.scale2);
                Chunk vc{};
                head_dim_product<D>(x, kr, qf, kr.chunk(1, 0), [&]() { vc = vr.chunk(1, 0); });
                if (kAhead) load_row_share<D>(qf, q, qi + kStep, job.len, h, p.scale2);
                else load_row_share<D>(dof, d_o, qi, job.len, h, 1.0f);
                head_dim_product<D>(dp, vr, dof, vc, []() {});
                if (kAhead) load_row_share<D>(dof, d_o, qi + kStep, job.len, h, 1.0f);
                if (key0 + 63 + strict > q0w) mask_step(x, key0 + 32 * h, qi, strict);
                stick_weights<true>(x, beta, R, lane);
                logit_grads<true>(x, beta, dp, Gc, lane);
            } else {
#pragma unroll
                for (int idx = 0; idx < 32; ++idx) { x[idx] = 0.f; dp[idx] = 0.f; }
                if (kAhead) {
                    load_row_share<D>(qf, q, qi + kStep, job.len, h, p.scale2);
                    load_row_share<D>(dof, d_o, qi + kStep, job.len, h, 1.0f);
                }
            }
            float* za = &ztile[0][(32 * wave + n) * SK + 32 * h];
            float* zd = &ztile[1][(32 * wave + n) * SK + 32 * h];
#pragma unroll
            for (int c = 0; c < 8; ++c) {
                *(f32x4*)(za + 4 * c) = f32x4{x[4 * c], x[4 * c + 1], x[4 * c + 2], x[4 * c + 3]};
                *(f32x4*)(zd + 4 * c) = f32x4{dp[4 * c], dp[4 * c + 1], dp[4 * c + 2], dp[4 * c + 3]};
            }
        }
        __syncthreads();
        // dV[key][d] += sum_q a[q][key] dO[q][d]  or  dK[key][d] += sum_q dz[q][key] Q[q][d], 32 queries at a time
#pragma unroll
        for (int t = 0; t < kBoth; ++t) {
            const bool is_dk = kBoth == 2 ? t == 1 : wave >= 4;
            const Slice reduced = is_dk ? q : d_o;
            const float* z = &ztile[is_dk ? 1 : 0][h * SK + 32 * kh + n];
            const uint32_t st = reduced.st;
            struct Rows { float v[kMine][16], z[16]; };
            auto load = [&](int r0) {
                Rows r;
                const int row0 = min(q_begin + r0, job.len - 1);                  // (rows past the end have zero weights)
                const char* rows = reduced.row(row0);
                uint32_t off = h * st + 128u * dbw + 4u * n;
                const uint32_t limit = (uint32_t)min(job.len - 1 - row0, 31) * st + 128u * dbw + 4u * n;
                asm volatile("" : "+v"(off));
#pragma unroll
                for (int i = 0; i < 16; ++i) {
#pragma unroll
                    for (int j = 0; j < kMine; ++j) r.v[j][i] = *(const float*)(rows + 256 * j + (size_t)min(off, limit));
                    off += 2 * st;
                    r.z[i] = z[(min(r0, kStep - 32) + 2 * i) * SK];
                }
                return r;
            };
            auto multiply = [&](const Rows& r) {
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int i = 0; i < 16; ++i)
#pragma unroll
                    for (int j = 0; j < kMine; ++j) acc[t][j] = mfma32(r.z[i], r.v[j][i], acc[t][j]);
                __builtin_amdgcn_sched_barrier(0);
            };
            // (rows_here in whole 64s: the rows of waves that had no queries to turn into weights are zeros)
            const int rows_here = min(kStep, (q_end - q_begin + 63) & ~63);
            Rows even = load(0);
            for (int r0 = 0; r0 < rows_here; r0 += 64) {
                const Rows odd = load(r0 + 32);
                multiply(even);
                even = load(r0 + 64);
                multiply(odd);
            }
        }
        __syncthreads();                       // the weight tiles are free
    }
    // accumulator rows are keys 32*kh + 8*(r/4) + 4*h + r%4, columns d = 32*(dbw + 2j) + n: dk = scale * dZ^T Q
#pragma unroll
    for (int t = 0; t < kBoth; ++t) {
        const bool is_dk = kBoth == 2 ? t == 1 : wave >= 4;
        const Slice out(is_dk ? p.dk : p.dv, job, head);
        const bool halved = kCut && q_live > job.rb * kRowBlock + cut;
        const float s = is_dk && !halved ? p.scale : 1.0f;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int key = key0 + 32 * kh + 8 * (r >> 2) + 4 * h + (r & 3);
            if (key >= job.len) continue;
            float* const row = halved ? half_row<D>(p, part, is_dk, job, head, key) : (float*)const_cast<char*>(out.row(key));
#pragma unroll
            for (int j = 0; j < kMine; ++j) row[32 * (dbw + 2 * j) + n] = acc[t][j][r] * s;
        }
    }
}

// dK and dV of the key blocks that two workgroups shared, 32 rows a workgroup: what bounds it is its launch (4 us in all at
// B=2, H=8, T=1024, d=64, of 159).
template <int D>
__global__ __launch_bounds__(kThreads) void add_halves_kernel(KParams p) {
    const int slot = slot_of_block(p, blockIdx.x), head = head_of_block(p, blockIdx.x);
    const Job job = decode_key_job(p, slot >> 2);
    if (live_end(p, head, job) <= job.rb * kRowBlock + first_half(job)) return;
    const int row0 = job.rb * kRowBlock + 32 * (slot & 3);
    constexpr int kChunks = 32 * D / 4;                    // of 16 bytes, per tensor
#pragma unroll
    for (int c = threadIdx.x; c < 2 * kChunks; c += kThreads) {
        const bool is_dk = c >= kChunks;
        const int key = row0 + c % kChunks / (D / 4), at = 4 * (c % (D / 4));
        if (key >= job.len) continue;
        const f32x4 a = *(const f32x4*)(half_row<D>(p, 0, is_dk, job, head, key) + at), b = *(const f32x4*)(half_row<D>(p, 1, is_dk, job, head, key) + at);
        const Slice out(is_dk ? p.dk : p.dv, job, head);
        *(f32x4*)(const_cast<char*>(out.row(key)) + 4 * at) = (a + b) * (is_dk ? p.scale : 1.0f);
    }
}

}  // namespace f32
}  // namespace sba

namespace {
using namespace sba;

template <int D, int S>
void launch_f32_fwd(const KParams& kp, hipStream_t s) {
    const dim3 grid(S * (unsigned)kp.n_jobs * kp.n_heads);
    const KParams turning = sba_turning(kp, D == 64 ? 3 : 2, S);
    if (kp.carry_only) hipLaunchKernelGGL((f32::fwd_kernel<D, true, S>), grid, dim3(kThreads), 0, s, turning);
    else hipLaunchKernelGGL((f32::fwd_kernel<D, false, S>), grid, dim3(kThreads), 0, s, turning);
}
template <int D>
void launch_f32_bwd(const KParams& kp, int phases, hipStream_t s) {
    const unsigned jobs = (unsigned)kp.n_jobs * kp.n_heads;
    // Sequences of one row block (at most 128 tokens) leave nothing to share among a sweep's waves: 8192 tokens in documents of
    // 16 .. 128 take 193 us forward + backward this way, 276 with S = 4 and W = 8.  Longer ones are 4-15 % ahead with eight
    // waves per workgroup in the key-owner pass.
    const bool one_block = kp.seq_len <= kRowBlock;
    if (phases != 2 && one_block) hipLaunchKernelGGL((f32::bwd_dq_kernel<D, 1>), dim3(jobs), dim3(kThreads), 0, s, kp);
    else if (phases != 2) hipLaunchKernelGGL((f32::bwd_dq_kernel<D, 4>), dim3(4 * jobs), dim3(kThreads), 0, s, sba_turning(kp, D == 64 ? 2 : 1, 4));
    if (phases != 1 && one_block) hipLaunchKernelGGL((f32::bwd_dkv_kernel<D, 4>), dim3(2 * jobs), dim3(4 * 64), 0, s, kp);
    else if (phases != 1 && kp.halves) {
        hipLaunchKernelGGL((f32::bwd_dkv_kernel<D, 8, true>), dim3(4 * jobs), dim3(8 * 64), 0, s, kp);
        hipLaunchKernelGGL((f32::add_halves_kernel<D>), dim3(4 * jobs), dim3(kThreads), 0, s, kp);
    } else if (phases != 1) hipLaunchKernelGGL((f32::bwd_dkv_kernel<D, 8>), dim3(2 * jobs), dim3(8 * 64), 0, s, kp);
}
}  // namespace

// A key-owner workgroup has its CU to itself, so a launch of few lasts as long as the one with the most steps.  Where that is more
// than 1.6 times the average share of a CU (an eighth of the tail ratio), two workgroups take half of the steps each (sequences of at most 256 tokens
// have a single step).  Both passes and the forward, with against without, by that measure: 7.1-7.8 0.71-0.78 (1.05-1.07 where hardly
// a sweep reaches its second half: one head of logits near 0, 72 us), 3.8 0.71-0.74, 3.2 0.78-0.84, 4.0 at T=300 0.93-0.97, 1.9 0.80-0.84, 1.8
// 0.90-0.95 (H=16, T=1024: 168 -> 159 us, D=128 305 -> 273);  1.6 1.05-1.10, 1.3 1.10-1.13, 1.2 0.95-1.08, 0.9-1.0 1.08-1.27: the second
// workgroup's prologue and the sums' way through memory.
bool sba_f32_halves_keys(int seq_len, int64_t columns, int n_heads) {
    return seq_len > 256 && columns > 0 && sba_tail_ratio(seq_len, columns, n_heads, 0) >= 13.0;
}

int sba_launch_mfma_f32_fwd(const sba::KParams& kp, hipStream_t s) {
    const bool one_block = kp.seq_len <= kRowBlock;
    if (kp.head_dim == 64) one_block ? launch_f32_fwd<64, 1>(kp, s) : launch_f32_fwd<64, 4>(kp, s);
    else one_block ? launch_f32_fwd<128, 1>(kp, s) : launch_f32_fwd<128, 4>(kp, s);
    return hipGetLastError() == hipSuccess ? SBA_OK : SBA_ERR_LAUNCH;
}

int sba_launch_mfma_f32_bwd(const sba::KParams& kp, int phases, hipStream_t s) {
    if (!kp.rtab || !kp.gtab) return SBA_ERR_WORKSPACE;
    if (kp.head_dim == 64) launch_f32_bwd<64>(kp, phases, s);
    else launch_f32_bwd<128>(kp, phases, s);
    return hipGetLastError() == hipSuccess ? SBA_OK : SBA_ERR_LAUNCH;
}
