// The language model's matrix products on the matrix cores: projections of token rows with what follows them (projection
// kernels, second half of the file) and weight gradients.  Compiled once for bf16 and, with SBA_ELEM_F16, once for float16.
//
// Weight gradients: C[m][n] = sum over t of A[t][m] * B[t][n], A and B 16-bit with the contracted index outermost, C fp32.
// Several products that share the contraction length run in one launch.
#include <type_traits>

#include "sba_mfma.h"
#include "sba_model.h"

namespace sba {
inline namespace SBA_ELEM_NS {

// A workgroup of four waves, one per SIMD, owns a TM x 256 tile of C; a wave holds TM/2 x 128 of it (with TM = 256 sixty-four 16 x 16
// accumulators, 256 registers).  That is the shape at which the LDS keeps up: per 32 rows of the contraction a wave reads sixteen
// operand fragments for sixty-four MFMAs, so the four waves' reads (64 KB) and the arriving tiles (32 KB) take 768 of the 1088 cycles
// that the MFMAs do; eight waves of 128 x 64 would ask for 96 + 32 KB.
// Both operands have the contracted index in rows, so every fragment is a transposing fetch (ds_read_b64_tr_b16).
// Stages of 32 rows, four tile buffers.  The operands of a stage are fetched under the MFMAs of the one before; then the waves meet: the
// buffer that was read is free for the stage four ahead (requested at once), and the next stage but one is known to have landed.
constexpr int kTileN = 256, kStageRows = 32, kBuffers = 4;
constexpr int kTileBytes = kStageRows * 256 * 2;             // one operand's stage: 16 KB
constexpr int kBBase = kBuffers * kTileBytes;                // A's buffers, then B's

struct TileSource {
    const char* at;              // next stage's first row, first column of the tile: uniform
    uint32_t off[4];             // this lane's chunk in each of the wave's four copies
    uint32_t row_bytes;
    int64_t step;

    // rows 2 * (w + 4 * i) + lane / 32 of a stage; the lane takes the chunk that belongs at its LDS position, clamped to the
    // matrix (columns past its edge are worked out from other columns' values and not stored)
    __device__ inline void init(const void* base, int64_t ld, int col0, int cols, int w, int lane) {
        at = (const char*)base + 2 * (int64_t)col0;
        row_bytes = (uint32_t)(2 * ld);
        step = 2 * ld * kStageRows;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int row = 2 * (w + 4 * i) + (lane >> 5);
            off[i] = (uint32_t)row * row_bytes + chunk_bytes(row, cols - col0, lane);
        }
    }
    __device__ static inline uint32_t chunk_bytes(int row, int cols_left, int lane) {
        const int c = (lane & 31) ^ swz<256>(row);
        return 16u * (uint32_t)min(c, cols_left / 8 - 1);
    }
};

__device__ inline h16x8 fragment(uint32_t a0, uint32_t a1, int imm) {
    union { s16x4 v[2]; h16x8 b; } u;
    u.v[0] = lds_read_tr_at(a0, imm);
    u.v[1] = lds_read_tr_at(a1, imm);
    return u.b;
}

typedef float f32x4 __attribute__((ext_vector_type(4)));
// 16 x 16 x 32: lane l holds row l % 16 (a) or column l % 16 (b), contracted indices 8 * (l / 16) .. + 7; of the result column l % 16,
// rows 4 * (l / 16) .. + 3.
__device__ inline f32x4 mfma16(h16x8 a, h16x8 b, f32x4 c) {
#ifdef SBA_ELEM_F16
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
#else
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
#endif
}

// The same with the sums kept where they are.  The compiler's own instruction may write its result elsewhere, and with 224 of the 256
// accumulation registers in use it does: 360 moves per four stages.  It does not see the instruction's latency either: settled()
// before the sums are read.
__device__ inline void mfma16_in_place(h16x8 a, h16x8 b, f32x4& c) {
#ifdef SBA_ELEM_F16
    asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %2, %0" : "+a"(c) : "v"(a), "v"(b));
#else
    asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(c) : "v"(a), "v"(b));
#endif
}
template <int N, int M> __device__ inline void settled(f32x4 (&acc)[N][M]) {
    asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");
#pragma unroll
    for (int i = 0; i < N; ++i)
#pragma unroll
        for (int j = 0; j < M; ++j) asm volatile("" : "+a"(acc[i][j]));
}

template <int TM>
__global__ __launch_bounds__(256, 1) void weight_grad_kernel(sba_model::WeightGrads g) {
    constexpr int TI = TM / 32, TJ = 8;                          // 16-wide blocks of a wave: rows and columns of C
    __shared__ __attribute__((aligned(1024))) char lds[2 * kBuffers * kTileBytes];
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);

    // workgroups are dealt to the eight XCDs in turn: each takes a run of neighbouring tiles, whose operands its L2 then shares
    const int per = (g.tiles + 7) / 8, t = (int)(blockIdx.x & 7) * per + (int)(blockIdx.x >> 3);
    if ((int)(blockIdx.x >> 3) >= per || t >= g.tiles) return;
    int which = 0;
    while (which + 1 < g.n && t >= g.first_tile[which + 1]) ++which;
    const sba_model::WeightGrad& pr = g.one[which];
    const int tiles_m = (pr.m + TM - 1) / TM, tiles_n = (pr.n + kTileN - 1) / kTileN, local = t - g.first_tile[which];
    // bands of four tile rows, walked column by column
    const int band = local / (4 * tiles_n), rows = min(4, tiles_m - 4 * band), in = local - band * 4 * tiles_n;
    const int m0 = (4 * band + in % rows) * TM, n0 = (in / rows) * kTileN;

    // this split's stages of the contraction
    const int all = (g.k + kStageRows - 1) / kStageRows, share = (all + (int)gridDim.y - 1) / (int)gridDim.y;
    const int first = min(all, (int)blockIdx.y * share), nk = min(all - first, share);
    const int ragged = g.k - (first + nk - 1) * kStageRows;          // rows of the last stage (32 unless it is the end)

    TileSource sa, sb;
    sa.init(pr.a, pr.lda, m0, min(pr.m, m0 + TM), w, lane);
    sb.init(pr.b, pr.ldb, n0, pr.n, w, lane);
    sa.at += first * sa.step;
    sb.at += first * sb.step;
    const uint32_t lds0 = lds_address(lds);

    auto request = [&](int stage, int buf) {
        if (stage + 1 < nk || ragged >= kStageRows) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                dma16(sa.at, sa.off[i], lds0 + buf * kTileBytes + (w + 4 * i) * 1024);
                dma16(sb.at, sb.off[i], lds0 + kBBase + buf * kTileBytes + (w + 4 * i) * 1024);
            }
        } else {
#pragma unroll
            for (int i = 0; i < 4; ++i) {            // rows past the end: the last one, cleared when it has landed
                const int row = 2 * (w + 4 * i) + (lane >> 5);
                const uint32_t back = (uint32_t)max(0, row - (ragged - 1));
                dma16(sa.at, sa.off[i] - back * sa.row_bytes, lds0 + buf * kTileBytes + (w + 4 * i) * 1024);
                dma16(sb.at, sb.off[i] - back * sb.row_bytes, lds0 + kBBase + buf * kTileBytes + (w + 4 * i) * 1024);
            }
        }
        sa.at += sa.step;
        sb.at += sb.step;
    };
    // rows of a stage that exist; the others are cleared once the stage's copies have landed
    auto rows_of = [&](int stage) { return stage + 1 < nk ? kStageRows : stage + 1 == nk ? min(ragged, kStageRows) : 0; };
    auto clear_from = [&](int row, int buf) {
        for (int c = threadIdx.x; c < (kStageRows - row) * 32; c += 256) {
            const u32x4 z = {0u, 0u, 0u, 0u};
            *(u32x4*)(lds + buf * kTileBytes + row * 512 + c * 16) = z;
            *(u32x4*)(lds + kBBase + buf * kTileBytes + row * 512 + c * 16) = z;
        }
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    };

    // fetch addresses: [half of the eight rows][column block]
    uint32_t fa[2][TI], fb[2][TJ];
    {
        const int h = lane >> 4, s = lane & 15;
        auto fetch_at = [&](int a, int col) {
            return lds0 + (uint32_t)tile_offset<256>(8 * h + 4 * a + (s >> 2), col / 8 + ((s & 3) >> 1)) + ((s & 1) << 3);
        };
#pragma unroll
        for (int a = 0; a < 2; ++a) {
#pragma unroll
            for (int c = 0; c < TI; ++c) {
                fa[a][c] = fetch_at(a, (w & 1) * (TM / 2) + 16 * c);
                asm("" : "+v"(fa[a][c]));
            }
#pragma unroll
            for (int c = 0; c < TJ; ++c) {
                fb[a][c] = kBBase + fetch_at(a, (w >> 1) * 128 + 16 * c);
                asm("" : "+v"(fb[a][c]));
            }
        }
    }

    // (formed transposed: a lane then holds four neighbouring columns of a row of C)
    f32x4 acc[TI][TJ];
#pragma unroll
    for (int i = 0; i < TI; ++i)
#pragma unroll
        for (int j = 0; j < TJ; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    h16x8 va[2][TI], vb[2][TJ];
    auto fetch = [&](int set, int n, int buf) {
        if (n < TJ) vb[set][n] = fragment(fb[0][n], fb[1][n], buf * kTileBytes);
        else va[set][n - TJ] = fragment(fa[0][n - TJ], fa[1][n - TJ], buf * kTileBytes);
    };
    constexpr int kFetchEvery = TI * TJ / (TI + TJ) - (TM == 256);       // (in time for the next stage)
    // behind the MFMAs of stage s: the next but one has landed, and the buffer of the next, which the operand registers now hold, is
    // free for the stage four behind that one
    auto turn = [&](int s, int b) __attribute__((always_inline)) {
        if (s + kBuffers < nk) asm volatile("s_waitcnt vmcnt(16) lgkmcnt(0)\n\ts_barrier" ::: "memory");
        else asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
        if (rows_of(s + 2) < kStageRows) clear_from(rows_of(s + 2), (b + 2) % kBuffers);
        if (s + 1 + kBuffers < nk) request(s + 1 + kBuffers, (b + 1) % kBuffers);
    };
    if (nk > 0) {
#pragma unroll
        for (int s = 0; s < kBuffers; ++s)
            if (s < nk) request(s, s);
        if (nk >= 4) asm volatile("s_waitcnt vmcnt(24)\n\ts_barrier" ::: "memory");
        else asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
        if (rows_of(0) < kStageRows) clear_from(rows_of(0), 0);
#pragma unroll
        for (int n = 0; n < TI + TJ; ++n) fetch(0, n, 0);
        turn(-1, kBuffers - 1);
        // whole groups of four stages, so that the loop has one exit (several cost the compiler copies of the accumulators, 128
        // spilled registers); a last group is filled up with stages of zeros
        int s0 = 0;
        settled(acc);
        do {
#pragma unroll
            for (int b = 0; b < kBuffers; ++b) {
#pragma unroll
                for (int n = 0; n < TI * TJ; ++n) {
                    mfma16_in_place(vb[b & 1][n % TJ], va[b & 1][n / TJ], acc[n / TJ][n % TJ]);
                    if (n % kFetchEvery == 0 && n / kFetchEvery < TI + TJ) fetch(~b & 1, n / kFetchEvery, (b + 1) % kBuffers);
                    __builtin_amdgcn_sched_barrier(0);
                }
                turn(s0 + b, b);
            }
            s0 += kBuffers;
        } while (s0 < nk);
        settled(acc);
    }

    // columns 4 * (lane / 16) .. + 3 of a block, row lane % 16 of it
    float* out = (gridDim.y == 1 ? g.out : g.partial + (int64_t)blockIdx.y * g.total) + pr.at;
#pragma unroll
    for (int i = 0; i < TI; ++i) {
        const int row = m0 + (w & 1) * (TM / 2) + i * 16 + (lane & 15);
#pragma unroll
        for (int j = 0; j < TJ; ++j) {
            const int col = n0 + (w >> 1) * 128 + j * 16 + 4 * (lane >> 4);
            if (row < pr.m && col < pr.n) *(f32x4*)(out + (int64_t)row * pr.n + col) = acc[i][j];
        }
    }
}

// ---------------------------------------------------------------------------------------------------- projections
// Y[t][n] = sum over k of X[t][k] * W[n][k] for token rows t, or W[k][n] (kRowsW: the product of a backward), 16-bit operands,
// fp32 sums, and what the model does with Y in the same pass (Epilogue).
//
using sba_model::Projection;

// What becomes of a wave's products: blocks of 16 features (TI of them; with swiglu TI/2 of gates, then their ups) by 16 tokens
// (TJ), lane l holding features 4 * (l / 16) .. + 3 of token l % 16 of each.  Rows leave straight from the registers: two blocks'
// 16-bit halves trade places between neighbouring sixteenths of the wave (v_permlane16_swap), after which a lane holds eight
// consecutive features of one block and four lanes 64 bytes of a token's row; in fp32 they do so as they are.  (Through LDS, in whole
// 128-byte lines, the stores of a 128 x 256 tile took 3 us with nothing beside them.)
// The residual, or gate and up of the backward, can be asked for ahead (`request`, TI loads per 16 tokens, every lane's within the
// tensor whatever the tile's edge, so that their number is known to the waits of the caller).
template <int kEpi, int TI, int TJ> struct Results {
    static constexpr bool kPart = kEpi == sba_model::kPartialSums;
    static constexpr bool kAdd = kEpi == sba_model::kAddResidual, kGlu = kEpi == sba_model::kSwigluFwd, kGluBwd = kEpi == sba_model::kSwigluBwd;
    static constexpr int kAhead = kAdd || kGluBwd ? TI : 0;        // loads per 16 tokens
    static constexpr int kStores = kAdd || kPart || kGluBwd ? TI : kGlu ? TI / 4 : TI / 2;      // stores per 16 tokens (at least)
    u32x4 ahead[TJ][kAhead ? kAhead : 1];
    int tok0, f0, h;               // this lane's first token; its features of block or pair 0

    // (the lane's indices from a copy that the compiler cannot see through: what is made of them would otherwise be worked out ahead of
    // the caller's loops and kept, 70 spilled registers)
    __device__ inline void aim(int lane, int tw, int nw) {
        asm volatile("" : "+v"(lane));
        h = lane >> 4;
        tok0 = tw + (lane & 15);
        f0 = nw + (kAdd || kPart ? 4 * h : (h & 1) * 16 + (h >> 1) * 8);
    }
    __device__ inline void request(const Projection& p, int j) {
        const int64_t tok = min(tok0 + 16 * j, p.m - 1);
#pragma unroll
        for (int i = 0; i < kAhead; ++i) {
            if (kAdd) ahead[j][i] = *(const u32x4*)(p.residual + tok * p.n + min(f0 + 16 * i, p.n - 4));
            else ahead[j][i] = *(const u32x4*)((const elem16*)p.pre + tok * 2 * p.n + min(f0 + 32 * (i / 2), p.n - 8) + (i & 1) * p.n);
        }
    }
    // features of block a and the block behind it, as 16-bit: eight consecutive ones a lane
    __device__ static inline h16x8 rows_of(const f32x4& a, const f32x4& b) {
        auto two = [](float x, float y) { return __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2{x, y}), h16x2)); };
        typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
        const u32x2 lo = __builtin_amdgcn_permlane16_swap(two(a[0], a[1]), two(b[0], b[1]), false, false);
        const u32x2 hi = __builtin_amdgcn_permlane16_swap(two(a[2], a[3]), two(b[2], b[3]), false, false);
        return __builtin_bit_cast(h16x8, (u32x4{lo[0], hi[0], lo[1], hi[1]}));
    }
    __device__ inline void store(const Projection& p, const f32x4 (&acc)[TI][TJ], int j) const {
        const int tok = tok0 + 16 * j, width = kGlu ? p.n / 2 : p.n;
        const int64_t row = (int64_t)tok * width;
        if (kAdd || kPart) {
            float* const out = kPart ? p.partial + (int64_t)blockIdx.y * p.m * p.n : (float*)p.out;
#pragma unroll
            for (int i = 0; i < TI; ++i)
                if (tok < p.m && f0 + 16 * i < p.n)
                    *(f32x4*)(out + row + f0 + 16 * i) = kPart ? acc[i][j] : __builtin_bit_cast(f32x4, ahead[j][i]) + acc[i][j];
            return;
        }
#pragma unroll
        for (int q = 0; q < (kGlu ? TI / 4 : TI / 2); ++q) {
            const int n = f0 + 32 * q;
            const h16x8 y = rows_of(acc[2 * q][j], acc[2 * q + 1][j]);
            if (kGlu) {
                const h16x8 u = rows_of(acc[TI / 2 + 2 * q][j], acc[TI / 2 + 2 * q + 1][j]);
                if (tok >= p.m || n >= width) continue;
                h16x8 o;
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    const float g = (float)y[e];
                    o[e] = (elem16)((float)(elem16)(g / (1.f + __expf(-g))) * (float)u[e]);
                }
                *(h16x8*)((elem16*)p.out + row + n) = o;
                if (p.pre) {
                    *(h16x8*)((elem16*)p.pre + 2 * row + n) = y;
                    *(h16x8*)((elem16*)p.pre + 2 * row + width + n) = u;
                }
            } else if (kGluBwd) {
                // y is the gradient of silu(gate) * up
                if (tok >= p.m || n >= width) continue;
                const h16x8 g = __builtin_bit_cast(h16x8, ahead[j][2 * q]), u = __builtin_bit_cast(h16x8, ahead[j][2 * q + 1]);
                h16x8 dg, du;
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    const float gf = (float)g[e], df = (float)y[e], sg = 1.f / (1.f + __expf(-gf));
                    du[e] = (elem16)(df * (float)(elem16)(gf * sg));
                    dg[e] = (elem16)((float)(elem16)(df * (float)u[e]) * sg * (1.f + gf * (1.f - sg)));
                }
                *(h16x8*)((elem16*)p.out + 2 * row + n) = dg;
                *(h16x8*)((elem16*)p.out + 2 * row + width + n) = du;
            } else if (tok < p.m && n < width) {
                *(h16x8*)((elem16*)p.out + row + n) = y;
            }
        }
    }
};


// Launches that are short of tiles: T x T tiles, kPerCu workgroups a CU, each of G groups of four waves (two by two, T/2 tokens x T/2
// features each) that share out the contraction: group g takes stages g, g + G, ...  The groups' fp32 sums meet in LDS, in the order of
// the groups, and as many groups as there are blocks of tokens write the results.  k a multiple of 32.
// Stages of 64 k, NB buffers a group, walked slice by slice as in the kernel for large products below.  Rows of 64 k are whole 128-byte
// lines: with 32 k the CU's memory pipe takes 16 lines for a kilobyte instead of 8, and 4096 x 1024, k = 2816, with the residual took 34 us (31
// now; four buffers of 32 k and one group, the shape before this: 37).  What bounds them: LDS, 128 bytes a cycle for the operands of 64 x 64
// products a wave and the arriving tiles (T = 128); the round trip to memory, 1.5 us with every CU asking (T = 64), which is what two
// stages more on their way are for: 1024 x 768, k = 4096, with four groups of two buffers 27 us inside a training step, with two groups of
// four 21; 2048 x 1024 with the residual, k = 1024, with two workgroups of two groups a CU 9.7, with three of one group and three buffers 9.3.
// A tile row of 64 k is eight 16-byte chunks; chunk c of row r lies at c ^ (r / 2 % 8), so that sixteen consecutive rows' chunks of one index
// fall on sixteen different bank groups.  The products are formed transposed (rows: features, columns: tokens).
template <int T, int G, int NB, int kPerCu, bool kRowsW, int kEpi>
__global__ __launch_bounds__(256 * G, G * kPerCu) void projection_kernel(Projection p) {
    constexpr int KS = 64;                                             // k of a stage
    constexpr bool kPadded = NB == 2;                                  // whole groups of turns, filled up with zeros
    constexpr int kX = T * KS * 2, kStage = 2 * kX;                    // bytes
    constexpr int PX = T / 32;                                         // copies of one operand per wave and stage
    constexpr int C = KS / 8;                                          // 16-byte chunks of a row of k
    constexpr int TI = T / 32, TJ = T / 32;                            // 16-wide blocks of a wave: features, tokens
    static_assert(kEpi != sba_model::kSwigluFwd || T == 128, "pairs of gate blocks");
    __shared__ __attribute__((aligned(1024))) char lds[G * NB * kStage];
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) & 3;
    const int group = __builtin_amdgcn_readfirstlane(threadIdx.x >> 8);
    const int m = lane & 15, h = lane >> 4;

    // a swiglu tile's features are T/2 gates and the T/2 ups that go with them
    constexpr bool kGlu = kEpi == sba_model::kSwigluFwd;
    const int features = kGlu ? p.n / 2 : p.n;
    constexpr int kOwn = kGlu ? T / 2 : T;
    const int tiles_m = (p.m + T - 1) / T, tiles_n = (features + kOwn - 1) / kOwn, tiles = tiles_m * tiles_n;
    const int per = (tiles + 7) / 8, t = (int)(blockIdx.x & 7) * per + (int)(blockIdx.x >> 3);
    if ((int)(blockIdx.x >> 3) >= per || t >= tiles) return;
    constexpr int kBand = 1024 / T;
    const int band = t / (kBand * tiles_n), rows = min(kBand, tiles_m - kBand * band), in = t - band * kBand * tiles_n;
    const int t0 = (kBand * band + in % rows) * T, n0 = (in / rows) * kOwn;
    const int stages = (p.k + KS - 1) / KS, turns = (stages + G - 1) / G, padded = kPadded ? (turns + NB - 1) / NB * NB : turns;
    const int nk = (stages + G - 1 - group) / G;                       // this group's stages: group, group + G, ...
    const bool odd = p.k % KS != 0;                                    // the last stage is half a one ...
    const int half_stage = odd && (stages - 1) % G == group ? nk - 1 : -1;      // ... and this group's, this turn's

    const char* xat = (const char*)p.x + 2 * (int64_t)t0 * p.ldx + 2 * KS * group;
    const char* wat = (const char*)p.w + (kRowsW ? 2 * (int64_t)n0 + 2 * KS * group * p.ldw : (int64_t)2 * KS * group);
    // chunk swizzle of W's rows of T columns: the transposing fetch of half a wave reads rows r .. r + 3 and r + 8 .. r + 11, two
    // neighbouring chunks of each, from 64 banks
    auto col_swz = [](int row) { return T == 64 ? (row & 2) | ((row >> 1) & 4) : swz<128>(row); };
    // and of rows of k: sixteen consecutive rows' chunks of one index fall on sixteen different bank groups
    auto row_swz = [](int row) { return row / (16 / C) % C; };
    uint32_t xoff[PX], woff[PX];
    auto aim = [&](int lane, bool half) {      // half: the second half of a stage does not exist and reads the first once more
        const int last_c = half ? C / 2 - 1 : C - 1;
#pragma unroll
        for (int i = 0; i < PX; ++i) {
            const int row = 64 / C * (w + 4 * i) + lane / C, c = (lane % C ^ row_swz(row)) & last_c;
            xoff[i] = (uint32_t)min(row, p.m - 1 - t0) * (uint32_t)(2 * p.ldx) + 16u * c;
            if (kRowsW) {
                constexpr int kPer = 512 / T;                  // rows of T columns per copy
                const int k = kPer * (w + 4 * i) + lane / (T / 8), cc = (lane & (T / 8 - 1)) ^ col_swz(k);
                woff[i] = (uint32_t)(half ? k & 31 : k) * (uint32_t)(2 * p.ldw) + 16u * (uint32_t)min(cc, (features - n0) / 8 - 1);
            } else {
                int feature = n0 + row, up = 0;
                if (kGlu) {                                    // a wave's half of the tile: T/4 gates, then their ups
                    feature = n0 + (row / (T / 2)) * (T / 4) + row % (T / 4);
                    up = (row % (T / 2)) / (T / 4) * features;
                }
                woff[i] = (uint32_t)(min(feature, features - 1) + up) * (uint32_t)(2 * p.ldw) + 16u * c;
            }
        }
    };
    aim(lane, half_stage == 0);
    const uint32_t lds0 = lds_address(lds) + group * NB * kStage;
    auto request = [&](int stage, int buf) {
        if (stage == half_stage && stage > 0) {                // (the last one: nothing is aimed at after it)
            int lane_here = lane;
            asm volatile("" : "+v"(lane_here));
            aim(lane_here, true);
        }
#pragma unroll
        for (int i = 0; i < PX; ++i) dma16(xat, xoff[i], lds0 + buf * kStage + (w + 4 * i) * 1024);
#pragma unroll
        for (int i = 0; i < PX; ++i) dma16(wat, woff[i], lds0 + buf * kStage + kX + (w + 4 * i) * 1024);
        xat += 2 * KS * G;
        wat += kRowsW ? 2 * KS * G * p.ldw : (int64_t)2 * KS * G;
    };
    // zeros in place of a stage, or of its second half, that does not exist
    auto clear = [&](int stage, int buf) {
        if (stage < nk && stage != half_stage) return;
        char* at = lds + (group * NB + buf) * kStage;
        for (int c = threadIdx.x & 255; c < kStage / 16; c += 256) {
            const int row = c % (kX / 16) / C;
            const bool second = kRowsW && c >= kX / 16 ? c - kX / 16 >= kX / 32 : (c % C ^ row_swz(row)) >= C / 2;
            if (stage >= nk || second) *(u32x4*)(at + c * 16) = u32x4{0u, 0u, 0u, 0u};
        }
    };

    // fetch addresses: X rows and, k contiguous, W rows [slice]; W columns [half of the eight rows][column block]
    uint32_t fx[2], fw[2], fc[2][TI];
#pragma unroll
    for (int q = 0; q < 2; ++q) {
        const int c = (4 * q + h) ^ row_swz(m);
        fx[q] = lds0 + ((w & 1) * (T / 2) + m) * (KS * 2) + c * 16;
        fw[q] = lds0 + kX + ((w >> 1) * (T / 2) + m) * (KS * 2) + c * 16;
        asm("" : "+v"(fx[q]), "+v"(fw[q]));
    }
    if (kRowsW) {
#pragma unroll
        for (int a = 0; a < 2; ++a)
#pragma unroll
            for (int c = 0; c < TI; ++c) {
                const int row = 8 * h + 4 * a + (m >> 2), chunk = (w >> 1) * (T / 16) + 2 * c + ((m & 3) >> 1);
                fc[a][c] = lds0 + kX + row * (T * 2) + ((chunk ^ col_swz(row)) << 4) + ((m & 1) << 3);
                asm("" : "+v"(fc[a][c]));
            }
    }
    auto at = [](uint32_t base, int imm) {
        return *(const __attribute__((address_space(3))) h16x8*)((__attribute__((address_space(3))) char*)(uintptr_t)base + imm);
    };

    f32x4 acc[TI][TJ];
#pragma unroll
    for (int i = 0; i < TI; ++i)
#pragma unroll
        for (int j = 0; j < TJ; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    h16x8 vx[2][TJ], vw[2][TI];
    // the n-th of the operands of slice q (32 k) of buffer `buf`, into one of the two sets of registers
    auto fetch = [&](int set, int n, int buf, int q) {
        if (n < TJ) vx[set][n] = at(fx[q], buf * kStage + n * 16 * KS * 2);
        else if (kRowsW) vw[set][n - TJ] = fragment(fc[0][n - TJ], fc[1][n - TJ], buf * kStage + q * 32 * T * 2);
        else vw[set][n - TJ] = at(fw[q], buf * kStage + (n - TJ) * 16 * KS * 2);
    };
    constexpr int kFetchEvery = TI * TJ / (TI + TJ);
    // MFMAs of the slice in register set `set`; under them the fetches of slice q of buffer `buf`, which is the one behind it
    auto slice = [&](int set, int buf, int q) __attribute__((always_inline)) {
#pragma unroll
        for (int n = 0; n < TI * TJ; ++n) {
            acc[n / TJ][n % TJ] = mfma16(vw[set][n / TJ], vx[set][n % TJ], acc[n / TJ][n % TJ]);
            if (n % kFetchEvery == 0 && n / kFetchEvery < TI + TJ) fetch(set ^ 1, n / kFetchEvery, buf, q);
            __builtin_amdgcn_sched_barrier(0);
        }
    };

    // Token blocks whose results this group finishes, summed over the groups: the first E groups, TJ / E blocks each.
    constexpr int E = G < TJ ? G : TJ, J = TJ / E;
    // What the epilogue reads is asked for in the last group of turns, behind all copies; where registers are short, half of it.
    constexpr int kEarly = G == 1 ? J / 2 : J;
    Results<kEpi, TI, J> res;
    constexpr int R = Results<kEpi, TI, J>::kAhead * kEarly;
    // Stage s is all in operand registers: its buffer b is free for stage s + NB, and the next stage has landed.  Stages that a group
    // does not have are made with zeros.
    auto turn = [&](int s, int b, bool asked) __attribute__((always_inline)) {
        if (asked && R) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" : : "n"(R) : "memory");
        else if (s + NB <= nk) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" : : "n"((NB - 2) * 2 * PX) : "memory");
        else asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
        if (s + 1 < padded && s + 1 >= stages / G - odd) {             // (some group may lack it: the same for all of them)
            clear(s + 1, (b + 1) % NB);
            asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        }
        if (s + NB < nk) request(s + NB, b);
    };

    res.aim(lane, t0 + (w & 1) * (T / 2) + 16 * J * (group % E), n0 + (w >> 1) * (kOwn / 2));
#pragma unroll
    for (int s = 0; s < NB; ++s)
        if (s < nk) request(s, s);
    if (nk >= NB) asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" : : "n"((NB - 1) * 2 * PX) : "memory");
    else asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
    if (stages < G + odd) {
        clear(0, 0);
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    }
#pragma unroll
    for (int n = 0; n < TI + TJ; ++n) fetch(0, n, 0, 0);
    for (int s0 = 0; s0 < turns; s0 += NB) {   // (filled up with zeros where an exit in between would cost copies of the sums)
        const bool asked = s0 + NB >= turns && group < E;      // (all copies are on their way by then)
        if (R && asked) {
#pragma unroll
            for (int j = 0; j < kEarly; ++j) res.request(p, j);
        }
#pragma unroll
        for (int b = 0; b < NB; ++b) {
            if (!kPadded && b > 0 && s0 + b >= turns) break;
            slice(0, b, 1);
            turn(s0 + b, b, asked);
            slice(1, (b + 1) % NB, 0);
        }
    }
    if constexpr (G == 1) {
        if (R) {
#pragma unroll
            for (int j = kEarly; j < J; ++j) res.request(p, j);
        }
#pragma unroll
        for (int j = 0; j < TJ; ++j) res.store(p, acc, j);
        return;
    }
    // the groups' sums meet in LDS: [group][wave][block][lane]
    auto part = [&](int g, int i, int j) { return (f32x4*)(lds + (((g * 4 + w) * TI + i) * TJ + j) * 1024 + lane * 16); };
    static_assert(G * 4 * TI * TJ * 1024 <= G * NB * kStage, "partial sums in the tiles' place");
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");      // (the last slice's fetches)
#pragma unroll
    for (int i = 0; i < TI; ++i)
#pragma unroll
        for (int j = 0; j < TJ; ++j) *part(group, i, j) = acc[i][j];
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    if (group >= E) return;
    f32x4 sum[TI][J];
#pragma unroll
    for (int i = 0; i < TI; ++i)
#pragma unroll
        for (int j = 0; j < J; ++j) {
            sum[i][j] = *part(0, i, group * J + j);
#pragma unroll
            for (int g = 1; g < G; ++g) sum[i][j] += *part(g, i, group * J + j);
        }
#pragma unroll
    for (int j = 0; j < J; ++j) res.store(p, sum, j);
}

// Large products: TM x 256 tiles, one resident workgroup a CU that walks tiles, one wave per SIMD with TM/2 x 128 of a tile.
// Stages of 64 k: rows of 64 k are whole 128-byte lines (with 32 k every line is fetched twice: -12 %).  A stage is four slices of
// TM/16 MFMAs a wave; the operands of a slice are fetched under the MFMAs of the one before.  After the third slice the waves meet:
// the stage's buffer has been read, the next stage has landed, and the copies of the stage NB ahead start into it, spread over the
// slices that follow (all under one they ask for 1024 cycles of the CU's memory pipe in 544 of MFMAs: 1.09 of the time per stage,
// which with 256 rows and every CU busy is 1.33 us in products of 90 us and 1.56 in products of 400, where the chip's power limit has
// taken the clock down).  The copies run through the list of (tile, stage) pairs without a break, so a tile's results are stored while
// the next tile's first stages arrive.  TM = 256 has two buffers of 64 KB, TM = 128, whose stages pass in half the time, three of
// 48 KB; the fetch addresses move from buffer to buffer, one add per address and stage.
// 8192 tokens, k = 1024: 5632 features with swiglu in 92 us with TM = 256 (1.03 PFLOP/s; 99 with 128, 102 in 128 x 128 tiles), 3072 features in
// 47 with TM = 128 (49; 50); k = 5632, W's rows: 1024 features in 79.6 with TM = 128 (103.5; 79.2).
template <int TM, bool kRowsW, int kEpi>
__global__ __launch_bounds__(256, 1) void large_projection_kernel(Projection p) {
    constexpr int NB = TM == 256 ? 2 : 3;
    constexpr int kX = TM * 128, kStage = kX + 256 * 128;
    constexpr int PX = TM / 32, P = PX + 8;                    // copies per wave and stage
    constexpr int TI = 8, TJ = TM / 32, kSlots = TI * TJ;       // blocks of 16 features and tokens of a wave; MFMAs of a slice
    __shared__ __attribute__((aligned(1024))) char lds[NB * kStage];
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int m = lane & 15, h = lane >> 4;
    constexpr bool kGlu = kEpi == sba_model::kSwigluFwd;
    const int features = kGlu ? p.n / 2 : p.n;
    constexpr int kOwn = kGlu ? 128 : 256;
    const int tiles_m = (p.m + TM - 1) / TM, tiles_n = (features + kOwn - 1) / kOwn, tiles = tiles_m * tiles_n;
    // every XCD takes a run of neighbouring tiles (bands of 1024 tokens, feature tile by feature tile); its workgroups walk it
    // side by side
    const int per = (tiles + 7) / 8, stride = (int)gridDim.x >> 3, run0 = (int)(blockIdx.x & 7) * per;
    const int run = min(per, tiles - run0);
    int local = (int)(blockIdx.x >> 3);
    if (local >= run) return;
    auto tile_at = [&](int l, int& t0, int& n0) {
        constexpr int kBand = 1024 / TM;
        const int t = run0 + l, band = t / (kBand * tiles_n), rows = min(kBand, tiles_m - kBand * band), in = t - band * kBand * tiles_n;
        t0 = (kBand * band + in % rows) * TM;
        n0 = (in / rows) * kOwn;
    };
    // kPartialSums: blockIdx.y's share of the stages
    const int share = kEpi == sba_model::kPartialSums ? (p.k / 64 + p.splits - 1) / p.splits : 0, first = share * (int)blockIdx.y;
    const int nk = share ? min(share, p.k / 64 - first) : p.k / 64;

    // ---- the stream of copies
    const char *xat, *wat;
    const int64_t wstep = kRowsW ? 128 * p.ldw : (int64_t)128;
    uint32_t xoff[PX], woff[8];
    int d_local = local, d_stage = 0;
    uint32_t d_lds = lds_address(lds) + w * 1024;
    auto aim = [&](int l) {
        int t0, n0;
        tile_at(l, t0, n0);
        xat = (const char*)p.x + 2 * (int64_t)t0 * p.ldx + 128 * (int64_t)first;
        wat = (const char*)p.w + (kRowsW ? 2 * (int64_t)n0 + first * wstep : (int64_t)0);
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const int row = 8 * (w + 4 * i) + (lane >> 3), c = (lane & 7) ^ ((row >> 1) & 7);
            if (i < PX) xoff[i] = (uint32_t)min(row, p.m - 1 - t0) * (uint32_t)(2 * p.ldx) + 16u * c;
            if (kRowsW) {
                const int k = 2 * (w + 4 * i) + (lane >> 5), cc = (lane & 31) ^ swz<256>(k);
                woff[i] = (uint32_t)k * (uint32_t)(2 * p.ldw) + 16u * (uint32_t)min(cc, (features - n0) / 8 - 1);
            } else {
                int feature = n0 + row, up = 0;
                if (kGlu) {                                    // a wave's half of the tile: 64 gates, then their ups
                    feature = n0 + (row >> 7) * 64 + (row & 63);
                    up = ((row >> 6) & 1) * features;
                }
                woff[i] = (uint32_t)(min(feature, features - 1) + up) * (uint32_t)(2 * p.ldw) + 16u * c;
            }
        }
    };
    const uint32_t lds_end = lds_address(lds) + w * 1024 + NB * kStage;
    auto next_stage = [&]() {
        xat += 128;
        wat += wstep;
        d_lds += kStage;
        if (d_lds == lds_end) d_lds -= NB * kStage;
        if (++d_stage == nk) {
            d_stage = 0;
            if (d_local + stride < run) d_local += stride;     // (behind the last tile: once more through it, unread)
            aim(d_local);
        }
    };
    auto copy = [&](int i) {
        if (i < PX) dma16(xat, xoff[i], d_lds + i * 4096);
        else dma16(wat, woff[i - PX], d_lds + kX + (i - PX) * 4096);
    };

    // ---- operand fetches: X rows and, k contiguous, W rows [slice]; W columns [half of the eight rows][column block]
    uint32_t fx[2], fw[2], fc[2][TI];
    const uint32_t lds0 = lds_address(lds);
#pragma unroll
    for (int q = 0; q < 2; ++q) {
        const int c = (4 * q + h) ^ ((m >> 1) & 7);
        fx[q] = lds0 + (w & 1) * (TM / 2) * 128 + m * 128 + c * 16;
        fw[q] = lds0 + kX + (w >> 1) * 128 * 128 + m * 128 + c * 16;
        asm("" : "+v"(fx[q]), "+v"(fw[q]));
    }
    if (kRowsW) {
#pragma unroll
        for (int a = 0; a < 2; ++a)
#pragma unroll
            for (int c = 0; c < TI; ++c) {
                fc[a][c] = lds0 + kX + (uint32_t)tile_offset<256>(8 * h + 4 * a + (m >> 2), (w >> 1) * 16 + 2 * c + ((m & 3) >> 1)) + ((m & 1) << 3);
                asm("" : "+v"(fc[a][c]));
            }
    }
    int f_buf = 0;
    auto next_buffer = [&]() {
        f_buf = f_buf + 1 == NB ? 0 : f_buf + 1;
        uint32_t by = f_buf == 0 ? (uint32_t)-((NB - 1) * kStage) : (uint32_t)kStage;
        asm("" : "+s"(by));
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            fx[q] += by;
            if (!kRowsW) fw[q] += by;
        }
        if (kRowsW) {
#pragma unroll
            for (int a = 0; a < 2; ++a)
#pragma unroll
                for (int c = 0; c < TI; ++c) fc[a][c] += by;
        }
    };
    auto at = [](uint32_t base, int imm) {
        return *(const __attribute__((address_space(3))) h16x8*)((__attribute__((address_space(3))) char*)(uintptr_t)base + imm);
    };
    h16x8 vx[2][TJ], vw[2][TI];
    auto fetch = [&](int set, int n, int q) {
        if (n < TJ) vx[set][n] = at(fx[q], n * 2048);
        else if (n < TJ + TI) {
            const int i = n - TJ;
            if (kRowsW) vw[set][i] = fragment(fc[0][i], fc[1][i], q * 32 * 512);
            else vw[set][i] = at(fw[q], i * 2048);
        }
    };
    f32x4 acc[TI][TJ];
    // MFMAs of one slice; under them the fetches of slice q and copies first .. first + count - 1
    constexpr int kFetchEvery = TM == 256 ? 3 : 2, kCopyEvery = 4;
    static_assert((TJ + TI) * kFetchEvery <= kSlots, "the fetches of a slice under the MFMAs of the one before");
    auto slice = [&](int cur, int q, int first, int count, bool fresh = false) __attribute__((always_inline)) {
#pragma unroll
        for (int n = 0; n < kSlots; ++n) {
            acc[n / TJ][n % TJ] = mfma16(vw[cur][n / TJ], vx[cur][n % TJ], fresh ? f32x4{0.f, 0.f, 0.f, 0.f} : acc[n / TJ][n % TJ]);
            if (n % kFetchEvery == 0) fetch(cur ^ 1, n / kFetchEvery, q);
            if (n % kCopyEvery == kCopyEvery - 1 && n / kCopyEvery < count) copy(first + n / kCopyEvery);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    // which slices the copies of a stage go under: TM = 256 the second, 128 both
    constexpr int C1 = TM == 256 ? 16 : 6, C0 = P - C1;
    static_assert(C1 <= kSlots / kCopyEvery && C0 <= kSlots / kCopyEvery, "copies of a slice");

    // ---- results
    // With one wave per SIMD nobody else has work while a load is on its way: what the epilogue reads is asked for before the tile's
    // last slice.
    Results<kEpi, TI, TJ> res;
    constexpr int kAhead = Results<kEpi, TI, TJ>::kAhead;
    auto request = [&](int t0, int n0) __attribute__((always_inline)) {
        res.aim(lane, t0 + (w & 1) * (TM / 2), n0 + (w >> 1) * (kOwn / 2));
        if (kAhead) {
#pragma unroll
            for (int j = 0; j < TJ; ++j) res.request(p, j);
        }
    };

    aim(local);
#pragma unroll
    for (int s = 0; s < NB; ++s) {
#pragma unroll
        for (int i = 0; i < P; ++i) copy(i);
        next_stage();
    }
    asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" : : "n"((NB - 1) * P) : "memory");
#pragma unroll
    for (int n = 0; n < TJ + TI; ++n) fetch(0, n, 0);
    // The stores of a tile lie in the queue behind the copies of the next tile's first NB stages, so its first wait can leave them
    // there - if the tile was a whole one, which is sure to have issued all of them.
    constexpr int kStores = Results<kEpi, TI, TJ>::kStores * TJ;
    constexpr int kLeave = (NB - 2) * P + kStores < 63 ? (NB - 2) * P + kStores : 63;           // (63: the most a wait can leave)
    bool stores_behind = false;
    for (; local < run; local += stride) {
        int t0, n0;
        tile_at(local, t0, n0);
        slice(0, 1, 0, 0, true);
        if (stores_behind) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" : : "n"(kLeave) : "memory");
        else asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" : : "n"((NB - 2) * P) : "memory");
        next_buffer();
        for (int s = 1; s < nk; ++s) {
            slice(1, 0, 0, C1);
            slice(0, 1, C1, C0);
            next_stage();
            asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" : : "n"((NB - 2) * P) : "memory");
            next_buffer();
        }
        request(t0, n0);
        slice(1, 0, 0, C1);
#pragma unroll
        for (int i = C1; i < P; ++i) copy(i);
        next_stage();
#pragma unroll
        for (int j = 0; j < TJ; ++j) res.store(p, acc, j);
        stores_behind = t0 + TM <= p.m && n0 + kOwn <= features;
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");           // the last copies, unread, have landed before the LDS is given back
}

template <int T, int G, int NB, int kPerCu>
int launch_projection(const Projection& p, hipStream_t s) {
    const int own = p.epilogue == sba_model::kSwigluFwd ? T / 2 : T, features = p.epilogue == sba_model::kSwigluFwd ? p.n / 2 : p.n;
    const int tiles = ((p.m + T - 1) / T) * ((features + own - 1) / own);
    const dim3 grid((unsigned)((tiles + 7) / 8 * 8)), block(256 * G);
    if (p.rows_w) {
        if (p.epilogue == sba_model::kSwigluBwd) hipLaunchKernelGGL((projection_kernel<T, G, NB, kPerCu, true, sba_model::kSwigluBwd>), grid, block, 0, s, p);
        else if (p.epilogue == sba_model::kStore) hipLaunchKernelGGL((projection_kernel<T, G, NB, kPerCu, true, sba_model::kStore>), grid, block, 0, s, p);
        else return -2;
    } else {
        if (p.epilogue == sba_model::kSwigluFwd) {
            if constexpr (T == 128) hipLaunchKernelGGL((projection_kernel<T, G, NB, kPerCu, false, sba_model::kSwigluFwd>), grid, block, 0, s, p);
            else return -2;                    // (swiglu pairs two blocks of gates)
        } else if (p.epilogue == sba_model::kAddResidual) hipLaunchKernelGGL((projection_kernel<T, G, NB, kPerCu, false, sba_model::kAddResidual>), grid, block, 0, s, p);
        else if (p.epilogue == sba_model::kStore) hipLaunchKernelGGL((projection_kernel<T, G, NB, kPerCu, false, sba_model::kStore>), grid, block, 0, s, p);
        else return -2;
    }
    return hipGetLastError() == hipSuccess ? 0 : -6;
}

template <int TM>
int launch_large_projection(const Projection& p, hipStream_t s) {
    const int own = p.epilogue == sba_model::kSwigluFwd ? 128 : 256, features = p.epilogue == sba_model::kSwigluFwd ? p.n / 2 : p.n;
    const int tiles = ((p.m + TM - 1) / TM) * ((features + own - 1) / own), cus = sba_cu_count() & ~7;
    const dim3 grid((unsigned)(((tiles < cus ? tiles : cus) + 7) & ~7)), block(256);
    if (p.splits > 1) {
        if (!p.rows_w || p.epilogue != sba_model::kStore) return -2;
        hipLaunchKernelGGL((large_projection_kernel<TM, true, sba_model::kPartialSums>), dim3(grid.x, (unsigned)p.splits), block, 0, s, p);
    } else if (p.rows_w) {
        if (p.epilogue == sba_model::kStore) hipLaunchKernelGGL((large_projection_kernel<TM, true, sba_model::kStore>), grid, block, 0, s, p);
        else return -2;
    } else {
        if (p.epilogue == sba_model::kAddResidual && TM == 128) hipLaunchKernelGGL((large_projection_kernel<128, false, sba_model::kAddResidual>), grid, block, 0, s, p);
        else if (p.epilogue == sba_model::kSwigluFwd) hipLaunchKernelGGL((large_projection_kernel<TM, false, sba_model::kSwigluFwd>), grid, block, 0, s, p);
        else if (p.epilogue == sba_model::kStore) hipLaunchKernelGGL((large_projection_kernel<TM, false, sba_model::kStore>), grid, block, 0, s, p);
        else return -2;
    }
    return hipGetLastError() == hipSuccess ? 0 : -6;
}

}  // namespace
}  // namespace sba

#ifdef SBA_ELEM_F16
#define SBA_WEIGHT_GRADS weight_grads_f16
#define SBA_PROJECT project_f16
#else
#define SBA_WEIGHT_GRADS weight_grads_bf16
#define SBA_PROJECT project_bf16
#endif
namespace sba_model {
int SBA_PROJECT(const Projection& p, ProjectionTile tile, hipStream_t s) {
    using namespace sba::SBA_ELEM_NS;
    if (tile == kTile256) return launch_large_projection<256>(p, s);
    if (tile == kTile128x256) return launch_large_projection<128>(p, s);
    if (tile == kTile128Halves) return launch_projection<128, 2, 2, 1>(p, s);
    if (tile == kTile64) return launch_projection<64, 1, 3, 3>(p, s);
    if (tile == kTile64Halves) return launch_projection<64, 2, 4, 1>(p, s);
    return launch_projection<128, 1, 2, 2>(p, s);
}
int SBA_WEIGHT_GRADS(const WeightGrads& g, int splits, hipStream_t stream) {
    const dim3 grid((unsigned)((g.tiles + 7) / 8 * 8), (unsigned)splits), block(256);
    if (g.tile_rows == 256) hipLaunchKernelGGL(sba::SBA_ELEM_NS::weight_grad_kernel<256>, grid, block, 0, stream, g);
    else hipLaunchKernelGGL(sba::SBA_ELEM_NS::weight_grad_kernel<224>, grid, block, 0, stream, g);
    return hipGetLastError() == hipSuccess ? 0 : -6;
}
}  // namespace sba_model
