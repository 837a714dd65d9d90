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

// A workgroup of four waves, one per SIMD, owns a 256 x 256 tile of C; a wave holds 128 x 128 of it (sixteen 32 x 32
// accumulators, 256 registers).  That is the shape at which the LDS keeps up: per 16 rows of the contraction a wave reads eight
// operand fragments for sixteen MFMAs, so the four waves' reads (32 KB) and the arriving tiles (16 KB) take 384 of the 544
// cycles that the MFMAs do; eight waves of 128 x 64 would ask for 48 + 16 KB.
// Both operands have the contracted index in rows, so every fragment is a transposing fetch (ds_read_b64_tr_b16).
// Stages of 32 rows, four tile buffers.  In a stage's first half the second half's operands are fetched, then the waves meet
// once: the buffer is free for stage s + 4 (requested at once, three and a half stages ahead of its use) and stage s + 1 is
// known to have landed, whose first operands are fetched under the second half's MFMAs.
constexpr int kTileM = 256, kTileN = 256, kStageRows = 32, kBuffers = 4;
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

__global__ __launch_bounds__(256, 1) void weight_grad_kernel(sba_model::WeightGrads g) {
    __shared__ __attribute__((aligned(1024))) char lds[2 * kBuffers * kTileBytes];
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);

    // workgroups are dealt to the eight XCDs in turn: each takes a run of neighbouring tiles, whose operands its L2 then shares
    const int per = (g.tiles + 7) / 8, t = (int)(blockIdx.x & 7) * per + (int)(blockIdx.x >> 3);
    if ((int)(blockIdx.x >> 3) >= per || t >= g.tiles) return;
    int which = 0;
    while (which + 1 < g.n && t >= g.first_tile[which + 1]) ++which;
    const sba_model::WeightGrad& pr = g.one[which];
    const int tiles_m = (pr.m + kTileM - 1) / kTileM, tiles_n = (pr.n + kTileN - 1) / kTileN, local = t - g.first_tile[which];
    // bands of four tile rows, walked column by column
    const int band = local / (4 * tiles_n), rows = min(4, tiles_m - 4 * band), in = local - band * 4 * tiles_n;
    const int m0 = (4 * band + in % rows) * kTileM, n0 = (in / rows) * kTileN;

    // this split's stages of the contraction
    const int all = (g.k + kStageRows - 1) / kStageRows, share = (all + (int)gridDim.y - 1) / (int)gridDim.y;
    const int first = min(all, (int)blockIdx.y * share), nk = min(all - first, share);
    const int ragged = g.k - (first + nk - 1) * kStageRows;          // rows of the last stage (32 unless it is the end)

    TileSource sa, sb;
    sa.init(pr.a, pr.lda, m0, pr.m, w, lane);
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

    // fetch addresses: [half of the eight rows][column block]; the wave's quarter of the tile is in the base
    uint32_t fa[2][4], fb[2][4];
    {
        const int h = lane >> 5, G1 = (lane >> 4) & 1, s = lane & 15;
#pragma unroll
        for (int a = 0; a < 2; ++a)
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                const uint32_t o = (uint32_t)tile_offset<256>(8 * h + 4 * a + (s >> 2), 4 * c + 2 * G1 + ((s & 3) >> 1)) + ((s & 1) << 3);
                fa[a][c] = lds0 + (w & 1) * 256 + o;
                fb[a][c] = lds0 + kBBase + (w >> 1) * 256 + o;
                asm("" : "+v"(fa[a][c]), "+v"(fb[a][c]));
            }
    }

    f32x16 acc[4][4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;

    h16x8 va[2][4], vb[2][4];
    if (nk > 0) {
#pragma unroll
        for (int s = 0; s < kBuffers; ++s)
            if (s < nk) request(s, s);
        if (nk >= 4) asm volatile("s_waitcnt vmcnt(24)\n\ts_barrier" ::: "memory");
        else asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
        if (rows_of(0) < kStageRows) clear_from(rows_of(0), 0);
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            va[0][c] = fragment(fa[0][c], fa[1][c], 0);
            vb[0][c] = fragment(fb[0][c], fb[1][c], 0);
        }
    }
    // sixteen MFMAs of one half stage, one fetch of the next half's operands under every second one
    auto half = [&](int cur, int buf, int row0) {
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                acc[i][j] = mfma(va[cur][i], vb[cur][j], acc[i][j]);
                const int n = i * 4 + j, imm = buf * kTileBytes + row0 * 512;
                if (n < 4) va[cur ^ 1][n] = fragment(fa[0][n], fa[1][n], imm);
                else if (n < 8) vb[cur ^ 1][n - 4] = fragment(fb[0][n - 4], fb[1][n - 4], imm);
                __builtin_amdgcn_sched_barrier(0);
            }
    };
    // whole groups of four stages, so that the loop has one exit (several cost the compiler copies of the accumulators, 128
    // spilled registers); a last group is filled up with stages of zeros
    for (int s0 = 0; s0 < nk; s0 += kBuffers) {
#pragma unroll
        for (int b = 0; b < kBuffers; ++b) {
            const int s = s0 + b;
            half(0, b, 16);
            if (s + 3 < nk) asm volatile("s_waitcnt vmcnt(16) lgkmcnt(0)\n\ts_barrier" ::: "memory");
            else asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
            if (rows_of(s + 1) < kStageRows) clear_from(rows_of(s + 1), (b + 1) & 3);
            if (s + kBuffers < nk) request(s + kBuffers, b);
            half(1, (b + 1) & 3, 0);
        }
    }

    // lane (column lane % 32, h), register r: row 8 * (r / 4) + 4 * h + r % 4
    float* out = (gridDim.y == 1 ? g.out : g.partial + (int64_t)blockIdx.y * g.total) + pr.at;
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int col = n0 + (w >> 1) * 128 + j * 32 + (lane & 31);
            const int row0 = m0 + (w & 1) * 128 + i * 32 + 4 * (lane >> 5);
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int row = row0 + 8 * (r >> 2) + (r & 3);
                if (row < pr.m && col < pr.n) out[(int64_t)row * pr.n + col] = acc[i][j][r];
            }
        }
}

// ---------------------------------------------------------------------------------------------------- projections
// Y[t][n] = sum over k of X[t][k] * W[n][k] for token rows t, or W[k][n] (kRowsW: the product of a backward), 16-bit operands,
// fp32 sums, and what the model does with Y in the same pass (Epilogue).
//
// Small products: 128 x 128 tiles, two workgroups a CU, k a multiple of 32.  Such launches are short of workgroups and of time to
// fill a pipeline; two resident ones hide each other's start and stores.  Four waves, two by two, each 64 tokens x 64 features.
// Stages of 32 k and four tile buffers, requested, awaited and walked as in the weight-gradient kernel.  A tile row of 32 k is 64
// bytes, four 16-byte chunks; chunk c of row r lies at c ^ (r / 4 % 4), so that sixteen consecutive rows' chunks of one index fall on
// sixteen different bank groups.  The products are formed transposed (rows: features, columns: tokens): a lane then holds runs of
// four features of one token, which leave through LDS as whole rows.  4096 x 1024, k = 1024: 13 us.
using sba_model::Projection;

template <bool kRowsW, int kEpi>
__global__ __launch_bounds__(256, 2) void projection_kernel(Projection p) {
    constexpr int TM = 128, TN = 128, NB = 4;
    constexpr int kX = TM * 64, kW = TN * 64, kStage = kX + kW;        // bytes
    constexpr int PX = TM / 64, PW = TN / 64, P = PX + PW;             // copies per wave and stage
    constexpr int TI = TN / 64, TJ = TM / 64;                          // 32-wide blocks of a wave: features, tokens
    __shared__ __attribute__((aligned(1024))) char lds[NB * kStage];
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int m = lane & 31, h = lane >> 5;

    // a swiglu tile's features are TN/2 gates and the TN/2 ups that go with them
    constexpr bool kGlu = kEpi == sba_model::kSwigluFwd;
    const int features = kGlu ? p.n / 2 : p.n;
    constexpr int kOwn = kGlu ? TN / 2 : TN;
    const int tiles_m = (p.m + TM - 1) / TM, tiles_n = (features + kOwn - 1) / kOwn, tiles = tiles_m * tiles_n;
    const int per = (tiles + 7) / 8, t = (int)(blockIdx.x & 7) * per + (int)(blockIdx.x >> 3);
    if ((int)(blockIdx.x >> 3) >= per || t >= tiles) return;
    constexpr int kBand = 1024 / TM;
    const int band = t / (kBand * tiles_n), rows = min(kBand, tiles_m - kBand * band), in = t - band * kBand * tiles_n;
    const int t0 = (kBand * band + in % rows) * TM, n0 = (in / rows) * kOwn;
    const int nk = p.k / 32;

    const char* xat = (const char*)p.x + 2 * (int64_t)t0 * p.ldx;
    const char* wat = (const char*)p.w + (kRowsW ? 2 * (int64_t)n0 : (int64_t)0);
    uint32_t xoff[PX], woff[PW];
#pragma unroll
    for (int i = 0; i < PX; ++i) {
        const int row = 16 * (w + 4 * i) + (lane >> 2), c = (lane & 3) ^ ((row >> 2) & 3);
        xoff[i] = (uint32_t)min(row, p.m - 1 - t0) * (uint32_t)(2 * p.ldx) + 16u * c;
    }
#pragma unroll
    for (int i = 0; i < PW; ++i) {
        if (kRowsW) {
            constexpr int kPer = 512 / TN;                     // rows of TN columns per copy
            const int row = kPer * (w + 4 * i) + lane / (TN / 8), c = (lane & (TN / 8 - 1)) ^ swz<TN>(row);
            woff[i] = (uint32_t)row * (uint32_t)(2 * p.ldw) + 16u * (uint32_t)min(c, (features - n0) / 8 - 1);
        } else {
            const int row = 16 * (w + 4 * i) + (lane >> 2), c = (lane & 3) ^ ((row >> 2) & 3);
            int feature = n0 + row, up = 0;
            if (kGlu) {                                        // a wave's half of the tile: TN/4 gates, then their ups
                feature = n0 + (row / (TN / 2)) * (TN / 4) + row % (TN / 4);
                up = (row % (TN / 2)) / (TN / 4) * features;
            }
            woff[i] = (uint32_t)(min(feature, features - 1) + up) * (uint32_t)(2 * p.ldw) + 16u * c;
        }
    }
    const uint32_t lds0 = lds_address(lds);
    auto request = [&](int buf) {
#pragma unroll
        for (int i = 0; i < PX; ++i) dma16(xat, xoff[i], lds0 + buf * kStage + (w + 4 * i) * 1024);
#pragma unroll
        for (int i = 0; i < PW; ++i) dma16(wat, woff[i], lds0 + buf * kStage + kX + (w + 4 * i) * 1024);
        xat += 64;
        wat += kRowsW ? 64 * p.ldw : (int64_t)64;
    };

    // fetch addresses: X rows and, k contiguous, W rows [k slice]; W columns [half of the eight rows][column block]
    uint32_t fx[2], fw[2], fc[2][TI];
#pragma unroll
    for (int s = 0; s < 2; ++s) {
        const int c = (2 * s + h) ^ ((m >> 2) & 3);
        fx[s] = lds0 + (w & 1) * (TM / 2) * 64 + m * 64 + c * 16;
        fw[s] = lds0 + kX + (w >> 1) * (TN / 2) * 64 + m * 64 + c * 16;
        asm("" : "+v"(fx[s]), "+v"(fw[s]));
    }
    if (kRowsW) {
        const int G1 = (lane >> 4) & 1, s = lane & 15;
#pragma unroll
        for (int a = 0; a < 2; ++a)
#pragma unroll
            for (int c = 0; c < TI; ++c) {
                fc[a][c] = lds0 + kX + (uint32_t)tile_offset<TN>(8 * h + 4 * a + (s >> 2), (w >> 1) * (TN / 16) + 4 * c + 2 * G1 + ((s & 3) >> 1)) + ((s & 1) << 3);
                asm("" : "+v"(fc[a][c]));
            }
    }
    auto at = [](uint32_t base, int imm) {
        return *(const __attribute__((address_space(3))) h16x8*)((__attribute__((address_space(3))) char*)(uintptr_t)base + imm);
    };

    f32x16 acc[TI][TJ];
#pragma unroll
    for (int i = 0; i < TI; ++i)
#pragma unroll
        for (int j = 0; j < TJ; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;
    h16x8 vx[2][TJ], vw[2][TI];
    // the n-th of the operands of k slice s of buffer `buf`
    auto fetch = [&](int set, int n, int buf, int s) {
        if (n < TJ) vx[set][n] = at(fx[s], buf * kStage + n * 2048);
        else if (n < TJ + TI) {
            if (kRowsW) vw[set][n - TJ] = fragment(fc[0][n - TJ], fc[1][n - TJ], buf * kStage + s * 16 * TN * 2);
            else vw[set][n - TJ] = at(fw[s], buf * kStage + (n - TJ) * 2048);
        }
    };
    auto half = [&](int cur, int buf, int s) {
#pragma unroll
        for (int n = 0; n < TI * TJ; ++n) {
            const int i = n / TJ, j = n % TJ;
            acc[i][j] = mfma(vw[cur][i], vx[cur][j], acc[i][j]);
            fetch(cur ^ 1, n, buf, s);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    static_assert(TI + TJ <= TI * TJ, "one fetch per MFMA");
    auto clear = [&](int buf) {
        for (int c = threadIdx.x; c < kStage / 16; c += 256) *(u32x4*)(lds + buf * kStage + c * 16) = u32x4{0u, 0u, 0u, 0u};
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    };

#pragma unroll
    for (int s = 0; s < NB; ++s)
        if (s < nk) request(s);
    if (nk >= NB) asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" : : "n"((NB - 1) * P) : "memory");
    else asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
#pragma unroll
    for (int n = 0; n < TI + TJ; ++n) fetch(0, n, 0, 0);
    for (int s0 = 0; s0 < nk; s0 += NB) {      // whole groups, filled up with stages of zeros (see the weight-gradient kernel)
#pragma unroll
        for (int b = 0; b < NB; ++b) {
            const int s = s0 + b;
            half(0, b, 1);
            if (s + NB - 1 < nk) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" : : "n"((NB - 2) * P) : "memory");
            else asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
            if (s + 1 >= nk) clear((b + 1) % NB);
            if (s + NB < nk) request(b);
            half(1, (b + 1) % NB, 0);
        }
    }
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");      // the tiles become the waves' staging

    // 32 tokens at a time: through the wave's own part of LDS into rows
    char* const stage = lds + w * (NB * kStage / 4);
    static_assert(NB * kStage / 4 >= 32 * (TN / 2) * 4, "a wave stages 32 tokens' features in fp32");
    constexpr int F = TN / 2;                                          // features of a wave
    const int tw = t0 + (w & 1) * (TM / 2), nw = n0 + (w >> 1) * (kOwn / 2);
#pragma unroll
    for (int j = 0; j < TJ; ++j) {
        const int tok0 = tw + 32 * j;
        if (tok0 >= p.m) break;
        if (kEpi == sba_model::kAddResidual) {
            // out = residual + y (rounded to 16 bits, as a tensor of its own would be): 16-byte chunks of four features
#pragma unroll
            for (int i = 0; i < TI; ++i)
#pragma unroll
                for (int g = 0; g < 4; ++g) {
                    typedef float f32x4 __attribute__((ext_vector_type(4)));
                    f32x4 v;
#pragma unroll
                    for (int e = 0; e < 4; ++e) v[e] = (float)(elem16)acc[i][j][4 * g + e];
                    *(f32x4*)(stage + m * (F * 4) + (((i * 8 + 2 * g + h) ^ m) & (F / 4 - 1)) * 16) = v;
                }
            for (int c = lane; c < 32 * F / 4; c += 64) {
                typedef float f32x4 __attribute__((ext_vector_type(4)));
                const int row = c / (F / 4), cc = c % (F / 4), tok = tok0 + row, n = nw + 4 * cc;
                if (tok < p.m && n < p.n) {
                    const f32x4 v = *(const f32x4*)(stage + row * (F * 4) + ((cc ^ row) & (F / 4 - 1)) * 16);
                    const f32x4 r = *(const f32x4*)(p.residual + (int64_t)tok * p.n + n);
                    *(f32x4*)((float*)p.out + (int64_t)tok * p.n + n) = v + r;
                }
            }
        } else {
            // 16-bit rows of F features, chunks of eight: chunk c of token r at c ^ r
            constexpr int kChunks = F / 8;
            auto put = [&](int chunk, const float* v) {
                const f32x2 a = {v[0], v[1]}, b = {v[2], v[3]};
                uint2 u;
                u.x = __builtin_bit_cast(uint32_t, __builtin_convertvector(a, h16x2));
                u.y = __builtin_bit_cast(uint32_t, __builtin_convertvector(b, h16x2));
                *(uint2*)(stage + m * (F * 2) + ((chunk ^ m) & (kChunks - 1)) * 16 + h * 8) = u;
            };
#pragma unroll
            for (int i = 0; i < TI; ++i)
#pragma unroll
                for (int g = 0; g < 4; ++g) {
                    const float v[4] = {acc[i][j][4 * g], acc[i][j][4 * g + 1], acc[i][j][4 * g + 2], acc[i][j][4 * g + 3]};
                    put(i * 4 + g, v);
                }
            auto chunk_of = [&](int row, int cc) { return *(const h16x8*)(stage + row * (F * 2) + ((cc ^ row) & (kChunks - 1)) * 16); };
            if (kGlu) {
                // gates are chunks 0 .. kChunks/2 - 1 of a row, their ups the rest
                for (int c = lane; c < 32 * kChunks / 2; c += 64) {
                    const int row = c / (kChunks / 2), cc = c % (kChunks / 2), tok = tok0 + row, n = nw + 8 * cc;
                    if (tok < p.m && n < features) {
                        const h16x8 g = chunk_of(row, cc), u = chunk_of(row, cc + kChunks / 2);
                        h16x8 a;
#pragma unroll
                        for (int e = 0; e < 8; ++e) {
                            const float gf = (float)g[e];
                            a[e] = (elem16)((float)(elem16)(gf / (1.f + __expf(-gf))) * (float)u[e]);
                        }
                        *(h16x8*)((elem16*)p.out + (int64_t)tok * features + n) = a;
                        if (p.pre) {
                            *(h16x8*)((elem16*)p.pre + (int64_t)tok * p.n + n) = g;
                            *(h16x8*)((elem16*)p.pre + (int64_t)tok * p.n + features + n) = u;
                        }
                    }
                }
            } else {
                for (int c = lane; c < 32 * kChunks; c += 64) {
                    const int row = c / kChunks, cc = c % kChunks, tok = tok0 + row, n = nw + 8 * cc;
                    if (tok >= p.m || n >= p.n) continue;
                    const h16x8 v = chunk_of(row, cc);
                    if (kEpi == sba_model::kSwigluBwd) {
                        // y is the gradient of silu(gate) * up: gate and up from `pre`, their gradients to `out`
                        const elem16* gu = (const elem16*)p.pre + (int64_t)tok * 2 * p.n + n;
                        elem16* o = (elem16*)p.out + (int64_t)tok * 2 * p.n + n;
                        const h16x8 g = *(const h16x8*)gu, u = *(const h16x8*)(gu + p.n);
                        h16x8 dg, du;
#pragma unroll
                        for (int e = 0; e < 8; ++e) {
                            const float gf = (float)g[e], df = (float)v[e], sg = 1.f / (1.f + __expf(-gf));
                            du[e] = (elem16)(df * (float)(elem16)(gf * sg));
                            dg[e] = (elem16)((float)(elem16)(df * (float)u[e]) * sg * (1.f + gf * (1.f - sg)));
                        }
                        *(h16x8*)o = dg;
                        *(h16x8*)(o + p.n) = du;
                    } else {
                        *(h16x8*)((elem16*)p.out + (int64_t)tok * p.n + n) = v;
                    }
                }
            }
        }
    }
}

// Large products: TM x 256 tiles, one resident workgroup a CU that walks tiles, one wave per SIMD with TM/2 x 128 of a tile.
// Stages of 64 k: rows of 64 k are whole 128-byte lines (with 32 k every line is fetched twice: -12 %).  A stage is four slices of
// TM/16 MFMAs a wave; the operands of a slice are fetched under the MFMAs of the one before.  After the third slice the waves meet:
// the stage's buffer has been read, the next stage has landed, and the copies of the stage NB ahead start into it, spread over the
// slices that follow (all under one they ask for 1024 cycles of the CU's memory pipe in 544 of MFMAs: 1.55 us per stage against
// 1.42 with 256 rows, every CU busy).  The copies run through the list of (tile, stage) pairs without a break, so a tile's results
// are stored while the next tile's first stages arrive.  TM = 256 has two buffers of 64 KB, TM = 128, whose stages pass in half the
// time, three of 48 KB; the fetch addresses move from buffer to buffer, one add per address and stage.
// 8192 tokens, k = 1024, TM = 256: 5632 features in 79 us (1.2 PFLOP/s; the library's kernel 96), with swiglu in 108 (its pass of its
// own would read and write 230 MB more); TM = 128: 1024 features in 18 us (library: 21), with the residual for k = 2816 46 us (40 + 15).
template <int TM, bool kRowsW, int kEpi>
__global__ __launch_bounds__(256, 1) void large_projection_kernel(Projection p) {
    constexpr int NB = TM == 256 ? 2 : 3;
    constexpr int kX = TM * 128, kStage = kX + 256 * 128;
    constexpr int PX = TM / 32, P = PX + 8;                    // copies per wave and stage
    constexpr int TJ = TM / 64, kSlots = 4 * TJ;               // blocks of 32 tokens of a wave; MFMAs of a slice
    __shared__ __attribute__((aligned(1024))) char lds[NB * kStage + 4 * 4096];
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int m = lane & 31, h = lane >> 5;
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
    const int nk = p.k / 64;

    // ---- the stream of copies
    const char *xat, *wat;
    uint32_t xoff[PX], woff[8];
    int d_local = local, d_stage = 0;
    uint32_t d_lds = lds_address(lds) + w * 1024;
    auto aim = [&](int l) {
        int t0, n0;
        tile_at(l, t0, n0);
        xat = (const char*)p.x + 2 * (int64_t)t0 * p.ldx;
        wat = (const char*)p.w + (kRowsW ? 2 * (int64_t)n0 : (int64_t)0);
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
    const int64_t wstep = kRowsW ? 128 * p.ldw : (int64_t)128;
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
    uint32_t fx[4], fw[4], fc[2][4];
    const uint32_t lds0 = lds_address(lds);
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const int c = (2 * q + h) ^ ((m >> 1) & 7);
        fx[q] = lds0 + (w & 1) * (TM / 2) * 128 + m * 128 + c * 16;
        fw[q] = lds0 + kX + (w >> 1) * 128 * 128 + m * 128 + c * 16;
        asm("" : "+v"(fx[q]), "+v"(fw[q]));
    }
    if (kRowsW) {
        const int G1 = (lane >> 4) & 1, s = lane & 15;
#pragma unroll
        for (int a = 0; a < 2; ++a)
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                fc[a][c] = lds0 + kX + (uint32_t)tile_offset<256>(8 * h + 4 * a + (s >> 2), (w >> 1) * 16 + 4 * c + 2 * G1 + ((s & 3) >> 1)) + ((s & 1) << 3);
                asm("" : "+v"(fc[a][c]));
            }
    }
    int f_buf = 0;
    auto next_buffer = [&]() {
        f_buf = f_buf + 1 == NB ? 0 : f_buf + 1;
        uint32_t by = f_buf == 0 ? (uint32_t)-((NB - 1) * kStage) : (uint32_t)kStage;
        asm("" : "+s"(by));
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            fx[q] += by;
            if (!kRowsW) fw[q] += by;
        }
        if (kRowsW) {
#pragma unroll
            for (int a = 0; a < 2; ++a)
#pragma unroll
                for (int c = 0; c < 4; ++c) fc[a][c] += by;
        }
    };
    auto at = [](uint32_t base, int imm) {
        return *(const __attribute__((address_space(3))) h16x8*)((__attribute__((address_space(3))) char*)(uintptr_t)base + imm);
    };
    h16x8 vx[2][TJ], vw[2][4];
    auto fetch = [&](int set, int n, int q) {
        if (n < TJ) vx[set][n] = at(fx[q], n * 4096);
        else if (n < TJ + 4) {
            const int i = n - TJ;
            if (kRowsW) vw[set][i] = fragment(fc[0][i], fc[1][i], q * 16 * 512);
            else vw[set][i] = at(fw[q], i * 4096);
        }
    };
    f32x16 acc[4][TJ];
    // MFMAs of one slice; under them the fetches of slice q and copies first .. first + count - 1
    auto slice = [&](int cur, int q, int first, int count, bool fresh = false) __attribute__((always_inline)) {
#pragma unroll
        for (int n = 0; n < kSlots; ++n) {
            acc[n / TJ][n % TJ] = mfma(vw[cur][n / TJ], vx[cur][n % TJ], fresh ? f32x16{0} : acc[n / TJ][n % TJ]);
            fetch(cur ^ 1, n, q);
            if ((n & 1) && n / 2 < count) copy(first + n / 2);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    // which slices the copies of a stage go under: TM = 256 the fourth and the first, 128 all of them
    constexpr int C3 = TM == 256 ? 8 : 3, C0 = TM == 256 ? 8 : 3, C1 = TM == 256 ? 0 : 3, C2 = P - C3 - C0 - C1;
    static_assert(C2 >= 0 && C3 <= kSlots / 2 && C2 <= kSlots / 2, "a copy under every second MFMA");

    // ---- results: 32 tokens at a time through the wave's 4 KB of staging, 128 bytes of a row: chunk c of token r at c ^ r / 2
    char* const stage = lds + NB * kStage + w * 4096;
    auto spot = [&](int row, int c) { return stage + row * 128 + ((c ^ (row >> 1)) & 7) * 16; };
    // The residual is requested a block of 32 features ahead (block 0 before the tile's last copies): with one wave per SIMD nobody
    // else has work meanwhile.
    typedef float f32x4 __attribute__((ext_vector_type(4)));
    constexpr bool kAdd = kEpi == sba_model::kAddResidual;
    constexpr int kChunkBlocks = kAdd ? 1 : 2;                 // blocks of 32 features that are stored together
    constexpr int kChunks = TJ * 4 / kChunkBlocks;
    f32x4 ahead[kAdd ? 2 : 1][4];
    auto read_ahead = [&](int chunk, int t0, int n0) __attribute__((always_inline)) {
        if (!kAdd || chunk >= kChunks) return;
        int lane_here = lane;
        asm volatile("" : "+v"(lane_here));
        const int tok0 = t0 + (w & 1) * (TM / 2) + 32 * (chunk / 4) + (lane_here >> 3);
        const int col = n0 + (w >> 1) * 128 + 32 * (chunk % 4) + 4 * (lane_here & 7);
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const int tok = tok0 + 8 * c;
            ahead[chunk & 1][c] = f32x4{0.f, 0.f, 0.f, 0.f};
            if (tok < p.m && col < p.n) ahead[chunk & 1][c] = *(const f32x4*)(p.residual + (int64_t)tok * p.n + col);
        }
    };
    auto store_tile = [&](int t0, int n0) {
        const int tw = t0 + (w & 1) * (TM / 2), nw = n0 + (w >> 1) * (kOwn / 2);
#pragma unroll
        for (int chunk = 0; chunk < kChunks; ++chunk) {
            // (this lane's indices from a copy that the compiler cannot see through: the addresses made from them would otherwise be
            // worked out ahead of the tile loop and kept, 70 spilled registers)
            int lane_here = lane;
            asm volatile("" : "+v"(lane_here));
            const int m = lane_here & 31, h = lane_here >> 5, row8 = lane_here >> 3, cc = lane_here & 7;
            const int j = chunk * kChunkBlocks / 4, i = chunk * kChunkBlocks % 4, tok0 = tw + 32 * j;
            read_ahead(chunk + 1, t0, n0);
            if (kAdd) {                                        // fp32; y rounded to 16 bits as a tensor of its own would be
#pragma unroll
                for (int g = 0; g < 4; ++g) {
                    f32x4 v;
#pragma unroll
                    for (int e = 0; e < 4; ++e) v[e] = (float)(elem16)acc[i][j][4 * g + e];
                    *(f32x4*)spot(m, 2 * g + h) = v;
                }
                const int n = nw + 32 * i + 4 * cc;
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    const int tok = tok0 + c * 8 + row8;
                    const f32x4 v = *(const f32x4*)spot(c * 8 + row8, cc);
                    if (tok < p.m && n < p.n) *(f32x4*)((float*)p.out + (int64_t)tok * p.n + n) = v + ahead[chunk & 1][c];
                }
            } else {                                           // 64 features: two blocks, with swiglu the gates and their ups
#pragma unroll
                for (int b = 0; b < 2; ++b)
#pragma unroll
                    for (int g = 0; g < 4; ++g) {
                        const f32x16& v = acc[kGlu ? i / 2 + 2 * b : i + b][j];
                        const f32x2 lo = {v[4 * g], v[4 * g + 1]}, hi = {v[4 * g + 2], v[4 * g + 3]};
                        uint2 u;
                        u.x = __builtin_bit_cast(uint32_t, __builtin_convertvector(lo, h16x2));
                        u.y = __builtin_bit_cast(uint32_t, __builtin_convertvector(hi, h16x2));
                        *(uint2*)(spot(m, 4 * b + g) + h * 8) = u;
                    }
                if (kGlu) {
#pragma unroll
                    for (int c = 0; c < 2; ++c) {
                        const int row = c * 16 + (lane_here >> 2), tok = tok0 + row, n = nw + 16 * i + 8 * (lane_here & 3);
                        const h16x8 g = *(const h16x8*)spot(row, lane_here & 3), u = *(const h16x8*)spot(row, 4 + (lane_here & 3));
                        if (tok < p.m && n < features) {
                            h16x8 a;
#pragma unroll
                            for (int e = 0; e < 8; ++e) {
                                const float gf = (float)g[e];
                                a[e] = (elem16)((float)(elem16)(gf / (1.f + __expf(-gf))) * (float)u[e]);
                            }
                            *(h16x8*)((elem16*)p.out + (int64_t)tok * features + n) = a;
                            if (p.pre) {
                                *(h16x8*)((elem16*)p.pre + (int64_t)tok * p.n + n) = g;
                                *(h16x8*)((elem16*)p.pre + (int64_t)tok * p.n + features + n) = u;
                            }
                        }
                    }
                    continue;
                }
                const int n = nw + 32 * i + 8 * cc;
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    const int tok = tok0 + c * 8 + row8;
                    const h16x8 v = *(const h16x8*)spot(c * 8 + row8, cc);
                    if (tok < p.m && n < p.n) *(h16x8*)((elem16*)p.out + (int64_t)tok * p.n + n) = v;
                }
            }
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
    for (int n = 0; n < TJ + 4; ++n) fetch(0, n, 0);
    // The stores of a tile lie in the queue behind the copies of the next tile's first NB stages, so its first wait can leave them
    // there - if the tile was a whole one, which is sure to have issued all of them.
    constexpr int kStores = kAdd ? 16 * TJ : kGlu ? 4 * TJ : 8 * TJ;     // (swiglu: 8 * TJ more where `pre` is kept)
    constexpr int kLeave = (NB - 2) * P + kStores < 63 ? (NB - 2) * P + kStores : 63;           // (63: the most a wait can leave)
    bool stores_behind = false;
    for (; local < run; local += stride) {
        int t0, n0;
        tile_at(local, t0, n0);
        slice(0, 1, 0, 0, true);
        slice(1, 2, 0, 0);
        slice(0, 3, 0, 0);
        if (stores_behind) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" : : "n"(kLeave) : "memory");
        else asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" : : "n"((NB - 2) * P) : "memory");
        next_buffer();
        slice(1, 0, 0, C3);
        for (int s = 1; s < nk; ++s) {
            slice(0, 1, C3, C0);
            slice(1, 2, C3 + C0, C1);
            slice(0, 3, C3 + C0 + C1, C2);
            next_stage();
            asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" : : "n"((NB - 2) * P) : "memory");
            next_buffer();
            slice(1, 0, 0, C3);
        }
        read_ahead(0, t0, n0);
#pragma unroll
        for (int i = C3; i < P; ++i) copy(i);
        next_stage();
        store_tile(t0, n0);
        stores_behind = t0 + TM <= p.m && n0 + kOwn <= features;
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");           // the last copies, unread, have landed before the LDS is given back
}

int launch_projection(const Projection& p, hipStream_t s) {
    const int own = p.epilogue == sba_model::kSwigluFwd ? 64 : 128, features = p.epilogue == sba_model::kSwigluFwd ? p.n / 2 : p.n;
    const int tiles = ((p.m + 127) / 128) * ((features + own - 1) / own);
    const dim3 grid((unsigned)((tiles + 7) / 8 * 8)), block(256);
    if (p.rows_w) {
        if (p.epilogue == sba_model::kSwigluBwd) hipLaunchKernelGGL((projection_kernel<true, sba_model::kSwigluBwd>), grid, block, 0, s, p);
        else if (p.epilogue == sba_model::kStore) hipLaunchKernelGGL((projection_kernel<true, sba_model::kStore>), grid, block, 0, s, p);
        else return -2;
    } else {
        if (p.epilogue == sba_model::kSwigluFwd) hipLaunchKernelGGL((projection_kernel<false, sba_model::kSwigluFwd>), grid, block, 0, s, p);
        else if (p.epilogue == sba_model::kAddResidual) hipLaunchKernelGGL((projection_kernel<false, sba_model::kAddResidual>), grid, block, 0, s, p);
        else if (p.epilogue == sba_model::kStore) hipLaunchKernelGGL((projection_kernel<false, sba_model::kStore>), grid, block, 0, s, p);
        else return -2;
    }
    return hipGetLastError() == hipSuccess ? 0 : -6;
}

template <int TM>
int launch_large_projection(const Projection& p, hipStream_t s) {
    const int own = p.epilogue == sba_model::kSwigluFwd ? 128 : 256, features = p.epilogue == sba_model::kSwigluFwd ? p.n / 2 : p.n;
    const int tiles = ((p.m + TM - 1) / TM) * ((features + own - 1) / own), cus = sba_cu_count() & ~7;
    const dim3 grid((unsigned)(((tiles < cus ? tiles : cus) + 7) & ~7)), block(256);
    if (p.rows_w) {
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
    return launch_projection(p, s);
}
int SBA_WEIGHT_GRADS(const WeightGrads& g, int splits, hipStream_t stream) {
    hipLaunchKernelGGL(sba::SBA_ELEM_NS::weight_grad_kernel, dim3((unsigned)((g.tiles + 7) / 8 * 8), (unsigned)splits), dim3(256), 0, stream, g);
    return hipGetLastError() == hipSuccess ? 0 : -6;
}
}  // namespace sba_model
