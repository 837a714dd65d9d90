// Weight gradients: C[m][n] = sum over t of A[t][m] * B[t][n], A and B 16-bit with the contracted index outermost, C fp32.
// Several products that share the contraction length run in one launch.  Compiled once for bf16 and, with SBA_ELEM_F16, once
// for float16.
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

}  // namespace
}  // namespace sba

#ifdef SBA_ELEM_F16
#define SBA_WEIGHT_GRADS weight_grads_f16
#else
#define SBA_WEIGHT_GRADS weight_grads_bf16
#endif
namespace sba_model {
int SBA_WEIGHT_GRADS(const WeightGrads& g, int splits, hipStream_t stream) {
    hipLaunchKernelGGL(sba::SBA_ELEM_NS::weight_grad_kernel, dim3((unsigned)((g.tiles + 7) / 8 * 8), (unsigned)splits), dim3(256), 0, stream, g);
    return hipGetLastError() == hipSuccess ? 0 : -6;
}
}  // namespace sba_model
