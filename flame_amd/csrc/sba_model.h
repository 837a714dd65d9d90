// Kernels around the attention operator in the language model (sba_model.hip): normalisation with the residual, SwiGLU, the
// weights' casts, cross-entropy, clipping with AdamW.  Rows are dense; `f16` selects float16 instead of bf16 for the 16-bit
// tensors; everything else is fp32.  Launches are asynchronous on `stream`.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace sba_model {

constexpr int kMaxNormWidth = 2048;      // columns of a row that a wave keeps in registers
constexpr int kCastTensors = 8;
constexpr int kOptChunk = 16384;         // weights to a partial sum of squares

// y = rms_norm(x) * w as 16-bit
struct NormFwd {
    const float* x; const float* w;
    void* y; float* rstd;
    int rows, cols; float eps;
};
int norm_fwd(const NormFwd& a, bool f16, hipStream_t stream);

// dx = dres + the gradient through the norm; dx16 its 16-bit copy (may be null), dw_part [norm_bwd_parts(rows)][cols].
struct NormBwd {
    const void* dy; const float* x; const float* w; const float* rstd; const float* dres;
    float* dx; void* dx16; float* dw_part;
    int rows, cols;
};
int norm_bwd_parts(int rows);
int norm_bwd(const NormBwd& a, bool f16, hipStream_t stream);
// out[i][c] = sum over the parts of part[i], for one or two of them in a launch
int sum_parts(const float* const (&part)[2], float* const (&out)[2], int n, int parts, int cols, hipStream_t stream);

// y = [rows][2 * width] = gate | up;  out = silu(gate) * up
int swiglu_fwd(const void* y, void* out, int64_t rows, int width, bool f16, hipStream_t stream);
int swiglu_bwd(const void* y, const void* d_out, void* dy, int64_t rows, int width, bool f16, hipStream_t stream);

// up to kCastTensors fp32 tensors, one after the other, as 16-bit
struct CastList {
    const float* src[kCastTensors];
    int64_t end[kCastTensors];           // running total of elements; every length is a multiple of 8
    int n;
};
int cast_list(const CastList& a, void* out, bool f16, hipStream_t stream);
int cast_one(const float* src, void* out, int64_t n, bool f16, hipStream_t stream);

// Next-token cross-entropy over rows of `classes` 16-bit logits: row r of a sequence of `len` is scored against
// labels[r + 1], the last row of a sequence and rows whose label is `ignore` are not.  lse, row_loss [rows]; mean, count [1].
int loss_fwd(const void* logits, const int64_t* labels, float* lse, float* row_loss, float* mean, float* count, int rows, int len,
             int classes, int64_t ignore, bool f16, hipStream_t stream);
int loss_bwd(const void* logits, const int64_t* labels, const float* lse, const float* count, const float* d_loss,
             void* d_logits, int rows, int len, int classes, int64_t ignore, bool f16, hipStream_t stream);

// Weight gradients c[m][n] = sum over k rows of a[.][m] * b[.][n] (16-bit operands, fp32 results) of up to four products with
// the same rows, in one launch (sba_gemm.hip).  m, n and the leading dimensions are multiples of 8 and the operands 16-byte aligned
// (the copies move whole 16-byte chunks of a row); others are refused with -2.  The results lie one after the other from `out` on.
struct WeightGrad {
    const void* a; const void* b; int64_t lda, ldb; int m, n;
    int64_t at;                          // first element of the result behind `out`
};
struct WeightGrads {
    WeightGrad one[4];
    int first_tile[4];
    int n, tiles, k;
    int tile_rows;                       // 256 or 224: rows of C in a workgroup's tile
    float* out; float* partial; int64_t total;
};
bool weight_grads_fit(const WeightGrads& g);             // whether the kernel takes it
int weight_grad_splits(WeightGrads& g, int cus);         // fills first_tile, tiles, tile_rows, at, total; partial sums of how many splits
int weight_grads(const WeightGrads& g, int splits, bool f16, hipStream_t stream);     // partial: [splits][total] if more than one
int weight_grads_bf16(const WeightGrads& g, int splits, hipStream_t stream);
int weight_grads_f16(const WeightGrads& g, int splits, hipStream_t stream);

// y[t][n] = sum over k of x[t][k] w[n][k] (rows_w: w[k][n]) for m token rows, k a multiple of 32, n of 8, and what follows:
//   kStore        out = y                                    16-bit [m][n]
//   kAddResidual  out = residual + y                         fp32   [m][n]; y is the fp32 sum, not rounded to 16 bits first
//   kSwigluFwd    w = gate rows | up rows: out = silu(gate) * up, 16-bit [m][n/2]; pre = y if given
//   kSwigluBwd    y = gradient of silu(gate) * up, pre = gate | up [m][2n]: out = their gradients, 16-bit [m][2n]
// x and w are 16-byte aligned with leading dimensions that are multiples of 8; outputs are dense.
enum { kStore, kAddResidual, kSwigluFwd, kSwigluBwd, kPartialSums };      // (kPartialSums: within the kernels, fp32 [splits][m][n])
struct Projection {
    const void* x; const void* w; int64_t ldx, ldw; int m, n, k;
    bool rows_w; int epilogue;
    const float* residual; void* pre; void* out;
    int splits; float* partial;          // kStore, rows_w: so many workgroups share a tile's contraction (0, 1: none); [splits][m][n]
};
bool addresses(const Projection& p);                     // whether the kernels can take it
bool projects(const Projection& p, int cus);             // whether they do
enum ProjectionTile { kTile256, kTile128x256, kTile128, kTile128Halves, kTile64, kTile64Halves };
ProjectionTile projection_tile(const Projection& p, int cus);
double tile_time(const Projection& p, ProjectionTile tile, int cus);    // an estimate, us; 1e30 where its kernel does not take it
// how many workgroups had better share the contraction of a tile, and of which tile; 1: as projection_tile() says
int projection_splits(const Projection& p, int cus, ProjectionTile& tile);
int project_tile(const Projection& p, ProjectionTile tile, bool f16, hipStream_t stream);
int project_bf16(const Projection& p, ProjectionTile tile, hipStream_t stream);
int project_f16(const Projection& p, ProjectionTile tile, hipStream_t stream);

// One weight tensor of a clip + AdamW step.
struct OptTensor {
    float* p; float* g; float* m; float* v; float* step;
    int64_t n; int64_t first_chunk;      // chunks of the tensors before this one
    double lr, beta1, beta2;
    float decay, one_minus_beta1, beta2_f, one_minus_beta2, eps;         // rounded once from the caller's doubles
    float step_size, denom_scale;        // filled on the device: lr / (1 - beta1^step), 1 / sqrt(1 - beta2^step)
};
// norm [1], partial [chunks + 1] (the last one: the clip coefficient).  Three launches: partial sums, norms and step counts, update.
int clip_and_adamw(OptTensor* tensors, int n_tensors, int64_t chunks, float max_norm, float* partial, float* norm,
                   hipStream_t stream);

}  // namespace sba_model
