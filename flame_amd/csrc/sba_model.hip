// Kernels around the attention operator in the language model.  All of them are bound by memory: what pays is that a tensor
// is read and written once where a chain of framework kernels passes over it several times, and that the fp32 residual stream
// and its 16-bit copies leave in the same pass.
#include "sba_model.h"

namespace sba_model {
namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));
template <typename E> struct Vec;
template <> struct Vec<__bf16> {
    typedef __bf16 x8 __attribute__((ext_vector_type(8)));
    typedef __bf16 x4 __attribute__((ext_vector_type(4)));
};
template <> struct Vec<_Float16> {
    typedef _Float16 x8 __attribute__((ext_vector_type(8)));
    typedef _Float16 x4 __attribute__((ext_vector_type(4)));
};

constexpr int kThreads = 256;
constexpr int kWaves = kThreads / 64;

__device__ inline float wave_sum(float v) {
#pragma unroll
    for (int d = 32; d; d >>= 1) v += __shfl_xor(v, d, 64);
    return v;
}
__device__ inline float wave_max(float v) {
#pragma unroll
    for (int d = 32; d; d >>= 1) v = fmaxf(v, __shfl_xor(v, d, 64));
    return v;
}

int launched() { return hipGetLastError() == hipSuccess ? 0 : -6; }

// ------------------------------------------------------------------------------------------------- RMS norm
// One wave per row, the row in registers (K groups of 256 columns, four columns a lane and group: 16-byte accesses, 1 KB per
// wave and instruction).
template <typename E, int K>
__global__ __launch_bounds__(kThreads) void norm_fwd_kernel(NormFwd a) {
    const int lane = threadIdx.x & 63, row = blockIdx.x * kWaves + (threadIdx.x >> 6);
    if (row >= a.rows) return;
    typedef typename Vec<E>::x4 e4;
    const int64_t base = (int64_t)row * a.cols;
    f32x4 x[K];
    float ss = 0.f;
#pragma unroll
    for (int k = 0; k < K; ++k) {
        const int c = (k * 64 + lane) * 4;
        x[k] = f32x4{0.f, 0.f, 0.f, 0.f};
        if (c < a.cols) {
            x[k] = *(const f32x4*)(a.x + base + c);
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) ss += x[k][i] * x[k][i];
    }
    ss = wave_sum(ss);
    const float rstd = rsqrtf(ss / (float)a.cols + a.eps);
    if (lane == 0) a.rstd[row] = rstd;
#pragma unroll
    for (int k = 0; k < K; ++k) {
        const int c = (k * 64 + lane) * 4;
        if (c < a.cols) {
            const f32x4 w = *(const f32x4*)(a.w + c);
            e4 y;
#pragma unroll
            for (int i = 0; i < 4; ++i) y[i] = (E)(x[k][i] * rstd * w[i]);
            *(e4*)((E*)a.y + base + c) = y;
        }
    }
}

// dx_i = dres_i + rstd * (dy_i w_i - x_i rstd^2 mean_j(dy_j w_j x_j)).  A wave walks rows and keeps its share of
// dw = sum over rows of dy x rstd in registers; the four waves of a workgroup add theirs in LDS and write one partial row.
template <typename E, int K>
__global__ __launch_bounds__(kThreads) void norm_bwd_kernel(NormBwd a) {
    typedef typename Vec<E>::x4 e4;
    __shared__ float part[kWaves][K * 256];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    f32x4 dw[K];
#pragma unroll
    for (int k = 0; k < K; ++k) dw[k] = f32x4{0.f, 0.f, 0.f, 0.f};
    for (int row = blockIdx.x * kWaves + wave; row < a.rows; row += gridDim.x * kWaves) {
        const int64_t base = (int64_t)row * a.cols;
        const float rstd = a.rstd[row];
        f32x4 x[K], g[K], r[K];
        float dot = 0.f;
#pragma unroll
        for (int k = 0; k < K; ++k) {
            const int c = (k * 64 + lane) * 4;
            x[k] = g[k] = r[k] = f32x4{0.f, 0.f, 0.f, 0.f};
            if (c < a.cols) {
                x[k] = *(const f32x4*)(a.x + base + c);
                const e4 dy = *(const e4*)((const E*)a.dy + base + c);
                if (a.dres) r[k] = *(const f32x4*)(a.dres + base + c);
#pragma unroll
                for (int i = 0; i < 4; ++i) g[k][i] = (float)dy[i];
            }
        }
#pragma unroll
        for (int k = 0; k < K; ++k) {
            const int c = (k * 64 + lane) * 4;
            const f32x4 w = c < a.cols ? *(const f32x4*)(a.w + c) : f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                dw[k][i] += g[k][i] * x[k][i] * rstd;
                g[k][i] *= w[i];
                dot += g[k][i] * x[k][i];
            }
        }
        const float c1 = wave_sum(dot) / (float)a.cols * rstd * rstd;
#pragma unroll
        for (int k = 0; k < K; ++k) {
            const int c = (k * 64 + lane) * 4;
            if (c >= a.cols) continue;
            e4 d16;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                r[k][i] += rstd * (g[k][i] - x[k][i] * c1);
                d16[i] = (E)r[k][i];
            }
            *(f32x4*)(a.dx + base + c) = r[k];
            if (a.dx16) *(e4*)((E*)a.dx16 + base + c) = d16;
        }
    }
#pragma unroll
    for (int k = 0; k < K; ++k) *(f32x4*)&part[wave][(k * 64 + lane) * 4] = dw[k];
    __syncthreads();
    for (int c = threadIdx.x; c < a.cols; c += kThreads)
        a.dw_part[(int64_t)blockIdx.x * a.cols + c] = part[0][c] + part[1][c] + part[2][c] + part[3][c];
}

// out[c] = sum over the parts: a workgroup takes 16 columns, 64 threads share a column's parts, eight loads of each in flight
__global__ __launch_bounds__(1024) void sum_parts_kernel(const float* part0, const float* part1, float* out0, float* out1, int parts, int cols) {
    const float* const part = blockIdx.y ? part1 : part0;
    float* const out = blockIdx.y ? out1 : out0;
    __shared__ float acc[64][17];
    const int lc = threadIdx.x & 15, c = blockIdx.x * 16 + lc, g = threadIdx.x >> 4;
    float s = 0.f;
    if (c < cols)
#pragma unroll 8
        for (int i = g; i < parts; i += 64) s += part[(int64_t)i * cols + c];
    acc[g][lc] = s;
    __syncthreads();
    if (g == 0 && c < cols) {
#pragma unroll
        for (int i = 1; i < 64; ++i) s += acc[i][lc];
        out[c] = s;
    }
}

// ------------------------------------------------------------------------------------------------- SwiGLU
// silu(gate) and d_out * up are rounded to 16 bits where the module path holds them as tensors: both paths give the same bits.
template <typename E>
__global__ __launch_bounds__(kThreads) void swiglu_fwd_kernel(const E* y, E* out, int64_t n8, int w8) {
    typedef typename Vec<E>::x8 e8;
    for (int64_t i = (int64_t)blockIdx.x * kThreads + threadIdx.x; i < n8; i += (int64_t)gridDim.x * kThreads) {
        const int64_t row = i / w8;
        const int c = (int)(i - row * w8);
        const E* r = y + (row * 2 * w8 + c) * 8;
        const e8 g = *(const e8*)r, u = *(const e8*)(r + (int64_t)w8 * 8);
        e8 o;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const float gf = (float)g[j];
            o[j] = (E)((float)(E)(gf / (1.f + __expf(-gf))) * (float)u[j]);
        }
        *(e8*)(out + i * 8) = o;
    }
}

template <typename E>
__global__ __launch_bounds__(kThreads) void swiglu_bwd_kernel(const E* y, const E* d_out, E* dy, int64_t n8, int w8) {
    typedef typename Vec<E>::x8 e8;
    for (int64_t i = (int64_t)blockIdx.x * kThreads + threadIdx.x; i < n8; i += (int64_t)gridDim.x * kThreads) {
        const int64_t row = i / w8;
        const int c = (int)(i - row * w8);
        const int64_t at = (row * 2 * w8 + c) * 8, up = (int64_t)w8 * 8;
        const e8 g = *(const e8*)(y + at), u = *(const e8*)(y + at + up), d = *(const e8*)(d_out + i * 8);
        e8 dg, du;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const float gf = (float)g[j], df = (float)d[j];
            const float sg = 1.f / (1.f + __expf(-gf));
            du[j] = (E)(df * (float)(E)(gf * sg));
            dg[j] = (E)((float)(E)(df * (float)u[j]) * sg * (1.f + gf * (1.f - sg)));
        }
        *(e8*)(dy + at) = dg;
        *(e8*)(dy + at + up) = du;
    }
}

// ------------------------------------------------------------------------------------------------- casts
template <typename E>
__global__ __launch_bounds__(kThreads) void cast_kernel(CastList a, E* out, int64_t n8) {
    typedef typename Vec<E>::x8 e8;
    for (int64_t i = (int64_t)blockIdx.x * kThreads + threadIdx.x; i < n8; i += (int64_t)gridDim.x * kThreads) {
        const int64_t e = i * 8;
        int t = 0;
        while (e >= a.end[t]) ++t;
        const float* s = a.src[t] + (t ? e - a.end[t - 1] : e);
        const f32x4 lo = *(const f32x4*)s, hi = *(const f32x4*)(s + 4);
        e8 o;
#pragma unroll
        for (int j = 0; j < 4; ++j) { o[j] = (E)lo[j]; o[4 + j] = (E)hi[j]; }
        *(e8*)(out + e) = o;
    }
}

// ------------------------------------------------------------------------------------------------- cross-entropy
__device__ inline int64_t target_of(const int64_t* labels, int row, int len, int64_t ignore) {
    return (row + 1) % len == 0 ? ignore : labels[row + 1];
}

// One workgroup per row, one pass with a running maximum: the logits are read once, as 16-bit.  __expf and __logf are the
// hardware's exp2 and log2 with a factor: the log-sum-exp's error against float64 is a percent or so above that with expf and logf at
// ordinary logits, 5 % at logits of unit scale.
template <typename E>
__global__ __launch_bounds__(kThreads) void loss_fwd_kernel(const E* logits, const int64_t* labels, float* lse, float* row_loss,
                                                            int len, int classes, int64_t ignore) {
    typedef typename Vec<E>::x8 e8;
    __shared__ float sm[kWaves], ss[kWaves];
    const int row = blockIdx.x, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const E* r = logits + (int64_t)row * classes;
    float m = -INFINITY, s = 0.f;
    for (int c = threadIdx.x * 8; c < classes; c += kThreads * 8) {
        const e8 v = *(const e8*)(r + c);
        float f[8], big = m;
#pragma unroll
        for (int j = 0; j < 8; ++j) { f[j] = (float)v[j]; big = fmaxf(big, f[j]); }
        const float base = big == -INFINITY ? 0.f : big;         // a row of -inf so far: nothing to rescale
        s *= __expf(m - base);
#pragma unroll
        for (int j = 0; j < 8; ++j) s += __expf(f[j] - base);
        m = big;
    }
    const float wm = wave_max(m);
    const float ws = wave_sum(s * __expf(m - (wm == -INFINITY ? 0.f : wm)));
    if (lane == 0) { sm[wave] = wm; ss[wave] = ws; }
    __syncthreads();
    if (threadIdx.x == 0) {
        float M = sm[0];
        for (int i = 1; i < kWaves; ++i) M = fmaxf(M, sm[i]);
        float S = 0.f;
        for (int i = 0; i < kWaves; ++i) S += ss[i] * __expf(sm[i] - (M == -INFINITY ? 0.f : M));
        const float l = M + __logf(S);
        lse[row] = l;
        const int64_t t = target_of(labels, row, len, ignore);
        // (a label outside the classes: no number stands for its loss)
        row_loss[row] = t == ignore ? 0.f : (t < 0 || t >= classes) ? NAN : l - (float)r[t];
    }
}

__global__ __launch_bounds__(1024) void loss_mean_kernel(const float* row_loss, const int64_t* labels, float* mean, float* count,
                                                         int rows, int len, int64_t ignore) {
    __shared__ float ss[16], sc[16];
    float s = 0.f, c = 0.f;
    for (int r = threadIdx.x; r < rows; r += 1024) {
        s += row_loss[r];
        c += target_of(labels, r, len, ignore) == ignore ? 0.f : 1.f;
    }
    s = wave_sum(s);
    c = wave_sum(c);
    if ((threadIdx.x & 63) == 0) { ss[threadIdx.x >> 6] = s; sc[threadIdx.x >> 6] = c; }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int i = 1; i < 16; ++i) { s += ss[i]; c += sc[i]; }
        *mean = s / c;
        *count = c;
    }
}

template <typename E>
__global__ __launch_bounds__(kThreads) void loss_bwd_kernel(const E* logits, const int64_t* labels, const float* lse,
                                                            const float* count, const float* d_loss, E* d_logits, int len,
                                                            int classes, int64_t ignore) {
    typedef typename Vec<E>::x8 e8;
    const int row = blockIdx.x;
    const int64_t t = target_of(labels, row, len, ignore);
    const float scale = t == ignore ? 0.f : *d_loss / *count, l = lse[row];
    const E* r = logits + (int64_t)row * classes;
    E* d = d_logits + (int64_t)row * classes;
    for (int c = threadIdx.x * 8; c < classes; c += kThreads * 8) {
        e8 o;
        if (t == ignore) {
#pragma unroll
            for (int j = 0; j < 8; ++j) o[j] = (E)0.f;
        } else {
            const e8 v = *(const e8*)(r + c);
#pragma unroll
            for (int j = 0; j < 8; ++j) o[j] = (E)((__expf((float)v[j] - l) - (c + j == t ? 1.f : 0.f)) * scale);
        }
        *(e8*)(d + c) = o;
    }
}

// ------------------------------------------------------------------------------------------------- clip + AdamW
__device__ inline int tensor_of(const OptTensor* t, int n, int64_t chunk) {
    int lo = 0, hi = n - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (t[mid].first_chunk <= chunk) lo = mid; else hi = mid - 1;
    }
    return lo;
}

__global__ __launch_bounds__(kThreads) void square_sum_kernel(const OptTensor* tensors, int n_tensors, float* partial) {
    __shared__ float ss[kWaves];
    const OptTensor& t = tensors[tensor_of(tensors, n_tensors, blockIdx.x)];
    const int64_t from = (blockIdx.x - t.first_chunk) * kOptChunk, to = from + kOptChunk < t.n ? from + kOptChunk : t.n;
    float s = 0.f;
    for (int64_t i = from + threadIdx.x * 4; i < to; i += kThreads * 4) {
        if (i + 4 <= to) {
            const f32x4 g = *(const f32x4*)(t.g + i);
#pragma unroll
            for (int j = 0; j < 4; ++j) s += g[j] * g[j];
        } else {
            for (int64_t j = i; j < to; ++j) s += t.g[j] * t.g[j];
        }
    }
    s = wave_sum(s);
    if ((threadIdx.x & 63) == 0) ss[threadIdx.x >> 6] = s;
    __syncthreads();
    if (threadIdx.x == 0) partial[blockIdx.x] = ss[0] + ss[1] + ss[2] + ss[3];
}

__global__ __launch_bounds__(1024) void norm_and_steps_kernel(OptTensor* tensors, int n_tensors, int64_t chunks,
                                                              float* partial, float max_norm, float* norm_out) {
    __shared__ double ss[16];
    double s = 0.0;
    for (int64_t i = threadIdx.x; i < chunks; i += 1024) s += (double)partial[i];
    for (int d = 32; d; d >>= 1) s += __shfl_xor(s, d, 64);
    if ((threadIdx.x & 63) == 0) ss[threadIdx.x >> 6] = s;
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int i = 1; i < 16; ++i) s += ss[i];
        const float norm = (float)sqrt(s);
        *norm_out = norm;
        const float c = max_norm / (norm + 1e-6f);
        partial[chunks] = c > 1.f ? 1.f : c;                  // (a norm that is NaN stays NaN)
    }
    for (int i = threadIdx.x; i < n_tensors; i += 1024) {
        OptTensor& t = tensors[i];
        const float step = *t.step + 1.f;
        *t.step = step;
        t.step_size = (float)(t.lr / (1.0 - pow(t.beta1, (double)step)));
        t.denom_scale = (float)(1.0 / sqrt(1.0 - pow(t.beta2, (double)step)));
    }
}

__device__ inline void adamw(float& p, float& g, float& m, float& v, float coef, const OptTensor& t) {
    g *= coef;
    m += t.one_minus_beta1 * (g - m);
    v = t.beta2_f * v + t.one_minus_beta2 * g * g;
    p = p * t.decay - t.step_size * m / (sqrtf(v) * t.denom_scale + t.eps);
}

// One pass over gradient, weight and both moments: 28 bytes a weight, and 4 more when the gradient is clipped, which is
// written back so that a caller finds the clipped one, as after a clipping pass of its own.
// Memory is all that bounds it.  A workgroup takes 1024 weights, four a thread, and ends, so that the launch moves through the seven streams
// on one front, and both ways past the caches, which nothing that follows would find them in.  374 M weights, with the square sums, on rows of a whole
// step: workgroups that walk 16384 weights 2340 us, of 1024 weights 2270, and with non-temporal loads and stores 1980 ... 2020 (6.7 TB/s for this kernel alone).
constexpr int kOptWeights = 4 * kThreads;
static_assert(kOptChunk % kOptWeights == 0, "whole workgroups to a chunk");
__global__ __launch_bounds__(kThreads) void adamw_kernel(const OptTensor* tensors, int n_tensors, const float* clip, int64_t first_chunk) {
    constexpr int kPerChunk = kOptChunk / kOptWeights;
    const int64_t chunk = first_chunk + blockIdx.x / kPerChunk;
    const OptTensor t = tensors[tensor_of(tensors, n_tensors, chunk)];
    const int64_t i = (chunk - t.first_chunk) * kOptChunk + (int64_t)(blockIdx.x % kPerChunk) * kOptWeights + threadIdx.x * 4;
    const float coef = *clip;
    const bool clipped = coef != 1.f;
    if (i + 4 <= t.n) {
        f32x4 g = __builtin_nontemporal_load((const f32x4*)(t.g + i)), p = __builtin_nontemporal_load((const f32x4*)(t.p + i)),
              m = __builtin_nontemporal_load((const f32x4*)(t.m + i)), v = __builtin_nontemporal_load((const f32x4*)(t.v + i));
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            float gj = g[j], pj = p[j], mj = m[j], vj = v[j];
            adamw(pj, gj, mj, vj, coef, t);
            g[j] = gj; p[j] = pj; m[j] = mj; v[j] = vj;
        }
        __builtin_nontemporal_store(p, (f32x4*)(t.p + i));
        __builtin_nontemporal_store(m, (f32x4*)(t.m + i));
        __builtin_nontemporal_store(v, (f32x4*)(t.v + i));
        if (clipped) __builtin_nontemporal_store(g, (f32x4*)(t.g + i));
    } else {
        for (int64_t j = i; j < t.n; ++j) {
            float g = t.g[j], p = t.p[j], m = t.m[j], v = t.v[j];
            adamw(p, g, m, v, coef, t);
            t.p[j] = p; t.m[j] = m; t.v[j] = v;
            if (clipped) t.g[j] = g;
        }
    }
}

__global__ __launch_bounds__(kThreads) void sum_splits_kernel(const float* part, float* out, int64_t n4, int splits) {
    for (int64_t i = (int64_t)blockIdx.x * kThreads + threadIdx.x; i < n4; i += (int64_t)gridDim.x * kThreads) {
        f32x4 s = *(const f32x4*)(part + i * 4);
        for (int k = 1; k < splits; ++k) s += *(const f32x4*)(part + (k * n4 + i) * 4);
        *(f32x4*)(out + i * 4) = s;
    }
}

template <typename E>
__global__ __launch_bounds__(kThreads) void sum_splits_to_kernel(const float* part, E* out, int64_t n8, int splits) {
    typedef typename Vec<E>::x8 e8;
    for (int64_t i = (int64_t)blockIdx.x * kThreads + threadIdx.x; i < n8; i += (int64_t)gridDim.x * kThreads) {
        f32x4 a = *(const f32x4*)(part + i * 8), b = *(const f32x4*)(part + i * 8 + 4);
#pragma unroll 4
        for (int k = 1; k < splits; ++k) {
            const float* more = part + (k * n8 + i) * 8;
            a += *(const f32x4*)more;
            b += *(const f32x4*)(more + 4);
        }
        e8 y;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            y[j] = (E)a[j];
            y[4 + j] = (E)b[j];
        }
        *(e8*)(out + i * 8) = y;
    }
}

unsigned grid_for(int64_t work_items) {
    const int64_t blocks = (work_items + kThreads - 1) / kThreads;
    return (unsigned)(blocks < 1 ? 1 : blocks > 16384 ? 16384 : blocks);
}

template <typename E>
int norm_fwd_t(const NormFwd& a, hipStream_t s) {
    const dim3 grid((a.rows + kWaves - 1) / kWaves), block(kThreads);
#define SBA_NORM(K)                                                                                          \
    if (a.cols <= K * 256) {                                                                                 \
        hipLaunchKernelGGL((norm_fwd_kernel<E, K>), grid, block, 0, s, a);                                   \
        return launched();                                                                                   \
    }
    SBA_NORM(1) SBA_NORM(2) SBA_NORM(4) SBA_NORM(8)
#undef SBA_NORM
    return -2;
}

template <typename E>
int norm_bwd_t(const NormBwd& a, hipStream_t s) {
    const dim3 grid(norm_bwd_parts(a.rows)), block(kThreads);
#define SBA_NORM(K)                                                                                          \
    if (a.cols <= K * 256) {                                                                                 \
        hipLaunchKernelGGL((norm_bwd_kernel<E, K>), grid, block, 0, s, a);                                   \
        return launched();                                                                                   \
    }
    SBA_NORM(1) SBA_NORM(2) SBA_NORM(4) SBA_NORM(8)
#undef SBA_NORM
    return -2;
}

}  // namespace

int norm_fwd(const NormFwd& a, bool f16, hipStream_t s) { return f16 ? norm_fwd_t<_Float16>(a, s) : norm_fwd_t<__bf16>(a, s); }
int norm_bwd(const NormBwd& a, bool f16, hipStream_t s) { return f16 ? norm_bwd_t<_Float16>(a, s) : norm_bwd_t<__bf16>(a, s); }

// two workgroups a CU, fewer when there is not a row for each of their waves (with four rows for each 1024 x 768 took 12.3 us against
// 5.5, 4096 x 1024 18.4 against 14.1; four workgroups a CU: 12.9 there, but 25.9 against 24.9 for 8192 x 1024)
int norm_bwd_parts(int rows) {
    const int by_rows = (rows + kWaves - 1) / kWaves;
    return by_rows < 1 ? 1 : by_rows > 512 ? 512 : by_rows;
}

int sum_parts(const float* const (&part)[2], float* const (&out)[2], int n, int parts, int cols, hipStream_t s) {
    hipLaunchKernelGGL(sum_parts_kernel, dim3((cols + 15) / 16, n), dim3(1024), 0, s, part[0], part[1], out[0], out[1], parts, cols);
    return launched();
}

int swiglu_fwd(const void* y, void* out, int64_t rows, int width, bool f16, hipStream_t s) {
    const int64_t n8 = rows * (width / 8);
    const dim3 grid(grid_for(n8)), block(kThreads);
    if (f16) hipLaunchKernelGGL(swiglu_fwd_kernel<_Float16>, grid, block, 0, s, (const _Float16*)y, (_Float16*)out, n8, width / 8);
    else hipLaunchKernelGGL(swiglu_fwd_kernel<__bf16>, grid, block, 0, s, (const __bf16*)y, (__bf16*)out, n8, width / 8);
    return launched();
}

int swiglu_bwd(const void* y, const void* d_out, void* dy, int64_t rows, int width, bool f16, hipStream_t s) {
    const int64_t n8 = rows * (width / 8);
    const dim3 grid(grid_for(n8)), block(kThreads);
    if (f16)
        hipLaunchKernelGGL(swiglu_bwd_kernel<_Float16>, grid, block, 0, s, (const _Float16*)y, (const _Float16*)d_out, (_Float16*)dy, n8, width / 8);
    else
        hipLaunchKernelGGL(swiglu_bwd_kernel<__bf16>, grid, block, 0, s, (const __bf16*)y, (const __bf16*)d_out, (__bf16*)dy, n8, width / 8);
    return launched();
}

bool weight_grads_fit(const WeightGrads& g) {
    if (g.n < 1 || g.n > 4 || g.k < 1) return false;
    for (int i = 0; i < g.n; ++i) {
        const WeightGrad& p = g.one[i];
        if (p.m < 8 || p.n < 8 || ((p.m | p.n) & 7) || ((p.lda | p.ldb) & 7) || (((uintptr_t)p.a | (uintptr_t)p.b) & 15)) return false;
        // (a stage of 32 rows is addressed with 32-bit byte offsets from its first)
        if (p.lda < p.m || p.ldb < p.n || p.lda >= (1 << 26) || p.ldb >= (1 << 26)) return false;
    }
    return true;
}

// Tile height, and how many workgroups share a tile's contraction.  A launch takes rounds of 1/splits of the rows each, 0.7 us per 32
// rows with 256 x 256 tiles and in proportion for 224 x 256 ones, which leave fewer CUs without work where the taller ones do not
// fill a round (the 340M model's block over 8192 rows, 235 tiles instead of 196: 184 against 196 us); tiles are dealt to the XCDs
// in eight equal parts, the last of them short, so that a round is full when the first XCD's CUs are.  Results are written, partial
// sums written, read and summed at about 5.5 TB/s.
int weight_grad_splits(WeightGrads& g, int cus) {
    auto tiles_of = [&](int i, int rows) { return ((g.one[i].m + rows - 1) / rows) * ((g.one[i].n + 255) / 256); };
    g.total = 0;
    for (int i = 0; i < g.n; ++i) {
        g.one[i].at = g.total;
        g.total += (int64_t)g.one[i].m * g.one[i].n;
    }
    const double stages = (g.k + 31) / 32;
    int best = 1;
    double best_us = 1e30;
    for (int rows : {256, 224}) {
        int64_t tiles = 0;
        for (int i = 0; i < g.n; ++i) tiles += tiles_of(i, rows);
        for (int s = 1; s <= 16 && s * 4 <= stages + 3; ++s) {
            const int64_t on_xcd = (tiles + 7) / 8 * s, slots = cus > 8 ? cus / 8 : 1;
            const double rounds = (double)((on_xcd + slots - 1) / slots);
            const double us = rounds * (0.7 * rows / 256 * stages / s + 3.0) + (s > 1 ? 2 * s + 1 : 1) * 4.0 * g.total / 5.5e6 + (s > 1 ? 3.0 : 0.0);
            if (us < best_us) { best_us = us; best = s; g.tile_rows = rows; }
        }
    }
    g.tiles = 0;
    for (int i = 0; i < g.n; ++i) {
        g.first_tile[i] = g.tiles;
        g.tiles += tiles_of(i, g.tile_rows);
    }
    return best;
}

// Time estimates in us of the projection kernels (sba_gemm.hip), fitted to sweeps of 300 .. 8192 rows, 512 .. 5632 features and k of 512
// .. 5632 with every epilogue and of plain products of k up to 32000 (333 products: the tile chosen takes 0.5 % more than the best on the
// average, 15 % at most).  Tiles are dealt to the XCDs in equal parts, so the fullest one's count: whole rounds of its resident workgroups,
// each k / 64 times `rate` of a full CU, then a last one at the rate of as many workgroups a CU as are left (one on half of the CUs or
// less: `half` of that rate, what lies between in proportion); `round` and what the epilogue adds that nothing hides, per round
// and in proportion to its fill; `launch`.
// Where each is ahead (us): 256 x 256 8192 x 5632 of swiglu, k = 1024 (92, next 99); 128 x 256 8192 x 3072, k = 1024 (47; 49);
// 128 x 128 two a CU 8192 x 2816 with the swiglu gradient, k = 1024 (69; 86), 8192 x 1024 with the residual, k = 2816 (47; 49); by halves
// 4096 x 1024, k = 5632 (49; 59); 64 x 64 three a CU 2048 x 2304, k = 768 (12.4; 13.3), 1500 x 2816 with the swiglu gradient, k = 1024 (20.8;
// 23.4); by halves 1024 x 768, k = 4096 (14.6; 18.5).
double tile_time(const Projection& p, ProjectionTile tile, int cus) {
    struct { int rows, features, per_cu; double rate[3], half, round, launch, add, swiglu_fwd, swiglu_bwd; } static const cost[] = {
        {256, 256, 1, {1.24}, 0.87, 3.8, 7.0, 0.0, 2.4, 0.0},                   // kTile256
        {128, 256, 1, {0.786}, 0.86, 1.0, 5.8, 10.5, 1.2, 0.0},                 // kTile128x256
        {128, 128, 2, {0.647, 0.85}, 0.95, 2.9, 2.2, 7.7, 0.3, 10.5},          // kTile128
        {128, 128, 1, {0.542}, 0.89, 1.3, 3.5, 3.8, 0.7, 7.5},                  // kTile128Halves
        {64, 64, 3, {0.256, 0.365, 0.551}, 0.90, 0.0, 2.7, 2.1, 0.0, 3.1},      // kTile64
        {64, 64, 1, {0.211}, 0.88, 1.0, 2.6, 0.5, 0.0, 1.6},                    // kTile64Halves
    };
    const auto& c = cost[tile];
    const bool glu = p.epilogue == kSwigluFwd;
    if (tile <= kTile128x256 && (p.k % 64 || p.epilogue == kSwigluBwd)) return 1e30;
    if (tile == kTile256 && p.epilogue == kAddResidual) return 1e30;       // its registers
    if (tile >= kTile64 && glu) return 1e30;
    const int64_t own = glu ? c.features / 2 : c.features, features = glu ? p.n / 2 : p.n;
    const int64_t tiles = (((int64_t)p.m + c.rows - 1) / c.rows * ((features + own - 1) / own) + 7) / 8, wide = std::max(cus / 8, 1);
    const int64_t rounds = tiles / (wide * c.per_cu), left = tiles % (wide * c.per_cu), deep = (left + wide - 1) / wide;
    const double round = c.round + (p.epilogue == kAddResidual ? c.add : glu ? c.swiglu_fwd : p.epilogue == kSwigluBwd ? c.swiglu_bwd : 0.0);
    const double k64 = (p.k + 63) / 64, fill = (double)left / wide;
    double us = rounds * (c.rate[c.per_cu - 1] * k64 + round) + c.launch;
    if (left) us += c.rate[deep - 1] * (deep > 1 ? 1.0 : c.half + (1.0 - c.half) * std::max(2.0 * fill - 1.0, 0.0)) * k64 + round * fill / c.per_cu;
    return us;
}

bool addresses(const Projection& p) {
    return p.k % 32 == 0 && p.k > 0 && p.n % (p.epilogue == kSwigluFwd ? 16 : 8) == 0 && p.n > 0 && p.m > 0 && p.ldx % 8 == 0 &&
           p.ldw % 8 == 0 && ((uintptr_t)p.x & 15) == 0 && ((uintptr_t)p.w & 15) == 0 && p.ldx < (1 << 22) && p.ldw < (1 << 22) &&
           (int64_t)(p.rows_w ? p.k : p.n) * p.ldw < (INT64_C(1) << 31);
}

bool projects(const Projection& p, int cus) {
    if (!addresses(p)) return false;
    if (p.epilogue == kSwigluBwd) {
        // against the plain product and a pass of its own, which reads and writes 12 bytes per product at 7.7 TB/s (much of it still in
        // the last-level cache): 8192 x 2816, k = 1024 69 against 48 + 36 us (91 in a training step)
        Projection plain = p;
        plain.epilogue = kStore;
        return tile_time(p, projection_tile(p, cus), cus) < tile_time(plain, projection_tile(plain, cus), cus) + 12e-6 * p.m * p.n / 7.7 + 1.5;
    }
    // plain products of four rounds of the largest tile and more (the language model's head): the library's is ahead there, 436 against
    // 466 us for 8192 x 32000, k = 1024
    return p.epilogue != kStore || p.rows_w || (int64_t)p.m * p.n < (int64_t)4 * 256 * 256 * cus;
}

ProjectionTile projection_tile(const Projection& p, int cus) {
    ProjectionTile best = kTile128;
    double best_us = 1e30;
    for (int t = kTile256; t <= kTile64Halves; ++t) {
        const double us = tile_time(p, (ProjectionTile)t, cus);
        if (us < best_us) { best = (ProjectionTile)t; best_us = us; }
    }
    return best;
}

// Long contractions over few tiles (the input gradient of a language model's head): the large tiles' kernels with as many workgroups to a
// tile as the CUs allow, their fp32 sums written, read and added at 5.5 TB/s.  (1.4 us a stage of 256 rows: a full chip slows from 1.38 to
// 1.59 in contractions as long as these, and tile_time()'s 1.24 fits shorter ones.)  k = 32000, one workgroup a tile against several (us): 300 x 768
// 94, 57;  1024 x 1024 121, 76;  2048 x 1024 208, 120;  3000 x 768 244, 150;  4096 x 1024 355, 237;  8192 x 1024 436, 423;  k = 8192:
// 2048 x 1024 52, 43;  4096 x 1024 68 either way;  k = 5632: 3000 x 768 48, 39.
int projection_splits(const Projection& p, int cus, ProjectionTile& tile) {
    tile = projection_tile(p, cus);
    if (!p.rows_w || p.epilogue != kStore || p.k % 64 || p.k < 4096) return 1;
    double best_us = tile_time(p, tile, cus);
    int best = 1;
    const int stages = p.k / 64;
    for (ProjectionTile t : {kTile256, kTile128x256}) {
        const int rows = t == kTile256 ? 256 : 128;
        const int tiles = (int)((((int64_t)p.m + rows - 1) / rows * ((p.n + 255) / 256) + 7) / 8 * 8);
        for (int splits = 2; splits <= 16 && tiles * splits <= cus; ++splits) {
            const int per = (stages + splits - 1) / splits;
            if ((stages + per - 1) / per != splits) continue;          // (the last one would have nothing)
            const double fill = (double)tiles * splits / cus, rate = (t == kTile256 ? 1.4 : 0.786) * (0.87 + 0.13 * std::max(2.0 * fill - 1.0, 0.0));
            const double us = (t == kTile256 ? 11.0 : 9.0) + rate * per + (8.0 * splits + 2.0) * p.m * p.n / 5.5e6;
            if (us < 0.9 * best_us) { best_us = us / 0.9; best = splits; tile = t; }
        }
    }
    return best;
}

int project_tile(const Projection& p, ProjectionTile tile, bool f16, hipStream_t s) {
    const int rc = f16 ? project_f16(p, tile, s) : project_bf16(p, tile, s);
    if (rc || p.splits < 2) return rc;
    const int64_t n8 = (int64_t)p.m * p.n / 8;
    const dim3 grid(grid_for(n8)), block(kThreads);
    if (f16) hipLaunchKernelGGL(sum_splits_to_kernel<_Float16>, grid, block, 0, s, p.partial, (_Float16*)p.out, n8, p.splits);
    else hipLaunchKernelGGL(sum_splits_to_kernel<__bf16>, grid, block, 0, s, p.partial, (__bf16*)p.out, n8, p.splits);
    return launched();
}

int weight_grads(const WeightGrads& g, int splits, bool f16, hipStream_t s) {
    if (!weight_grads_fit(g)) return -2;
    const int rc = f16 ? weight_grads_f16(g, splits, s) : weight_grads_bf16(g, splits, s);
    if (rc || splits == 1) return rc;
    hipLaunchKernelGGL(sum_splits_kernel, dim3(grid_for(g.total / 4)), dim3(kThreads), 0, s, g.partial, g.out, g.total / 4, splits);
    return launched();
}

int cast_list(const CastList& a, void* out, bool f16, hipStream_t s) {
    const int64_t n8 = a.end[a.n - 1] / 8;
    const dim3 grid(grid_for(n8)), block(kThreads);
    if (f16) hipLaunchKernelGGL(cast_kernel<_Float16>, grid, block, 0, s, a, (_Float16*)out, n8);
    else hipLaunchKernelGGL(cast_kernel<__bf16>, grid, block, 0, s, a, (__bf16*)out, n8);
    return launched();
}

int cast_one(const float* src, void* out, int64_t n, bool f16, hipStream_t s) {
    CastList a = {};
    a.src[0] = src;
    a.end[0] = n;
    a.n = 1;
    return cast_list(a, out, f16, s);
}

int loss_fwd(const void* logits, const int64_t* labels, float* lse, float* row_loss, float* mean, float* count, int rows, int len,
             int classes, int64_t ignore, bool f16, hipStream_t s) {
    if (f16)
        hipLaunchKernelGGL(loss_fwd_kernel<_Float16>, dim3(rows), dim3(kThreads), 0, s, (const _Float16*)logits, labels, lse, row_loss, len, classes, ignore);
    else
        hipLaunchKernelGGL(loss_fwd_kernel<__bf16>, dim3(rows), dim3(kThreads), 0, s, (const __bf16*)logits, labels, lse, row_loss, len, classes, ignore);
    hipLaunchKernelGGL(loss_mean_kernel, dim3(1), dim3(1024), 0, s, row_loss, labels, mean, count, rows, len, ignore);
    return launched();
}

int loss_bwd(const void* logits, const int64_t* labels, const float* lse, const float* count, const float* d_loss,
             void* d_logits, int rows, int len, int classes, int64_t ignore, bool f16, hipStream_t s) {
    if (f16)
        hipLaunchKernelGGL(loss_bwd_kernel<_Float16>, dim3(rows), dim3(kThreads), 0, s, (const _Float16*)logits, labels, lse, count, d_loss, (_Float16*)d_logits, len, classes, ignore);
    else
        hipLaunchKernelGGL(loss_bwd_kernel<__bf16>, dim3(rows), dim3(kThreads), 0, s, (const __bf16*)logits, labels, lse, count, d_loss, (__bf16*)d_logits, len, classes, ignore);
    return launched();
}

int clip_and_adamw(OptTensor* tensors, int n_tensors, int64_t chunks, float max_norm, float* partial, float* norm,
                   hipStream_t s) {
    hipLaunchKernelGGL(square_sum_kernel, dim3((unsigned)chunks), dim3(kThreads), 0, s, tensors, n_tensors, partial);
    hipLaunchKernelGGL(norm_and_steps_kernel, dim3(1), dim3(1024), 0, s, tensors, n_tensors, chunks, partial, max_norm, norm);
    for (int64_t first = 0; first < chunks; first += 1 << 19) {          // (a grid has fewer than 2^32 threads)
        const unsigned n = (unsigned)(chunks - first < 1 << 19 ? chunks - first : 1 << 19);
        hipLaunchKernelGGL(adamw_kernel, dim3(n * (kOptChunk / kOptWeights)), dim3(kThreads), 0, s, tensors, n_tensors, partial + chunks, first);
    }
    return launched();
}

}  // namespace sba_model
