// dh_rows.hip -- row-wise kernels on gfx950: softmax / log_softmax and layer norm, forward and
// backward, fp32, rows of C contiguous values.
//
// Replaces the reference's scalar per-row loops: dream_softmax (runtime/ops/elementwise.inc:
// 338-358), dream_log_softmax (elementwise.inc:1550-1570), dream_layer_norm
// (runtime/io/builtins.inc:167-188) and their backward branches (runtime/ops/autograd.inc:
// 212-233, 396-409, 453-471).  All four are HBM-bound: each reads its inputs once and writes
// its output once.
//
// Rows of up to 1024 values: a segment of G lanes (G = 4, 16 or 64, the smallest that holds
// the row in at most 16 values per lane) owns one row and keeps it in registers, so every
// statistic (max, sums, mean, variance) is a segment reduction over registers and no value is
// read twice.  Lane s of a segment holds chunks s, s + G, s + 2G, ... of the row, so one load
// instruction covers G consecutive chunks of every row in the wave.
// Rows of up to 32768 values: one work-group per row holds it the same way (see row_block).
// Longer rows: one 256-thread work-group per row, streaming the row from L2 once per pass.
//
// A chunk is 4 values, loaded and stored as one 16-byte access that needs only the 4-byte
// alignment every row has: rows of any C and any pointer take the same path, and only the
// chunk that holds a row's end goes value by value.
#include "dh_common.hpp"

namespace dh {
namespace {

template <int G>
__device__ inline float seg_sum(float v) {
#pragma unroll
    for (int m = 1; m < G; m <<= 1) v += __shfl_xor(v, m, 64);
    return v;
}
template <int G>
__device__ inline float seg_max(float v) {
#pragma unroll
    for (int m = 1; m < G; m <<= 1) v = fmaxf(v, __shfl_xor(v, m, 64));
    return v;
}

// 16-byte access at 4-byte alignment.
typedef float f4u __attribute__((ext_vector_type(4), aligned(4)));

// NV chunks of 4 values of one row over g lanes, chunk t of lane s at element 4 (t g + s).
template <int NV>
struct Row {
    float v[NV][4];
    __device__ void load(const float* __restrict__ p, int C, int s, int g, float fill) {
#pragma unroll
        for (int t = 0; t < NV; ++t) {
            const int e = 4 * (t * g + s);
            if (e + 4 <= C) {
                const f4u x = *reinterpret_cast<const f4u*>(p + e);
#pragma unroll
                for (int q = 0; q < 4; ++q) v[t][q] = x[q];
            } else {
#pragma unroll
                for (int q = 0; q < 4; ++q) v[t][q] = e + q < C ? p[e + q] : fill;
            }
        }
    }
    // Non-temporal: the output row is streamed out and not read again here, and keeping it
    // out of the caches leaves them to the inputs.
    __device__ void store(float* __restrict__ p, int C, int s, int g) const {
#pragma unroll
        for (int t = 0; t < NV; ++t) {
            const int e = 4 * (t * g + s);
            if (e + 4 <= C) {
                __builtin_nontemporal_store(f4u{v[t][0], v[t][1], v[t][2], v[t][3]},
                                            reinterpret_cast<f4u*>(p + e));
            } else {
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    if (e + q < C) __builtin_nontemporal_store(v[t][q], p + e + q);
            }
        }
    }
};

#define ROW_LOOP(stmt)                              \
    _Pragma("unroll") for (int t = 0; t < NV; ++t)  \
        _Pragma("unroll") for (int q = 0; q < 4; ++q) { stmt; }

// Reductions over the lanes that hold a row: a segment of G lanes within a wave, or a whole
// work-group (wave sums through LDS, added in wave order).
template <int G>
struct SegLanes {
    __device__ float sum(float v) const { return seg_sum<G>(v); }
    __device__ float max(float v) const { return seg_max<G>(v); }
};

template <typename Op>
__device__ inline float block_reduce(float v, Op op, float* red) {
    v = wave_reduce(v, op);
    const int w = threadIdx.x >> 6, nw = blockDim.x >> 6;
    __syncthreads();   // red[] may still be read from a previous reduction
    if ((threadIdx.x & 63) == 0) red[w] = v;
    __syncthreads();
    v = red[0];
    for (int i = 1; i < nw; ++i) v = op(v, red[i]);
    return v;
}

struct BlockLanes {
    float* red;   // 16 floats of LDS
    __device__ float sum(float v) const { return block_reduce(v, OpSum(), red); }
    __device__ float max(float v) const { return block_reduce(v, OpMax(), red); }
};

// The four row operations on a row held by g lanes, lane s (`L` reduces over them); off is the
// row's first element.
template <int NV, typename L>
__device__ inline void softmax_row(const float* __restrict__ X, float* __restrict__ Y, size_t off,
                                   int C, int s, int g, L lanes, int logsm) {
    Row<NV> x;
    x.load(X + off, C, s, g, -INFINITY);
    float mx = -INFINITY;
    ROW_LOOP(mx = fmaxf(mx, x.v[t][q]));
    mx = lanes.max(mx);
    float sum = 0.f;
    if (logsm) {
        ROW_LOOP(sum += __expf(x.v[t][q] - mx));
        const float lse = mx + __logf(lanes.sum(sum));
        ROW_LOOP(x.v[t][q] -= lse);
    } else {
        ROW_LOOP(x.v[t][q] = __expf(x.v[t][q] - mx); sum += x.v[t][q]);
        const float inv = 1.f / lanes.sum(sum);
        ROW_LOOP(x.v[t][q] *= inv);
    }
    x.store(Y + off, C, s, g);
}

// softmax:     gx (+)= y (g - sum(g y))
// log_softmax: gx (+)= g - exp(y) sum(g)      (y = log_softmax(x), so exp(y) = softmax(x))
template <int NV, typename L>
__device__ inline void softmax_bwd_row(const float* __restrict__ Yf, const float* __restrict__ Gr,
                                       float* __restrict__ GX, size_t off, int C, int s, int g,
                                       L lanes, int logsm, int acc) {
    Row<NV> y, d;
    y.load(Yf + off, C, s, g, 0.f);
    d.load(Gr + off, C, s, g, 0.f);
    float red = 0.f;
    if (logsm) {
        ROW_LOOP(red += d.v[t][q]);
    } else {
        ROW_LOOP(red += d.v[t][q] * y.v[t][q]);
    }
    red = lanes.sum(red);
    if (logsm) {
        ROW_LOOP(y.v[t][q] = d.v[t][q] - __expf(y.v[t][q]) * red);
    } else {
        ROW_LOOP(y.v[t][q] = y.v[t][q] * (d.v[t][q] - red));
    }
    if (acc) {
        Row<NV> o;
        o.load(GX + off, C, s, g, 0.f);
        ROW_LOOP(y.v[t][q] += o.v[t][q]);
    }
    y.store(GX + off, C, s, g);
}

// Per-row mean and inverse standard deviation (biased variance, eps 1e-5) from registers;
// padding chunks hold 0 and are excluded from the variance by the element count.
template <int NV, typename L>
__device__ inline void row_stats(const Row<NV>& x, int C, int s, int g, L lanes, float& mu,
                                 float& inv_std) {
    float sum = 0.f;
    ROW_LOOP(sum += x.v[t][q]);
    mu = lanes.sum(sum) / (float)C;
    float var = 0.f;
#pragma unroll
    for (int t = 0; t < NV; ++t)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const float d = 4 * (t * g + s) + q < C ? x.v[t][q] - mu : 0.f;
            var += d * d;
        }
    var = lanes.sum(var) / (float)C;
    inv_std = rsqrtf(var + 1e-5f);
}

template <int NV, typename L>
__device__ inline void layer_norm_row(const float* __restrict__ X, float* __restrict__ Y,
                                      size_t off, int C, int s, int g, L lanes) {
    Row<NV> x;
    x.load(X + off, C, s, g, 0.f);
    float mu, inv_std;
    row_stats(x, C, s, g, lanes, mu, inv_std);
    ROW_LOOP(x.v[t][q] = (x.v[t][q] - mu) * inv_std);
    x.store(Y + off, C, s, g);
}

// gx (+)= inv_std / C (C dy - sum(dy) - y sum(dy y)), inv_std recomputed from x.
template <int NV, typename L>
__device__ inline void layer_norm_bwd_row(const float* __restrict__ X, const float* __restrict__ Yf,
                                          const float* __restrict__ DY, float* __restrict__ GX,
                                          size_t off, int C, int s, int g, L lanes, int acc) {
    float mu, inv_std;
    {
        Row<NV> x;
        x.load(X + off, C, s, g, 0.f);
        row_stats(x, C, s, g, lanes, mu, inv_std);
    }
    Row<NV> y, dy;
    y.load(Yf + off, C, s, g, 0.f);
    dy.load(DY + off, C, s, g, 0.f);
    float sdy = 0.f, sdyy = 0.f;
    ROW_LOOP(sdy += dy.v[t][q]; sdyy += dy.v[t][q] * y.v[t][q]);
    sdy = lanes.sum(sdy);
    sdyy = lanes.sum(sdyy);
    const float k = inv_std / (float)C, fc = (float)C;
    ROW_LOOP(y.v[t][q] = k * (fc * dy.v[t][q] - sdy - y.v[t][q] * sdyy));
    if (acc) {
        Row<NV> o;
        o.load(GX + off, C, s, g, 0.f);
        ROW_LOOP(y.v[t][q] += o.v[t][q]);
    }
    y.store(GX + off, C, s, g);
}

// Segment kernels, rows of at most 16 G values: 256 threads = 256 / G rows per work-group; a
// row index past R exits the whole segment (segments never straddle a wave, so the reductions
// stay within live lanes).
#define SEG_PROLOGUE()                                                    \
    const int s = threadIdx.x & (G - 1);                                  \
    const int row = blockIdx.x * (256 / G) + threadIdx.x / G;             \
    if (row >= R) return;                                                 \
    const size_t off = (size_t)row * C;

template <int G>
__global__ void __launch_bounds__(256) softmax_seg(const float* __restrict__ X,
                                                   float* __restrict__ Y, int R, int C, int logsm) {
    SEG_PROLOGUE();
    softmax_row<4>(X, Y, off, C, s, G, SegLanes<G>(), logsm);
}
template <int G>
__global__ void __launch_bounds__(256) softmax_bwd_seg(const float* __restrict__ Yf,
                                                       const float* __restrict__ Gr,
                                                       float* __restrict__ GX, int R, int C,
                                                       int logsm, int acc) {
    SEG_PROLOGUE();
    softmax_bwd_row<4>(Yf, Gr, GX, off, C, s, G, SegLanes<G>(), logsm, acc);
}
template <int G>
__global__ void __launch_bounds__(256) layer_norm_seg(const float* __restrict__ X,
                                                      float* __restrict__ Y, int R, int C) {
    SEG_PROLOGUE();
    layer_norm_row<4>(X, Y, off, C, s, G, SegLanes<G>());
}
template <int G>
__global__ void __launch_bounds__(256) layer_norm_bwd_seg(const float* __restrict__ X,
                                                          const float* __restrict__ Yf,
                                                          const float* __restrict__ DY,
                                                          float* __restrict__ GX, int R, int C,
                                                          int acc) {
    SEG_PROLOGUE();
    layer_norm_bwd_row<4>(X, Yf, DY, GX, off, C, s, G, SegLanes<G>(), acc);
}

// row_block: one work-group per row of 1025 to 32768 values, held in registers at 4 NV values
// per lane (NV = 4 up to 16384, then 8; blockDim.x = the fewest whole waves that hold it).
// Bound by HBM: each input is read once and the output written once, where the streaming
// kernels below read the row once per pass.  Same box, 4096 x 5000 log_softmax, streaming /
// registers: forward 62.6 / 25.5 us, backward 59.9 / 38.2 us (6.4 and 6.4 TB/s).
template <int NV>
__global__ void __launch_bounds__(1024) softmax_block(const float* __restrict__ X,
                                                      float* __restrict__ Y, int C, int logsm) {
    __shared__ float red[16];
    softmax_row<NV>(X, Y, (size_t)blockIdx.x * C, C, threadIdx.x, blockDim.x, BlockLanes{red},
                    logsm);
}
template <int NV>
__global__ void __launch_bounds__(1024) softmax_bwd_block(const float* __restrict__ Yf,
                                                          const float* __restrict__ Gr,
                                                          float* __restrict__ GX, int C, int logsm,
                                                          int acc) {
    __shared__ float red[16];
    softmax_bwd_row<NV>(Yf, Gr, GX, (size_t)blockIdx.x * C, C, threadIdx.x, blockDim.x,
                        BlockLanes{red}, logsm, acc);
}
template <int NV>
__global__ void __launch_bounds__(1024) layer_norm_block(const float* __restrict__ X,
                                                         float* __restrict__ Y, int C) {
    __shared__ float red[16];
    layer_norm_row<NV>(X, Y, (size_t)blockIdx.x * C, C, threadIdx.x, blockDim.x, BlockLanes{red});
}
template <int NV>
__global__ void __launch_bounds__(1024) layer_norm_bwd_block(const float* __restrict__ X,
                                                             const float* __restrict__ Yf,
                                                             const float* __restrict__ DY,
                                                             float* __restrict__ GX, int C,
                                                             int acc) {
    __shared__ float red[16];
    layer_norm_bwd_row<NV>(X, Yf, DY, GX, (size_t)blockIdx.x * C, C, threadIdx.x, blockDim.x,
                           BlockLanes{red}, acc);
}

// ---- rows above 32768 values: one work-group of 256 threads per row, streaming --------------
__global__ void __launch_bounds__(256) softmax_blk(const float* __restrict__ X,
                                                   float* __restrict__ Y, int C, int logsm) {
    __shared__ float red[4];
    const float* x = X + (size_t)blockIdx.x * C;
    float* y = Y + (size_t)blockIdx.x * C;
    float mx = -INFINITY;
    for (int j = threadIdx.x; j < C; j += 256) mx = fmaxf(mx, x[j]);
    mx = block_reduce(mx, OpMax(), red);
    float sum = 0.f;
    for (int j = threadIdx.x; j < C; j += 256) sum += __expf(x[j] - mx);
    sum = block_reduce(sum, OpSum(), red);
    if (logsm) {
        const float lse = mx + __logf(sum);
        for (int j = threadIdx.x; j < C; j += 256) y[j] = x[j] - lse;
    } else {
        const float inv = 1.f / sum;
        for (int j = threadIdx.x; j < C; j += 256) y[j] = __expf(x[j] - mx) * inv;
    }
}

__global__ void __launch_bounds__(256) softmax_bwd_blk(const float* __restrict__ Yf,
                                                       const float* __restrict__ Gr,
                                                       float* __restrict__ GX, int C, int logsm,
                                                       int acc) {
    __shared__ float red[4];
    const size_t off = (size_t)blockIdx.x * C;
    const float *y = Yf + off, *g = Gr + off;
    float* gx = GX + off;
    float r = 0.f;
    for (int j = threadIdx.x; j < C; j += 256) r += logsm ? g[j] : g[j] * y[j];
    r = block_reduce(r, OpSum(), red);
    for (int j = threadIdx.x; j < C; j += 256) {
        const float v = logsm ? g[j] - __expf(y[j]) * r : y[j] * (g[j] - r);
        gx[j] = acc ? gx[j] + v : v;
    }
}

__device__ inline void blk_stats(const float* x, int C, float* red, float& mu, float& inv_std) {
    float sum = 0.f;
    for (int j = threadIdx.x; j < C; j += 256) sum += x[j];
    mu = block_reduce(sum, OpSum(), red) / (float)C;
    float var = 0.f;
    for (int j = threadIdx.x; j < C; j += 256) {
        const float d = x[j] - mu;
        var += d * d;
    }
    inv_std = rsqrtf(block_reduce(var, OpSum(), red) / (float)C + 1e-5f);
}

__global__ void __launch_bounds__(256) layer_norm_blk(const float* __restrict__ X,
                                                      float* __restrict__ Y, int C) {
    __shared__ float red[4];
    const float* x = X + (size_t)blockIdx.x * C;
    float* y = Y + (size_t)blockIdx.x * C;
    float mu, inv_std;
    blk_stats(x, C, red, mu, inv_std);
    for (int j = threadIdx.x; j < C; j += 256) y[j] = (x[j] - mu) * inv_std;
}

__global__ void __launch_bounds__(256) layer_norm_bwd_blk(const float* __restrict__ X,
                                                          const float* __restrict__ Yf,
                                                          const float* __restrict__ DY,
                                                          float* __restrict__ GX, int C, int acc) {
    __shared__ float red[4];
    const size_t off = (size_t)blockIdx.x * C;
    const float *x = X + off, *y = Yf + off, *dy = DY + off;
    float* gx = GX + off;
    float mu, inv_std;
    blk_stats(x, C, red, mu, inv_std);
    float sdy = 0.f, sdyy = 0.f;
    for (int j = threadIdx.x; j < C; j += 256) {
        sdy += dy[j];
        sdyy += dy[j] * y[j];
    }
    sdy = block_reduce(sdy, OpSum(), red);
    sdyy = block_reduce(sdyy, OpSum(), red);
    const float k = inv_std / (float)C, fc = (float)C;
    for (int j = threadIdx.x; j < C; j += 256) {
        const float v = k * (fc * dy[j] - sdy - y[j] * sdyy);
        gx[j] = acc ? gx[j] + v : v;
    }
}

// ---- linear backward: ReLU mask and bias gradient ------------------------------------------
// Work-group (bx, by): 64 columns (one per lane, so each row's piece is one coalesced load) and
// the rows by, by + P, by + 2P, ... split over its 4 waves, BG_ROWS of them loaded before the
// first is used.  Partial column sums go to part[by][col] and a second pass adds the P partials
// in a fixed order: no atomics, so reruns are bit-identical.
constexpr int BG_ROWS = 8;

__global__ void __launch_bounds__(256) bias_grad_partial(const float* __restrict__ Y,
                                                         float* __restrict__ dY,
                                                         float* __restrict__ part, int N,
                                                         int out, int relu) {
    __shared__ float red[4][64];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int col = blockIdx.x * 64 + lane;
    const int P = gridDim.y;
    float s = 0.f;
    if (col < out) {
        for (int i0 = blockIdx.y + P * w; i0 < N; i0 += 4 * P * BG_ROWS) {
            float g[BG_ROWS], y[BG_ROWS];
#pragma unroll
            for (int r = 0; r < BG_ROWS; ++r) {   // past the end: row i0 again, so no branch per load
                const long long i = i0 + 4LL * P * r;
                const size_t e = (size_t)(i < N ? i : i0) * out + col;
                g[r] = dY[e];
                y[r] = relu ? Y[e] : 1.f;
            }
#pragma unroll
            for (int r = 0; r < BG_ROWS; ++r) {
                const long long i = i0 + 4LL * P * r;
                if (i >= N) break;
                if (!(y[r] > 0.f)) {   // the reference zeroes dY where Y <= 0, in place
                    g[r] = 0.f;
                    dY[(size_t)i * out + col] = 0.f;
                }
                s += g[r];
            }
        }
    }
    red[w][lane] = s;
    __syncthreads();
    if (w == 0 && col < out)
        part[(size_t)blockIdx.y * out + col] = (red[0][lane] + red[1][lane]) + (red[2][lane] + red[3][lane]);
}

// Latency-bound (at most 1024 partials of 64 columns): 16 waves share a column group's
// partials and add through LDS in wave order.  P = 64 partials of 257 columns: 4.7 us
// (16.1 us with one thread adding a column's partials one after the other).
__global__ void __launch_bounds__(1024) bias_grad_final(const float* __restrict__ part,
                                                        float* __restrict__ db, int P, int out,
                                                        int acc) {
    __shared__ float red[16][64];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int col = blockIdx.x * 64 + lane;
    float s = 0.f;
    if (col < out)
#pragma unroll 4
        for (int p = w; p < P; p += 16) s += part[(size_t)p * out + col];
    red[w][lane] = s;
    __syncthreads();
    if (w != 0 || col >= out) return;
#pragma unroll
    for (int i = 1; i < 16; ++i) s += red[i][lane];
    db[col] = acc ? db[col] + s : s;
}

// ---- dispatch --------------------------------------------------------------------------------
constexpr int SEG_MAX_C = 1024, BLOCK_MAX_C = 32768;

// Launches the segment, row_block or streaming form of a row operation for R rows of C values:
// KERNEL_seg<G>(ARGS, R, C, ...), KERNEL_block<NV>(ARGS, C, ...) or KERNEL_blk(ARGS, C, ...).
#define ROW_LAUNCH(KERNEL, WHAT, R, C, ARGS, ...)                                               \
    do {                                                                                        \
        if ((C) <= 64) KERNEL##_seg<4><<<((R) + 63) / 64, 256, 0, stream()>>>(                  \
            UNPAREN ARGS, R, C __VA_OPT__(, ) __VA_ARGS__);                                     \
        else if ((C) <= 256) KERNEL##_seg<16><<<((R) + 15) / 16, 256, 0, stream()>>>(           \
            UNPAREN ARGS, R, C __VA_OPT__(, ) __VA_ARGS__);                                     \
        else if ((C) <= SEG_MAX_C) KERNEL##_seg<64><<<((R) + 3) / 4, 256, 0, stream()>>>(       \
            UNPAREN ARGS, R, C __VA_OPT__(, ) __VA_ARGS__);                                     \
        else if ((C) <= BLOCK_MAX_C / 2) KERNEL##_block<4><<<R, 64 * (((C) + 1023) / 1024), 0,  \
                                                             stream()>>>(                       \
            UNPAREN ARGS, C __VA_OPT__(, ) __VA_ARGS__);                                        \
        else if ((C) <= BLOCK_MAX_C) KERNEL##_block<8><<<R, 64 * (((C) + 2047) / 2048), 0,      \
                                                         stream()>>>(                           \
            UNPAREN ARGS, C __VA_OPT__(, ) __VA_ARGS__);                                        \
        else KERNEL##_blk<<<R, 256, 0, stream()>>>(UNPAREN ARGS, C __VA_OPT__(, ) __VA_ARGS__); \
        return check_launch(WHAT);                                                              \
    } while (0)
#define UNPAREN(...) __VA_ARGS__

int check_rows(const char* op, int R, int C) {
    if (R < 0 || C < 0) return set_error(DH_ERR_INVALID, "%s: negative shape", op);
    return DH_OK;
}

}  // namespace
}  // namespace dh

using namespace dh;

extern "C" {

int dh_row_softmax(const float* X, float* Y, int R, int C, int log_softmax) {
    DH_TRY(ensure_init());
    DH_TRY(check_rows("dh_row_softmax", R, C));
    if (R == 0 || C == 0) return DH_OK;
    if (!X || !Y) return set_error(DH_ERR_INVALID, "dh_row_softmax: null pointer");
    ROW_LAUNCH(softmax, "dh_row_softmax", R, C, (X, Y), log_softmax);
}

int dh_row_softmax_bwd(const float* Y, const float* G, float* GX, int R, int C, int log_softmax,
                       int accumulate) {
    DH_TRY(ensure_init());
    DH_TRY(check_rows("dh_row_softmax_bwd", R, C));
    if (R == 0 || C == 0) return DH_OK;
    if (!Y || !G || !GX) return set_error(DH_ERR_INVALID, "dh_row_softmax_bwd: null pointer");
    ROW_LAUNCH(softmax_bwd, "dh_row_softmax_bwd", R, C, (Y, G, GX), log_softmax, accumulate);
}

int dh_layer_norm(const float* X, float* Y, int R, int C) {
    DH_TRY(ensure_init());
    DH_TRY(check_rows("dh_layer_norm", R, C));
    if (R == 0 || C == 0) return DH_OK;
    if (!X || !Y) return set_error(DH_ERR_INVALID, "dh_layer_norm: null pointer");
    ROW_LAUNCH(layer_norm, "dh_layer_norm", R, C, (X, Y));
}

int dh_layer_norm_bwd(const float* X, const float* Y, const float* DY, float* GX, int R, int C,
                      int accumulate) {
    DH_TRY(ensure_init());
    DH_TRY(check_rows("dh_layer_norm_bwd", R, C));
    if (R == 0 || C == 0) return DH_OK;
    if (!X || !Y || !DY || !GX) return set_error(DH_ERR_INVALID, "dh_layer_norm_bwd: null pointer");
    ROW_LAUNCH(layer_norm_bwd, "dh_layer_norm_bwd", R, C, (X, Y, DY, GX), accumulate);
}

int dh_linear_bias_grad(const float* Y, float* dY, float* db, int N, int out, int relu,
                        int accumulate) {
    DH_TRY(ensure_init());
    if (N < 0 || out < 0) return set_error(DH_ERR_INVALID, "dh_linear_bias_grad: negative shape");
    if (out == 0) return DH_OK;
    if (!dY || !db || (relu && !Y))
        return set_error(DH_ERR_INVALID, "dh_linear_bias_grad: null pointer");
    const int cgroups = (out + 63) / 64;
    int P = 1024 / cgroups;                       // enough work-groups to cover the chip
    P = P < 1 ? 1 : P;
    P = P > (N + 63) / 64 ? (N + 63) / 64 : P;    // at least 64 rows per partial
    if (P < 1) P = 1;
    float* part = static_cast<float*>(dh_malloc((size_t)P * out * sizeof(float)));
    if (!part) return set_error(DH_ERR_OOM, "dh_linear_bias_grad: scratch of %d x %d", P, out);
    bias_grad_partial<<<dim3(cgroups, P), 256, 0, stream()>>>(Y, dY, part, N, out, relu);
    int st = check_launch("dh_linear_bias_grad");
    if (st == DH_OK) {
        bias_grad_final<<<cgroups, 1024, 0, stream()>>>(part, db, P, out, accumulate);
        st = check_launch("dh_linear_bias_grad");
    }
    dh_free(part);   // pooled: the buffer returns to its bucket, stream order keeps it safe
    return st;
}

}  // extern "C"
