// hk_softmax.hip — row softmax / log-softmax, forward and backward, for gfx950.
//
// Semantics (reference rust-ascend-compiler/src/ascend/row_programs.rs:135-143 and :152-163,
// driven by rust-ascend-driver/src/tensor/runtime/rows.rs:50-79 and wide_rows.rs:162-232):
//   softmax      m = max_j x_j;  e_j = exp(x_j - m);  s = sum_j e_j;  y_j = e_j / s
//   log_softmax  y_j = (x_j - m) - log(s)
//   backward     softmax:      dot = sum_j y_j dy_j;  dx_j = y_j (dy_j - dot)
//                log_softmax:  dot = sum_j dy_j;      dx_j = dy_j - exp(y_j) dot
// over the last axis of a contiguous FP32 tensor (any positive width; the reference runs
// widths of 32..4096 in multiples of 32 as one row program and tiles the others).
//
// Layout: x/y/dy/dx [rows, W] row-major F32. HBM-bound: the forward moves 8 bytes per element,
// the backward 12.
//
// Fast path (W % 4 == 0, W <= 4096, 16-byte aligned): one wavefront owns one row; lane l holds
// the float4 chunks l, l+64, ... of the row in registers, so the row is read once, and row
// maxima and sums are butterfly reductions across the wave. Wide path (W % 4 == 0,
// 4096 < W <= 32768, aligned; vocabulary-sized rows): one 1024-thread workgroup owns one row,
// thread t holding the float4 chunks t, t+1024, ... in registers, so the row is again read once
// (non-temporal: these working sets exceed the on-package cache), with wave then workgroup
// reductions. General path: one workgroup per row, the row re-read from cache for each pass,
// reductions through LDS.
#include "hk_common.hpp"
#include "hk_kernels.hpp"

#include <initializer_list>
#include <type_traits>

namespace hk {

namespace {

constexpr int kFastThreads = 256;  // 4 rows per workgroup on the fast path
constexpr int kRowThreads = 256;   // one row per workgroup on the general path
constexpr int kWideThreads = 1024; // one row per workgroup on the wide path
constexpr int kWideMaxWidth = kWideThreads * 4 * 8;  // 8 float4 chunks per thread

template <int MAXJ>
__device__ __forceinline__ void load_row4(const float* rowp, int lane, int chunks, f32x4_t (&v)[MAXJ]) {
#pragma unroll
    for (int j = 0; j < MAXJ; ++j) {
        const int c = lane + 64 * j;
        v[j] = c < chunks ? *reinterpret_cast<const f32x4_t*>(rowp + 4 * c) : f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
    }
}

template <int MAXJ, bool LOG>
__global__ void __launch_bounds__(kFastThreads)
softmax_fwd_fast(const float* __restrict__ x, float* __restrict__ y, int64_t rows, int width) {
    const int lane = threadIdx.x & 63;
    for (int64_t row = static_cast<int64_t>(blockIdx.x) * (kFastThreads / 64) + (threadIdx.x >> 6); row < rows;
         row += static_cast<int64_t>(gridDim.x) * (kFastThreads / 64)) {
        const int chunks = width >> 2;
        f32x4_t v[MAXJ];
        load_row4<MAXJ>(x + row * width, lane, chunks, v);
        float m = -INFINITY;
#pragma unroll
        for (int j = 0; j < MAXJ; ++j)
            if (lane + 64 * j < chunks)
#pragma unroll
                for (int e = 0; e < 4; ++e) m = fmaxf(m, v[j][e]);
        m = wave_max(m);
        float s = 0.0f;
#pragma unroll
        for (int j = 0; j < MAXJ; ++j)
            if (lane + 64 * j < chunks)
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const float ex = expf(v[j][e] - m);
                    s += ex;
                    if (!LOG) v[j][e] = ex;
                }
        s = wave_sum(s);
        float* yr = y + row * width;
        if (LOG) {
            const float ls = logf(s);
#pragma unroll
            for (int j = 0; j < MAXJ; ++j) {
                const int c = lane + 64 * j;
                if (c < chunks) {
                    f32x4_t o;
#pragma unroll
                    for (int e = 0; e < 4; ++e) o[e] = (v[j][e] - m) - ls;
                    *reinterpret_cast<f32x4_t*>(yr + 4 * c) = o;
                }
            }
        } else {
            const float inv = 1.0f / s;
#pragma unroll
            for (int j = 0; j < MAXJ; ++j) {
                const int c = lane + 64 * j;
                if (c < chunks) {
                    f32x4_t o;
#pragma unroll
                    for (int e = 0; e < 4; ++e) o[e] = v[j][e] * inv;
                    *reinterpret_cast<f32x4_t*>(yr + 4 * c) = o;
                }
            }
        }
    }
}

template <int MAXJ, bool LOG>
__global__ void __launch_bounds__(kFastThreads)
softmax_bwd_fast(const float* __restrict__ y, const float* __restrict__ dy, float* __restrict__ dx,
                 int64_t rows, int width) {
    const int lane = threadIdx.x & 63;
    for (int64_t row = static_cast<int64_t>(blockIdx.x) * (kFastThreads / 64) + (threadIdx.x >> 6); row < rows;
         row += static_cast<int64_t>(gridDim.x) * (kFastThreads / 64)) {
        const int chunks = width >> 2;
        f32x4_t yv[MAXJ], gv[MAXJ];
        load_row4<MAXJ>(y + row * width, lane, chunks, yv);
        load_row4<MAXJ>(dy + row * width, lane, chunks, gv);
        float dot = 0.0f;
#pragma unroll
        for (int j = 0; j < MAXJ; ++j)
            if (lane + 64 * j < chunks)
#pragma unroll
                for (int e = 0; e < 4; ++e) dot += LOG ? gv[j][e] : yv[j][e] * gv[j][e];
        dot = wave_sum(dot);
        float* dr = dx + row * width;
#pragma unroll
        for (int j = 0; j < MAXJ; ++j) {
            const int c = lane + 64 * j;
            if (c < chunks) {
                f32x4_t o;
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    o[e] = LOG ? gv[j][e] - expf(yv[j][e]) * dot : yv[j][e] * (gv[j][e] - dot);
                *reinterpret_cast<f32x4_t*>(dr + 4 * c) = o;
            }
        }
    }
}

// ---- composed attention: the row passes between its GEMMs
//
// The chain scale, + mask, softmax, cast (and in the backward softmax's gradient, scale, cast) ran as
// one kernel per step over [rows, N] F32 scores; these take a score row from the GEMM to the BF16
// operand of the next one in registers, with the same operations in the same order. HBM-bound: the
// forward moves 4 (scores) + 4 (mask) + 2 bytes per score instead of 26, the backward 4 + 4 + 4 + 4
// instead of 44. At 33280 rows of 1056 scores: forward 193 -> 57 us (6.2 TB/s), backward 330 -> 110
// us (5.1 TB/s; the second operand row in registers leaves half the waves in flight).
//
// The probabilities of a lane's chunks of a row, as scale_mask and softmax_fwd_fast compute them.
template <int MAXJ>
__device__ __forceinline__ void masked_probs(const float* srow, const float* mrow, float scale, int lane, int chunks,
                                             f32x4_t (&v)[MAXJ]) {
    load_row4<MAXJ>(srow, lane, chunks, v);
    f32x4_t k[MAXJ];
    if (mrow) load_row4<MAXJ>(mrow, lane, chunks, k);
    float m = -INFINITY;
#pragma unroll
    for (int j = 0; j < MAXJ; ++j)
        if (lane + 64 * j < chunks)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                v[j][e] = mrow ? v[j][e] * scale + k[j][e] : v[j][e] * scale;
                m = fmaxf(m, v[j][e]);
            }
    m = wave_max(m);
    float s = 0.0f;
#pragma unroll
    for (int j = 0; j < MAXJ; ++j)
        if (lane + 64 * j < chunks)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                v[j][e] = expf(v[j][e] - m);
                s += v[j][e];
            }
    const float inv = 1.0f / wave_sum(s);
#pragma unroll
    for (int j = 0; j < MAXJ; ++j)
#pragma unroll
        for (int e = 0; e < 4; ++e) v[j][e] *= inv;
}

__device__ __forceinline__ void store_bf16x4(uint16_t* p, const f32x4_t& v) {
    *reinterpret_cast<u32x2_t*>(p) = u32x2_t{pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
}

// p = bf16(softmax(s * scale + mask))
template <int MAXJ>
__global__ void __launch_bounds__(kFastThreads)
masked_softmax_rows(const float* __restrict__ s, const float* __restrict__ mask, float scale, uint16_t* __restrict__ p,
                    int64_t rows, int width) {
    const int lane = threadIdx.x & 63, chunks = width >> 2;
    for (int64_t row = static_cast<int64_t>(blockIdx.x) * (kFastThreads / 64) + (threadIdx.x >> 6); row < rows;
         row += static_cast<int64_t>(gridDim.x) * (kFastThreads / 64)) {
        f32x4_t v[MAXJ];
        masked_probs<MAXJ>(s + row * width, mask ? mask + row * width : nullptr, scale, lane, chunks, v);
#pragma unroll
        for (int j = 0; j < MAXJ; ++j)
            if (lane + 64 * j < chunks) store_bf16x4(p + row * width + 4 * (lane + 64 * j), v[j]);
    }
}

// P recomputed as above; ds = P (dP - sum(P dP)); p = bf16(P), dsb = bf16(ds * scale), and, when ds is
// given, ds in F32 (it may be dP's own buffer: a lane stores only what it has read).
template <int MAXJ>
__global__ void __launch_bounds__(kFastThreads)
masked_softmax_bwd_rows(const float* __restrict__ s, const float* __restrict__ mask, const float* dp, float scale,
                        uint16_t* __restrict__ p, uint16_t* __restrict__ dsb, float* ds, int64_t rows, int width) {
    const int lane = threadIdx.x & 63, chunks = width >> 2;
    for (int64_t row = static_cast<int64_t>(blockIdx.x) * (kFastThreads / 64) + (threadIdx.x >> 6); row < rows;
         row += static_cast<int64_t>(gridDim.x) * (kFastThreads / 64)) {
        f32x4_t v[MAXJ], g[MAXJ];
        load_row4<MAXJ>(dp + row * width, lane, chunks, g);
        masked_probs<MAXJ>(s + row * width, mask ? mask + row * width : nullptr, scale, lane, chunks, v);
        float dot = 0.0f;
#pragma unroll
        for (int j = 0; j < MAXJ; ++j)
            if (lane + 64 * j < chunks)
#pragma unroll
                for (int e = 0; e < 4; ++e) dot += v[j][e] * g[j][e];
        dot = wave_sum(dot);
#pragma unroll
        for (int j = 0; j < MAXJ; ++j) {
            const int c = lane + 64 * j;
            if (c < chunks) {
                const int64_t at = row * width + 4 * c;
                store_bf16x4(p + at, v[j]);
                f32x4_t d;
#pragma unroll
                for (int e = 0; e < 4; ++e) d[e] = v[j][e] * (g[j][e] - dot);
                if (ds) *reinterpret_cast<f32x4_t*>(ds + at) = d;
#pragma unroll
                for (int e = 0; e < 4; ++e) d[e] *= scale;
                store_bf16x4(dsb + at, d);
            }
        }
    }
}

// Workgroup-wide reduction through LDS (wave results combined in wave order).
template <bool MAX, int NT = kRowThreads>
__device__ __forceinline__ float block_reduce(float v, float* scratch) {
    v = MAX ? wave_max(v) : wave_sum(v);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    if (lane == 0) scratch[wave] = v;
    __syncthreads();
    float r = scratch[0];
#pragma unroll
    for (int i = 1; i < NT / 64; ++i) r = MAX ? fmaxf(r, scratch[i]) : r + scratch[i];
    __syncthreads();  // scratch is reused by the next reduction
    return r;
}

// chunks past the row's end read as `pad`
template <int MAXJ>
__device__ __forceinline__ void load_row_wide(const float* rowp, int chunks, f32x4_t (&v)[MAXJ], float pad = 0.0f) {
#pragma unroll
    for (int j = 0; j < MAXJ; ++j) {
        const int c = threadIdx.x + kWideThreads * j;
        v[j] = c < chunks ? stream_load(reinterpret_cast<const f32x4_t*>(rowp) + c) : f32x4_t{pad, pad, pad, pad};
    }
}

// At most 64 VGPRs (8 waves per SIMD), so two rows' workgroups share a CU and one streams
// while the other waits in its reductions.
template <int MAXJ, bool LOG>
__global__ void __launch_bounds__(kWideThreads) __attribute__((amdgpu_waves_per_eu(8)))
softmax_fwd_wide(const float* __restrict__ x, float* __restrict__ y, int64_t rows, int width) {
    __shared__ float scratch[kWideThreads / 64];
    for (int64_t row = blockIdx.x; row < rows; row += gridDim.x) {  // uniform per workgroup
        const int chunks = width >> 2;
        // chunks past the end hold -inf: they leave the maximum alone and add exp(-inf) = 0
        f32x4_t v[MAXJ];
        load_row_wide<MAXJ>(x + row * width, chunks, v, -INFINITY);
        float m = -INFINITY;
#pragma unroll
        for (int j = 0; j < MAXJ; ++j)
#pragma unroll
            for (int e = 0; e < 4; ++e) m = fmaxf(m, v[j][e]);
        m = block_reduce<true, kWideThreads>(m, scratch);
        float s = 0.0f;
#pragma unroll
        for (int j = 0; j < MAXJ; ++j)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const float ex = expf(v[j][e] - m);
                s += ex;
                if (!LOG) v[j][e] = ex;
            }
        s = block_reduce<false, kWideThreads>(s, scratch);
        f32x4_t* yr = reinterpret_cast<f32x4_t*>(y + row * width);
        const float ls = LOG ? logf(s) : 0.0f, inv = LOG ? 0.0f : 1.0f / s;
#pragma unroll
        for (int j = 0; j < MAXJ; ++j) {
            const int c = threadIdx.x + kWideThreads * j;
            if (c < chunks) {
                f32x4_t o;
#pragma unroll
                for (int e = 0; e < 4; ++e) o[e] = LOG ? (v[j][e] - m) - ls : v[j][e] * inv;
                stream_store(o, yr + c);
            }
        }
    }
}

template <int MAXJ, bool LOG>
__global__ void __launch_bounds__(kWideThreads)
softmax_bwd_wide(const float* __restrict__ y, const float* __restrict__ dy, float* __restrict__ dx, int64_t rows, int width) {
    __shared__ float scratch[kWideThreads / 64];
    for (int64_t row = blockIdx.x; row < rows; row += gridDim.x) {  // uniform per workgroup
        const int chunks = width >> 2;
        f32x4_t yv[MAXJ], gv[MAXJ];
        load_row_wide<MAXJ>(y + row * width, chunks, yv);
        load_row_wide<MAXJ>(dy + row * width, chunks, gv);
        float dot = 0.0f;
#pragma unroll
        for (int j = 0; j < MAXJ; ++j)
            if (static_cast<int>(threadIdx.x) + kWideThreads * j < chunks)
#pragma unroll
                for (int e = 0; e < 4; ++e) dot += LOG ? gv[j][e] : yv[j][e] * gv[j][e];
        dot = block_reduce<false, kWideThreads>(dot, scratch);
        f32x4_t* dr = reinterpret_cast<f32x4_t*>(dx + row * width);
#pragma unroll
        for (int j = 0; j < MAXJ; ++j) {
            const int c = threadIdx.x + kWideThreads * j;
            if (c < chunks) {
                f32x4_t o;
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    o[e] = LOG ? gv[j][e] - expf(yv[j][e]) * dot : yv[j][e] * (gv[j][e] - dot);
                stream_store(o, dr + c);
            }
        }
    }
}

// ---- log-softmax with the NLL row term (cross entropy), and any width's log-softmax
//
// A row of any width and alignment in registers: thread t holds the 16-byte chunks t, t + NT, ... of
// the row's aligned middle, and threads 0 .. 5 one each of the at most three values before and after
// it. (x and y are 16-byte aligned, so a row's split is the same in both.) HBM-bound: 8 bytes per
// value in one pass; rows off 16 bytes used to take three scalar passes of softmax_fwd_general.
struct CeRows {
    const void* target;  // labels, null for a plain log-softmax
    int id_bytes;
    const float* weight;  // class weights, null for one
    int64_t ignore;
    float* row_v;  // -weight[t] * y[t] and weight[t] per row (0 for an ignored or out-of-range label)
    float* row_w;
    float* out;  // reduction None: the row terms again (the loss), else null
};

// Up to 8 chunks per thread within 64 VGPRs (8 waves per SIMD: two rows' workgroups share a CU): [4096,
// 32000] 216 -> 183 us.
template <int NT, int MAXJ, bool STREAM>
__global__ void __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(MAXJ <= 8 ? 8 : 4)))
log_softmax_rows(const float* __restrict__ x, float* __restrict__ y, int64_t rows, int width, CeRows ce) {
    __shared__ float scratch[NT / 64];
    const int t = threadIdx.x;
    for (int64_t row = blockIdx.x; row < rows; row += gridDim.x) {  // uniform per workgroup
        const int64_t base = row * width;
        const float* xr = x + base;
        float* yr = y + base;
        const int head = min(static_cast<int>((4 - (base & 3)) & 3), width);
        const int chunks = (width - head) >> 2, tail = (width - head) & 3;
        const f32x4_t* x4 = reinterpret_cast<const f32x4_t*>(xr + head);
        // chunks past the end hold -inf: they leave the maximum alone and add exp(-inf) = 0
        f32x4_t v[MAXJ];
#pragma unroll
        for (int j = 0; j < MAXJ; ++j) {
            const int c = t + NT * j;
            if (c < chunks) v[j] = STREAM ? stream_load(x4 + c) : x4[c];
            else v[j] = f32x4_t{-INFINITY, -INFINITY, -INFINITY, -INFINITY};
        }
        const int edge = t < head ? t : width - tail + (t - head);
        const bool has_edge = t < head + tail;
        const float ve = has_edge ? xr[edge] : -INFINITY;
        int64_t label = -1;
        float xt = 0.0f, wt = 0.0f;
        bool counted = false;
        if (ce.target && t == 0) {
            label = ce.id_bytes == 8 ? static_cast<const int64_t*>(ce.target)[row] : static_cast<const int32_t*>(ce.target)[row];
            counted = label != ce.ignore && label >= 0 && label < width;
            if (counted) xt = xr[label], wt = ce.weight ? ce.weight[label] : 1.0f;
        }
        float m = ve;
#pragma unroll
        for (int j = 0; j < MAXJ; ++j)
#pragma unroll
            for (int e = 0; e < 4; ++e) m = fmaxf(m, v[j][e]);
        m = block_reduce<true, NT>(m, scratch);
        float s = expf(ve - m);
#pragma unroll
        for (int j = 0; j < MAXJ; ++j)
#pragma unroll
            for (int e = 0; e < 4; ++e) s += expf(v[j][e] - m);
        s = block_reduce<false, NT>(s, scratch);
        const float ls = logf(s);
        f32x4_t* y4 = reinterpret_cast<f32x4_t*>(yr + head);
#pragma unroll
        for (int j = 0; j < MAXJ; ++j) {
            const int c = t + NT * j;
            if (c < chunks) {
                f32x4_t o;
#pragma unroll
                for (int e = 0; e < 4; ++e) o[e] = (v[j][e] - m) - ls;
                if (STREAM) stream_store(o, y4 + c);
                else y4[c] = o;
            }
        }
        if (has_edge) yr[edge] = (ve - m) - ls;
        if (ce.target && t == 0) {
            const float term = counted ? -(wt * ((xt - m) - ls)) : 0.0f;
            ce.row_v[row] = term;
            ce.row_w[row] = counted ? wt : 0.0f;
            if (ce.out) ce.out[row] = term;
        }
    }
}

// Cross entropy's gradient: dx = d [c == label] - exp(y) d with d = -(weight[label] * g) (0 for an ignored
// or out-of-range label): what nll_backward's dense gradient followed by softmax_bwd (LOG) computes,
// whose row sum has the one term d. 8 bytes per value instead of 20.
struct CeRow {
    float d;
    int64_t label;
};
__device__ __forceinline__ CeRow ce_row(const CeRows& ce, const float* grad, const float* total, int reduction, int64_t r,
                                        int64_t classes) {
    const int64_t label = ce.id_bytes == 8 ? static_cast<const int64_t*>(ce.target)[r] : static_cast<const int32_t*>(ce.target)[r];
    CeRow out = {0.0f, label};
    if (label != ce.ignore && label >= 0 && label < classes) {
        float g = grad[reduction == 0 ? r : 0];
        if (reduction == 1) g = g / total[0];
        out.d = -((ce.weight ? ce.weight[label] : 1.0f) * g);
    }
    return out;
}
__device__ __forceinline__ float ce_grad(float y, const CeRow& r, int64_t c) {
    return (c == r.label ? r.d : 0.0f) - expf(y) * r.d;
}

// Rows of at least 2048 values: a workgroup takes a segment of one row, so the label, weight and upstream
// gradient are uniform, and a thread has 8 loads in flight: [4096, 32000] 188 us (5.6 TB/s) against 205 by
// the flat kernel and 453 by the two kernels.
constexpr int kCeSegChunks = 256 * 8;
template <bool STREAM>
__global__ void __launch_bounds__(256)
cross_entropy_bwd_rows(const float* __restrict__ grad, const float* __restrict__ y, const float* __restrict__ total,
                       float* __restrict__ dx, int64_t segments, int segs_per_row, int width, int reduction, CeRows ce) {
    const int t = threadIdx.x;
    for (int64_t unit = blockIdx.x; unit < segments; unit += gridDim.x) {
        const int64_t r = unit / segs_per_row;
        const int seg = static_cast<int>(unit - r * segs_per_row);
        const int64_t base = r * width;
        const int head = static_cast<int>((4 - (base & 3)) & 3);
        const int chunks = (width - head) >> 2, tail = (width - head) & 3;
        const f32x4_t* y4 = reinterpret_cast<const f32x4_t*>(y + base + head);
        f32x4_t* d4 = reinterpret_cast<f32x4_t*>(dx + base + head);
        const int c0 = seg * kCeSegChunks + t;
        f32x4_t v[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const int c = min(c0 + 256 * j, chunks - 1);
            v[j] = STREAM ? stream_load(y4 + c) : y4[c];
        }
        const CeRow row = ce_row(ce, grad, total, reduction, r, width);
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const int c = c0 + 256 * j;
            if (c < chunks) {
                f32x4_t o;
#pragma unroll
                for (int e = 0; e < 4; ++e) o[e] = ce_grad(v[j][e], row, head + 4 * c + e);
                if (STREAM) stream_store(o, d4 + c);
                else d4[c] = o;
            }
        }
        if (seg == 0 && t < head + tail) {
            const int c = t < head ? t : width - tail + (t - head);
            dx[base + c] = ce_grad(y[base + c], row, c);
        }
    }
}

// Any width: flat over the values, a label per 16-byte chunk and row it touches. vec: y and dx are
// 16-byte aligned (otherwise every value takes the element loop).
template <bool STREAM, bool WIDE_INDEX>
__global__ void __launch_bounds__(256)
cross_entropy_bwd_kernel(const float* __restrict__ grad, const float* __restrict__ y, const float* __restrict__ total,
                         float* __restrict__ dx, int64_t rows, int64_t classes, int reduction, bool vec, CeRows ce) {
    const int64_t count = rows * classes, chunks = vec ? count >> 2 : 0;
    auto row_of = [&](int64_t r) __attribute__((always_inline)) { return ce_row(ce, grad, total, reduction, r, classes); };
    for (int64_t i = flat_begin(256); i < chunks; i += flat_stride(256)) {
        const f32x4_t v = STREAM ? stream_load(reinterpret_cast<const f32x4_t*>(y) + i) : reinterpret_cast<const f32x4_t*>(y)[i];
        int64_t r, c;
        if constexpr (WIDE_INDEX) {
            r = 4 * i / classes, c = 4 * i - r * classes;
        } else {  // count < 2^32
            const uint32_t i4 = static_cast<uint32_t>(4 * i), k = static_cast<uint32_t>(classes);
            r = i4 / k, c = i4 - static_cast<uint32_t>(r) * k;
        }
        CeRow row = row_of(r);
        f32x4_t o;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            if (c == classes) row = row_of(++r), c = 0;  // the chunk crosses into the next row
            o[e] = ce_grad(v[e], row, c);
            ++c;
        }
        if (STREAM) stream_store(o, reinterpret_cast<f32x4_t*>(dx) + i);
        else reinterpret_cast<f32x4_t*>(dx)[i] = o;
    }
    for (int64_t i = 4 * chunks + flat_begin(256); i < count; i += flat_stride(256))
        dx[i] = ce_grad(y[i], row_of(i / classes), i % classes);
}

template <bool LOG>
__global__ void __launch_bounds__(kRowThreads)
softmax_fwd_general(const float* __restrict__ x, float* __restrict__ y, int64_t rows, int64_t width) {
    __shared__ float scratch[kRowThreads / 64];
    for (int64_t row = blockIdx.x; row < rows; row += gridDim.x) {  // uniform per workgroup
        const float* xr = x + row * width;
        float* yr = y + row * width;
        float m = -INFINITY;
        for (int64_t c = threadIdx.x; c < width; c += kRowThreads) m = fmaxf(m, xr[c]);
        m = block_reduce<true>(m, scratch);
        float s = 0.0f;
        for (int64_t c = threadIdx.x; c < width; c += kRowThreads) s += expf(xr[c] - m);
        s = block_reduce<false>(s, scratch);
        if (LOG) {
            const float ls = logf(s);
            for (int64_t c = threadIdx.x; c < width; c += kRowThreads) yr[c] = (xr[c] - m) - ls;
        } else {
            const float inv = 1.0f / s;
            for (int64_t c = threadIdx.x; c < width; c += kRowThreads) yr[c] = expf(xr[c] - m) * inv;
        }
    }
}

template <bool LOG>
__global__ void __launch_bounds__(kRowThreads)
softmax_bwd_general(const float* __restrict__ y, const float* __restrict__ dy, float* __restrict__ dx,
                    int64_t rows, int64_t width) {
    __shared__ float scratch[kRowThreads / 64];
    for (int64_t row = blockIdx.x; row < rows; row += gridDim.x) {  // uniform per workgroup
        const float* yr = y + row * width;
        const float* gr = dy + row * width;
        float* dr = dx + row * width;
        float dot = 0.0f;
        for (int64_t c = threadIdx.x; c < width; c += kRowThreads) dot += LOG ? gr[c] : yr[c] * gr[c];
        dot = block_reduce<false>(dot, scratch);
        for (int64_t c = threadIdx.x; c < width; c += kRowThreads)
            dr[c] = LOG ? gr[c] - expf(yr[c]) * dot : yr[c] * (gr[c] - dot);
    }
}

bool fast_softmax(int64_t width, std::initializer_list<const void*> ptrs) {
    return width % 4 == 0 && width <= 4096 && aligned16(ptrs);
}

bool wide_softmax(int64_t width, std::initializer_list<const void*> ptrs) {
    return width % 4 == 0 && width > 4096 && width <= kWideMaxWidth && aligned16(ptrs);
}

// float4 chunks per thread of the wide path: 2, 4 or 8
int wide_per_thread(int64_t width) {
    const int64_t per = (width / 4 + kWideThreads - 1) / kWideThreads;
    return per <= 2 ? 2 : (per <= 4 ? 4 : 8);
}

constexpr int64_t kRowsMaxWidth = 1024 * 4 * 16;  // log_softmax_rows: 16 chunks per thread

// log_softmax_rows takes rows of up to 65536 values (16-byte aligned tensors); 256 threads up to 4096. Below 257
// values a row gives its workgroup less than a chunk a thread, and the passes that it replaced are faster: log-softmax
// of 34 M values, us, general against rows: width 3 5800 8800, 50 380 580, 130 187 227, 255 107 119, 257 132 119, 399 101 82.
bool log_rows_applies(int64_t width, const float* x, const float* y) { return width <= kRowsMaxWidth && aligned16({x, y}); }

void launch_log_rows(const float* x, float* y, int64_t rows, int64_t width, const CeRows& ce, hipStream_t s) {
    const dim3 grid(flat_blocks(rows, 1));
    const int w = static_cast<int>(width);
    const bool stream = rows * width * 8 > (int64_t{1} << 28);  // x and y past the on-package cache
    auto go = [&](auto nt, auto maxj) {
        constexpr int NT = decltype(nt)::value, MAXJ = decltype(maxj)::value;
        if (stream) hipLaunchKernelGGL((log_softmax_rows<NT, MAXJ, true>), grid, dim3(NT), 0, s, x, y, rows, w, ce);
        else hipLaunchKernelGGL((log_softmax_rows<NT, MAXJ, false>), grid, dim3(NT), 0, s, x, y, rows, w, ce);
    };
    if (width <= 1024) go(std::integral_constant<int, 256>{}, std::integral_constant<int, 1>{});
    else if (width <= 4096) go(std::integral_constant<int, 256>{}, std::integral_constant<int, 4>{});
    else if (width <= 8192) go(std::integral_constant<int, 1024>{}, std::integral_constant<int, 2>{});
    else if (width <= 16384) go(std::integral_constant<int, 1024>{}, std::integral_constant<int, 4>{});
    else if (width <= 32768) go(std::integral_constant<int, 1024>{}, std::integral_constant<int, 8>{});
    else go(std::integral_constant<int, 1024>{}, std::integral_constant<int, 16>{});
}

template <bool LOG>
void launch_fwd(const float* x, float* y, int64_t rows, int64_t width, hipStream_t s) {
    if (fast_softmax(width, {x, y})) {
        const dim3 grid(flat_blocks(rows, 4));
        const int per_lane = static_cast<int>((width / 4 + 63) / 64);
        const int w = static_cast<int>(width);
        if (per_lane <= 1) hipLaunchKernelGGL((softmax_fwd_fast<1, LOG>), grid, dim3(kFastThreads), 0, s, x, y, rows, w);
        else if (per_lane <= 2) hipLaunchKernelGGL((softmax_fwd_fast<2, LOG>), grid, dim3(kFastThreads), 0, s, x, y, rows, w);
        else if (per_lane <= 4) hipLaunchKernelGGL((softmax_fwd_fast<4, LOG>), grid, dim3(kFastThreads), 0, s, x, y, rows, w);
        else if (per_lane <= 8) hipLaunchKernelGGL((softmax_fwd_fast<8, LOG>), grid, dim3(kFastThreads), 0, s, x, y, rows, w);
        else hipLaunchKernelGGL((softmax_fwd_fast<16, LOG>), grid, dim3(kFastThreads), 0, s, x, y, rows, w);
    } else if (wide_softmax(width, {x, y})) {
        const dim3 grid(flat_blocks(rows, 1));
        const int w = static_cast<int>(width);
        switch (wide_per_thread(width)) {
            case 2: hipLaunchKernelGGL((softmax_fwd_wide<2, LOG>), grid, dim3(kWideThreads), 0, s, x, y, rows, w); break;
            case 4: hipLaunchKernelGGL((softmax_fwd_wide<4, LOG>), grid, dim3(kWideThreads), 0, s, x, y, rows, w); break;
            default: hipLaunchKernelGGL((softmax_fwd_wide<8, LOG>), grid, dim3(kWideThreads), 0, s, x, y, rows, w); break;
        }
    } else if (LOG && width > 256 && log_rows_applies(width, x, y)) {
        launch_log_rows(x, y, rows, width, CeRows{}, s);
    } else {
        hipLaunchKernelGGL((softmax_fwd_general<LOG>), dim3(flat_blocks(rows, 1)), dim3(kRowThreads), 0, s, x, y,
                           rows, width);
    }
}

template <bool LOG>
void launch_bwd(const float* y, const float* dy, float* dx, int64_t rows, int64_t width, hipStream_t s) {
    if (fast_softmax(width, {y, dy, dx})) {
        const dim3 grid(flat_blocks(rows, 4));
        const int per_lane = static_cast<int>((width / 4 + 63) / 64);
        const int w = static_cast<int>(width);
        if (per_lane <= 1) hipLaunchKernelGGL((softmax_bwd_fast<1, LOG>), grid, dim3(kFastThreads), 0, s, y, dy, dx, rows, w);
        else if (per_lane <= 2) hipLaunchKernelGGL((softmax_bwd_fast<2, LOG>), grid, dim3(kFastThreads), 0, s, y, dy, dx, rows, w);
        else if (per_lane <= 4) hipLaunchKernelGGL((softmax_bwd_fast<4, LOG>), grid, dim3(kFastThreads), 0, s, y, dy, dx, rows, w);
        else if (per_lane <= 8) hipLaunchKernelGGL((softmax_bwd_fast<8, LOG>), grid, dim3(kFastThreads), 0, s, y, dy, dx, rows, w);
        else hipLaunchKernelGGL((softmax_bwd_fast<16, LOG>), grid, dim3(kFastThreads), 0, s, y, dy, dx, rows, w);
    } else if (wide_softmax(width, {y, dy, dx})) {
        const dim3 grid(flat_blocks(rows, 1));
        const int w = static_cast<int>(width);
        switch (wide_per_thread(width)) {
            case 2: hipLaunchKernelGGL((softmax_bwd_wide<2, LOG>), grid, dim3(kWideThreads), 0, s, y, dy, dx, rows, w); break;
            case 4: hipLaunchKernelGGL((softmax_bwd_wide<4, LOG>), grid, dim3(kWideThreads), 0, s, y, dy, dx, rows, w); break;
            default: hipLaunchKernelGGL((softmax_bwd_wide<8, LOG>), grid, dim3(kWideThreads), 0, s, y, dy, dx, rows, w); break;
        }
    } else {
        hipLaunchKernelGGL((softmax_bwd_general<LOG>), dim3(flat_blocks(rows, 1)), dim3(kRowThreads), 0, s, y, dy,
                           dx, rows, width);
    }
}

// f(integral_constant<MAXJ>) for the float4 chunks per lane of a row of at most 4096 values
template <class F>
void by_chunks(int64_t width, F&& f) {
    const int per_lane = static_cast<int>((width / 4 + 63) / 64);
    if (per_lane <= 1) f(std::integral_constant<int, 1>{});
    else if (per_lane <= 2) f(std::integral_constant<int, 2>{});
    else if (per_lane <= 4) f(std::integral_constant<int, 4>{});
    else if (per_lane <= 6) f(std::integral_constant<int, 6>{});
    else if (per_lane <= 8) f(std::integral_constant<int, 8>{});
    else f(std::integral_constant<int, 16>{});
}

}  // namespace

bool masked_softmax_applies(int64_t width, const float* mask, const float* ds) { return fast_softmax(width, {mask, ds}); }

hipError_t masked_softmax(const float* scores, const float* mask, float scale, void* p, int64_t rows, int64_t width,
                          hipStream_t s) {
    if (rows == 0) return hipSuccess;
    by_chunks(width, [&](auto j) {
        hipLaunchKernelGGL((masked_softmax_rows<decltype(j)::value>), dim3(flat_blocks(rows, 4)), dim3(kFastThreads), 0, s,
                           scores, mask, scale, static_cast<uint16_t*>(p), rows, static_cast<int>(width));
    });
    return hipGetLastError();
}

hipError_t masked_softmax_backward(const float* scores, const float* mask, const float* dp, float scale, void* p, void* dsb,
                                   float* ds, int64_t rows, int64_t width, hipStream_t s) {
    if (rows == 0) return hipSuccess;
    by_chunks(width, [&](auto j) {
        hipLaunchKernelGGL((masked_softmax_bwd_rows<decltype(j)::value>), dim3(flat_blocks(rows, 4)), dim3(kFastThreads), 0,
                           s, scores, mask, dp, scale, static_cast<uint16_t*>(p), static_cast<uint16_t*>(dsb), ds, rows,
                           static_cast<int>(width));
    });
    return hipGetLastError();
}

hipError_t softmax_forward(const float* x, float* y, int64_t rows, int64_t width, int logarithmic, hipStream_t s) {
    if (rows == 0) return hipSuccess;
    if (logarithmic) launch_fwd<true>(x, y, rows, width, s);
    else launch_fwd<false>(x, y, rows, width, s);
    return hipGetLastError();
}

// The NLL term joins the row pass where that pass is the faster log-softmax. Rows of a multiple of 4 have the
// wave-a-row kernel to beat, which is ahead up to 768 values: cross entropy forward of 34 M logits, us, two passes
// against one: width 32 846 1627, 128 226 411, 256 132 212, 512 90 115, 768 79 85, 1000 75 72; 17 2530 3100,
// 201 254 268, 255 208 213, 257 252 212.
bool log_softmax_nll_applies(int64_t width, const float* x, const float* y) {
    return width > (width % 4 == 0 ? 768 : 256) && log_rows_applies(width, x, y);
}

hipError_t log_softmax_nll(const float* x, float* y, int64_t rows, int64_t width, const void* target, int id_bytes,
                           const float* weight, int64_t ignore, float* row_v, float* row_w, float* out, hipStream_t s) {
    if (rows == 0) return hipSuccess;
    launch_log_rows(x, y, rows, width, CeRows{target, id_bytes, weight, ignore, row_v, row_w, out}, s);
    return hipGetLastError();
}

hipError_t cross_entropy_backward(const float* grad, const float* y, const void* target, int id_bytes, const float* weight,
                                  const float* total, float* dx, int64_t rows, int64_t classes, int reduction,
                                  int64_t ignore, hipStream_t s) {
    const int64_t count = rows * classes;
    if (count == 0) return hipSuccess;
    const CeRows ce{target, id_bytes, weight, ignore, nullptr, nullptr, nullptr};
    const bool vec = aligned16({y, dx});
    const bool stream = count * 8 > (int64_t{1} << 28);
    if (vec && classes >= 2048 && classes <= INT32_MAX - 4 * kCeSegChunks) {
        const int segs = static_cast<int>((classes / 4 + kCeSegChunks - 1) / kCeSegChunks), w = static_cast<int>(classes);
        const dim3 rows_grid(flat_blocks(rows * segs, 1));
        if (stream)
            hipLaunchKernelGGL((cross_entropy_bwd_rows<true>), rows_grid, dim3(256), 0, s, grad, y, total, dx, rows * segs, segs, w, reduction, ce);
        else
            hipLaunchKernelGGL((cross_entropy_bwd_rows<false>), rows_grid, dim3(256), 0, s, grad, y, total, dx, rows * segs, segs, w, reduction, ce);
        return hipGetLastError();
    }
    const dim3 grid(flat_blocks((count + 3) / 4, 256));
    if (count >= (int64_t{1} << 32))
        hipLaunchKernelGGL((cross_entropy_bwd_kernel<true, true>), grid, dim3(256), 0, s, grad, y, total, dx, rows, classes, reduction, vec, ce);
    else if (stream)
        hipLaunchKernelGGL((cross_entropy_bwd_kernel<true, false>), grid, dim3(256), 0, s, grad, y, total, dx, rows, classes, reduction, vec, ce);
    else
        hipLaunchKernelGGL((cross_entropy_bwd_kernel<false, false>), grid, dim3(256), 0, s, grad, y, total, dx, rows, classes, reduction, vec, ce);
    return hipGetLastError();
}

hipError_t softmax_backward(const float* y, const float* dy, float* dx, int64_t rows, int64_t width, int logarithmic,
                            hipStream_t s) {
    if (rows == 0) return hipSuccess;
    if (logarithmic) launch_bwd<true>(y, dy, dx, rows, width, s);
    else launch_bwd<false>(y, dy, dx, rows, width, s);
    return hipGetLastError();
}

}  // namespace hk
