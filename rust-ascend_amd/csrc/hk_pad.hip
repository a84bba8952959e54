// hk_pad.hip — zero padding and cropping of matrix tails for the padded BF16-compute GEMM.
//
// Reference (paths relative to the shuqi2077/rust-ascend root): runtime/padded_matrix.rs:6-43
// pads each matrix axis of a rank-2/3 tensor up to a multiple of 16 with zeros ("prefix
// resize", positive end padding), rounding F32 to BF16 first (conversion::cast, RNE), runs the
// native GEMM on the padded operands with F32 output, and crops the F32 result back to its
// logical shape (negative end padding: retained values are copied bit for bit).
//
// Layout: [batch, rows, cols] row-major on both sides. pad_bf16 writes the whole padded
// [batch, R, C] destination (zeros outside the source), so no separate clearing pass is needed;
// crop_f32 reads only the retained [batch, rows, cols] window. Both are HBM-bound. Rows of at least
// 512 (pad) or 256 (crop) columns with 16-byte aligned destinations go through the row kernels
// (a workgroup per row at a time, 16-byte chunks per thread); the rest through element kernels (one
// work item per destination element pair or element in a grid-stride walk).
#include "hk_common.hpp"
#include "hk_kernels.hpp"

namespace hk {

namespace {

constexpr int kPadThreads = 256;

// dst[b, r, c] = bf16(src[b, r, c]) inside the source, 0 outside; two BF16 per thread.
template <typename T>
__global__ void __launch_bounds__(kPadThreads)
pad_bf16_kernel(const T* __restrict__ src, uint16_t* __restrict__ dst, int64_t rows, int64_t cols, int64_t R,
                int64_t C, int64_t total_pairs) {
    for (int64_t pair = flat_begin(kPadThreads); pair < total_pairs; pair += flat_stride(kPadThreads)) {
        const int64_t i = 2 * pair;  // C is even (a multiple of 16), so a pair never crosses a row
        const int64_t c = i % C, rb = i / C;
        const int64_t r = rb % R, b = rb / R;
        uint16_t v[2];
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            const int64_t cc = c + e;
            if (r < rows && cc < cols) {
                const int64_t s = (b * rows + r) * cols + cc;
                if constexpr (sizeof(T) == 4) v[e] = f32_to_bf16(src[s]);
                else v[e] = src[s];
            } else {
                v[e] = 0;
            }
        }
        *reinterpret_cast<uint32_t*>(dst + i) = static_cast<uint32_t>(v[0]) | (static_cast<uint32_t>(v[1]) << 16);
    }
}

// dst[b, r, c] = src[b, r, c] for the retained window of a [batch, R, C] F32 source.
__global__ void __launch_bounds__(kPadThreads)
crop_f32_kernel(const float* __restrict__ src, float* __restrict__ dst, int64_t rows, int64_t cols, int64_t R,
                int64_t C, int64_t total) {
    for (int64_t i = flat_begin(kPadThreads); i < total; i += flat_stride(kPadThreads)) {
        const int64_t c = i % cols, rb = i / cols;
        const int64_t r = rb % rows, b = rb / rows;
        dst[i] = src[(b * R + r) * C + c];
    }
}

// pad_bf16_kernel's result, row by row, of up to two matrices in one launch: destination row rb of [batch,
// R, C] (its batch and row from one division per row), thread j its 8 columns 8j .. 8j+7 as one
// 16-byte store. Where all 8 exist in the source, F32 loads them as two vectors of any 4-byte
// alignment (rows of odd length: with eight strided loads a thread, 1777 x 2001, 3003 x 2001 and 1777 x
// 3003 took 47 us in three launches, so 19 in two; 90 MB) and BF16 as one where vec says that its rows are 16-byte aligned; else per element, zero outside the
// source. BF16 is copied bit for bit, F32 rounded as pad_bf16_kernel rounds it.
typedef float f32x4_any_t __attribute__((ext_vector_type(4), aligned(4)));
struct PadRows {
    const void* src;
    uint16_t* dst;
    int64_t rows, cols, R, C, nrows;
    int vec;
};

template <typename T>
__device__ __forceinline__ void pad_row(const PadRows& p, int64_t rb) {
    const int64_t b = rb / p.R, r = rb - b * p.R;
    const T* srow = static_cast<const T*>(p.src) + (b * p.rows + r) * p.cols;  // read only for r < rows
    uint16_t* drow = p.dst + rb * p.C;
    for (int64_t j = threadIdx.x; j < p.C / 8; j += kPadThreads) {  // C is a multiple of 16
        const int64_t c0 = 8 * j;
        u32x4_t w;
        if ((sizeof(T) == 4 || p.vec) && r < p.rows && c0 + 8 <= p.cols) {
            if constexpr (sizeof(T) == 2) {
                w = *reinterpret_cast<const u32x4_t*>(srow + c0);
            } else {
                const f32x4_any_t u = *reinterpret_cast<const f32x4_any_t*>(srow + c0);
                const f32x4_any_t v = *reinterpret_cast<const f32x4_any_t*>(srow + c0 + 4);
                w = u32x4_t{pack_bf16x2(u[0], u[1]), pack_bf16x2(u[2], u[3]), pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
            }
        } else {
            uint16_t h[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                h[e] = 0;
                if (r < p.rows && c0 + e < p.cols) {
                    if constexpr (sizeof(T) == 4) h[e] = f32_to_bf16(srow[c0 + e]);
                    else h[e] = srow[c0 + e];
                }
            }
#pragma unroll
            for (int i = 0; i < 4; ++i) w[i] = static_cast<uint32_t>(h[2 * i]) | (static_cast<uint32_t>(h[2 * i + 1]) << 16);
        }
        *reinterpret_cast<u32x4_t*>(drow + c0) = w;
    }
}

template <typename T>
__global__ void __launch_bounds__(kPadThreads)
pad_rows_kernel(PadRows p, PadRows q) {
    for (int64_t rb = blockIdx.x; rb < p.nrows + q.nrows; rb += gridDim.x) {
        if (rb < p.nrows) pad_row<T>(p, rb);
        else pad_row<T>(q, rb - p.nrows);
    }
}

// crop_f32_kernel's result, row by row: destination row rb of [batch, rows, cols] copied from its
// source row of [batch, R, C] as 16-byte chunks (vec: cols % 4 == 0 and both bases 16-byte
// aligned), else per element.
__global__ void __launch_bounds__(kPadThreads)
crop_rows_kernel(const float* __restrict__ src, float* __restrict__ dst, int64_t rows, int64_t cols, int64_t R,
                 int64_t C, int64_t nrows, int vec) {
    for (int64_t rb = blockIdx.x; rb < nrows; rb += gridDim.x) {
        const int64_t b = rb / rows, r = rb - b * rows;
        const float* srow = src + (b * R + r) * C;
        float* drow = dst + rb * cols;
        if (vec) {
            for (int64_t j = threadIdx.x; j < cols / 4; j += kPadThreads)
                *reinterpret_cast<f32x4_t*>(drow + 4 * j) = *reinterpret_cast<const f32x4_t*>(srow + 4 * j);
        } else {
            for (int64_t c = threadIdx.x; c < cols; c += kPadThreads) drow[c] = srow[c];
        }
    }
}

unsigned blocks_for(int64_t work) { return flat_blocks(work, kPadThreads); }
bool aligned16(const void* p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; }

template <typename T>
void launch_pad_rows(const PadRows& p, const PadRows& q, hipStream_t s) {
    const int64_t nrows = p.nrows + q.nrows;
    hipLaunchKernelGGL(pad_rows_kernel<T>, dim3(static_cast<unsigned>(nrows < kMaxFlatBlocks ? nrows : kMaxFlatBlocks)),
                       dim3(kPadThreads), 0, s, p, q);
}

}  // namespace

hipError_t pad_bf16(int src_bf16, const void* src, void* dst, int64_t batch, int64_t rows, int64_t cols, int64_t R,
                    int64_t C, hipStream_t s) {
    const int64_t pairs = batch * R * C / 2;
    if (pairs == 0) return hipSuccess;
    if (C >= 512 && aligned16(dst)) {
        const PadRows p{src, static_cast<uint16_t*>(dst), rows, cols, R, C, batch * R, aligned16(src) && cols % 8 == 0};
        if (src_bf16) launch_pad_rows<uint16_t>(p, PadRows{}, s);
        else launch_pad_rows<float>(p, PadRows{}, s);
        return hipGetLastError();
    }
    if (src_bf16)
        hipLaunchKernelGGL(pad_bf16_kernel<uint16_t>, dim3(blocks_for(pairs)), dim3(kPadThreads), 0, s,
                           static_cast<const uint16_t*>(src), static_cast<uint16_t*>(dst), rows, cols, R, C, pairs);
    else
        hipLaunchKernelGGL(pad_bf16_kernel<float>, dim3(blocks_for(pairs)), dim3(kPadThreads), 0, s,
                           static_cast<const float*>(src), static_cast<uint16_t*>(dst), rows, cols, R, C, pairs);
    return hipGetLastError();
}

hipError_t pad_bf16_two(const PadJob& a, const PadJob& b, int64_t batch, hipStream_t s) {
    if (a.C >= 512 && b.C >= 512 && aligned16(a.dst) && aligned16(b.dst)) {
        auto rows = [&](const PadJob& j) {
            return PadRows{j.src, static_cast<uint16_t*>(j.dst), j.rows, j.cols, j.R, j.C, batch * j.R, 0};
        };
        launch_pad_rows<float>(rows(a), rows(b), s);
        return hipGetLastError();
    }
    const hipError_t e = pad_bf16(0, a.src, a.dst, batch, a.rows, a.cols, a.R, a.C, s);
    return e != hipSuccess ? e : pad_bf16(0, b.src, b.dst, batch, b.rows, b.cols, b.R, b.C, s);
}

hipError_t crop_f32(const float* src, float* dst, int64_t batch, int64_t rows, int64_t cols, int64_t R, int64_t C,
                    hipStream_t s) {
    const int64_t total = batch * rows * cols;
    if (total == 0) return hipSuccess;
    if (cols >= 256) {
        const int64_t nrows = batch * rows;
        const int vec = cols % 4 == 0 && aligned16(src) && aligned16(dst);
        const dim3 grid(static_cast<unsigned>(nrows < kMaxFlatBlocks ? nrows : kMaxFlatBlocks));
        hipLaunchKernelGGL(crop_rows_kernel, grid, dim3(kPadThreads), 0, s, src, dst, rows, cols, R, C, nrows, vec);
        return hipGetLastError();
    }
    hipLaunchKernelGGL(crop_f32_kernel, dim3(blocks_for(total)), dim3(kPadThreads), 0, s, src, dst, rows, cols, R, C,
                       total);
    return hipGetLastError();
}

}  // namespace hk
