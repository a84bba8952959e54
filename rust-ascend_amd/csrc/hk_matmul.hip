// hk_matmul.hip — the generic floating matmul (F32, F16, BF16 with the input's own dtype out,
// FP32 accumulation), batch dimensions broadcast, any positive M/N/K, for gfx950.
//
// Semantics (reference: AscendRuntime::tensor_matmul, rust-ascend-driver/src/tensor/runtime/
// mod.rs:156-158 -> generic_matrix::matmul (generic_matrix.rs:17-54) -> worker.rs:128-162, which
// runs aclnnMatmul with cubeMathType 0 = KEEP_DTYPE): out[b..., i, j] = sum_k A[b_a..., i, k] *
// B[b_b..., k, j], A [..., M, K] and B [..., K, N] row-major, batch dims broadcast numpy-style
// (layout.rs:106-142), FP32 products and sums, the output rounded to the inputs' dtype (RNE).
//
// Design: F32 operands are read in place by matmul_f32_tile, whatever their extents, batch strides and
// alignment. F16 and BF16 operands (and F32 past 32-bit offsets) are first gathered into packed, zero-padded NT operands in the
// workspace, A' [G, Mp, Kp] and B' [G, Np, Kp] (B transposed on the way), one slice per output batch
// with the broadcast applied by the gather's batch strides (0 along a broadcast dim). Padding with
// zeros adds nothing to the sums. The product then runs on MFMA tiles without any bounds logic: BF16
// on the library's BF16 GEMM (hk_gemm.hip), F16 and F32 on 64x64-tile kernels, into C' [G, Mp, Np],
// from which the [G, M, N] output is cropped. This path serves the generic backend op (float_matmul);
// the transformer's own GEMMs use hk_gemm.hip directly.
#include "hk_common.hpp"
#include "hk_kernels.hpp"

#include <algorithm>
#include <cmath>
#include <type_traits>

namespace hk {

namespace {

typedef _Float16 f16x8_t __attribute__((ext_vector_type(8)));

constexpr int kMT = 64;  // output tile edge of both kernels
constexpr int kThreads = 256;

// dst[g][r][c] = src[batch g][r][c] (or, transposed, src[batch g][c][r]) for r < rows, c < cols,
// zero elsewhere; dst is [G, R, C]. The source offset of batch g is sum_d idx_d(g) * stride_d over
// the output batch dims (innermost last), a zero stride broadcasting that dim.
template <typename T>
__global__ void __launch_bounds__(256)
gather_pad(const T* __restrict__ src, T* __restrict__ dst, MatmulBatch mb, int64_t rows, int64_t cols,
           int64_t ld, int transpose, int64_t R, int64_t C) {
    const int64_t plane = R * C, total = plane * mb.count;
    for (int64_t i = flat_begin(256); i < total; i += flat_stride(256)) {
        const int64_t g = i / plane, rc = i - g * plane;
        const int64_t r = rc / C, c = rc - r * C;
        T v = T(0);
        if (r < rows && c < cols) {
            int64_t off = 0, rest = g;
            for (int d = mb.dims - 1; d >= 0; --d) {
                const int64_t idx = rest % mb.shape[d];
                rest /= mb.shape[d];
                off += idx * mb.stride[d];
            }
            v = transpose ? src[off + c * ld + r] : src[off + r * ld + c];
        }
        dst[i] = v;
    }
}

// dst[g][r][c] = src[g][r][c] for r < rows, c < cols; src is [G, R, C], dst [G, rows, cols].
template <typename T>
__global__ void __launch_bounds__(256)
crop(const T* __restrict__ src, T* __restrict__ dst, int64_t G, int64_t rows, int64_t cols, int64_t R, int64_t C) {
    const int64_t plane = rows * cols, total = plane * G;
    for (int64_t i = flat_begin(256); i < total; i += flat_stride(256)) {
        const int64_t g = i / plane, rc = i - g * plane;
        const int64_t r = rc / cols, c = rc - r * cols;
        dst[i] = src[(g * R + r) * C + c];
    }
}

__global__ void __launch_bounds__(256) zero_u8(unsigned char* p, int64_t n) {
    for (int64_t i = flat_begin(256); i < n; i += flat_stride(256)) p[i] = 0;
}

// Epilogue of a 64x64 tile computed as four 32x32 MFMA blocks, B as the MFMA's first operand:
// lane l holds C[m = tm*64 + 32 wm + l%32][n = tn*64 + 32 wn + 8 grp + 4 (l/32) + 0..3] in
// acc[4 grp .. 4 grp + 3].
template <typename T>
__device__ __forceinline__ void store_tile64(T* C, int64_t ldc, int m0, int n0, int lane, const f32x16_t& acc) {
    const int m = m0 + (lane & 31);
#pragma unroll
    for (int grp = 0; grp < 4; ++grp) {
        const int n = n0 + grp * 8 + (lane >> 5) * 4;
        T* p = C + m * ldc + n;
#pragma unroll
        for (int e = 0; e < 4; ++e) p[e] = static_cast<T>(acc[grp * 4 + e]);
    }
}

// F32: C'[g] = A'[g] B'[g]^T with v_mfma_f32_32x32x2_f32. 64x64 tile per workgroup, four waves
// (2x2) of 32x32, K steps of 32 through LDS (rows padded to 36 floats: the 32 lanes of a
// half-wave read 32 rows at a 144-byte stride, each 8-lane group over distinct banks), the next
// step prefetched into registers. An MFMA takes one k pair per lane half: lane l contributes
// k = 8s + 4(l/32) + u to MFMA (s, u) for A and B alike, so the 16 MFMAs of a step cover its 32 k.
constexpr int kF32K = 32, kF32Ld = kF32K + 4;
__global__ void __launch_bounds__(kThreads)
matmul_f32_nt(const float* __restrict__ A, const float* __restrict__ B, float* __restrict__ C, int tiles_n,
              int64_t Mp, int64_t Np, int64_t Kp) {
    __shared__ __attribute__((aligned(16))) float la[2][kMT * kF32Ld];
    __shared__ __attribute__((aligned(16))) float lb[2][kMT * kF32Ld];
    const int tm = blockIdx.x / tiles_n, tn = blockIdx.x - (blockIdx.x / tiles_n) * tiles_n;
    const int64_t g = blockIdx.z;
    A += (g * Mp + tm * kMT) * Kp;
    B += (g * Np + tn * kMT) * Kp;
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const int wm = wave >> 1, wn = wave & 1, lr = lane & 31, h = lane >> 5;
    const int row = t >> 3, col = (t & 7) * 4;
    f32x4_t ra[2], rb[2];
    auto load = [&](int kt) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            ra[i] = *reinterpret_cast<const f32x4_t*>(A + (row + 32 * i) * Kp + kt * kF32K + col);
            rb[i] = *reinterpret_cast<const f32x4_t*>(B + (row + 32 * i) * Kp + kt * kF32K + col);
        }
    };
    auto stash = [&](int buf) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            *reinterpret_cast<f32x4_t*>(&la[buf][(row + 32 * i) * kF32Ld + col]) = ra[i];
            *reinterpret_cast<f32x4_t*>(&lb[buf][(row + 32 * i) * kF32Ld + col]) = rb[i];
        }
    };
    f32x16_t acc;
#pragma unroll
    for (int v = 0; v < 16; ++v) acc[v] = 0.0f;
    const int nk = static_cast<int>(Kp / kF32K);
    load(0);
    stash(0);
    if (nk > 1) load(1);
    __syncthreads();
    for (int kt = 0; kt < nk; ++kt) {
        const int cur = kt & 1;
#pragma unroll
        for (int s = 0; s < kF32K / 8; ++s) {
            const f32x4_t fa = *reinterpret_cast<const f32x4_t*>(&la[cur][(wm * 32 + lr) * kF32Ld + 8 * s + 4 * h]);
            const f32x4_t fb = *reinterpret_cast<const f32x4_t*>(&lb[cur][(wn * 32 + lr) * kF32Ld + 8 * s + 4 * h]);
#pragma unroll
            for (int u = 0; u < 4; ++u) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(fb[u], fa[u], acc, 0, 0, 0);
        }
        if (kt + 1 < nk) {
            stash(cur ^ 1);
            if (kt + 2 < nk) load(kt + 2);
        }
        __syncthreads();
    }
    store_tile64(C + g * Mp * Np, Np, tm * kMT + wm * 32, tn * kMT + wn * 32, lane, acc);
}

// F16: the same tile with v_mfma_f32_32x32x16_f16, K steps of 64 halves (LDS rows padded to 72
// halves = 144 bytes); lane l contributes k = 16s + 8(l/32) + 0..7 to MFMA s.
constexpr int kF16K = 64, kF16Ld = kF16K + 8;
template <typename TO>
__global__ void __launch_bounds__(kThreads)
matmul_f16_nt(const _Float16* __restrict__ A, const _Float16* __restrict__ B, TO* __restrict__ C, int tiles_n,
              int64_t Mp, int64_t Np, int64_t Kp) {
    __shared__ __attribute__((aligned(16))) _Float16 la[2][kMT * kF16Ld];
    __shared__ __attribute__((aligned(16))) _Float16 lb[2][kMT * kF16Ld];
    const int tm = blockIdx.x / tiles_n, tn = blockIdx.x - (blockIdx.x / tiles_n) * tiles_n;
    const int64_t g = blockIdx.z;
    A += (g * Mp + tm * kMT) * Kp;
    B += (g * Np + tn * kMT) * Kp;
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const int wm = wave >> 1, wn = wave & 1, lr = lane & 31, h = lane >> 5;
    const int row = t >> 3, col = (t & 7) * 8;
    f16x8_t ra[2], rb[2];
    auto load = [&](int kt) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            ra[i] = *reinterpret_cast<const f16x8_t*>(A + (row + 32 * i) * Kp + kt * kF16K + col);
            rb[i] = *reinterpret_cast<const f16x8_t*>(B + (row + 32 * i) * Kp + kt * kF16K + col);
        }
    };
    auto stash = [&](int buf) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            *reinterpret_cast<f16x8_t*>(&la[buf][(row + 32 * i) * kF16Ld + col]) = ra[i];
            *reinterpret_cast<f16x8_t*>(&lb[buf][(row + 32 * i) * kF16Ld + col]) = rb[i];
        }
    };
    f32x16_t acc;
#pragma unroll
    for (int v = 0; v < 16; ++v) acc[v] = 0.0f;
    const int nk = static_cast<int>(Kp / kF16K);
    load(0);
    stash(0);
    if (nk > 1) load(1);
    __syncthreads();
    for (int kt = 0; kt < nk; ++kt) {
        const int cur = kt & 1;
#pragma unroll
        for (int s = 0; s < kF16K / 16; ++s) {
            const f16x8_t fa = *reinterpret_cast<const f16x8_t*>(&la[cur][(wm * 32 + lr) * kF16Ld + 16 * s + 8 * h]);
            const f16x8_t fb = *reinterpret_cast<const f16x8_t*>(&lb[cur][(wn * 32 + lr) * kF16Ld + 16 * s + 8 * h]);
            acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(fb, fa, acc, 0, 0, 0);
        }
        if (kt + 1 < nk) {
            stash(cur ^ 1);
            if (kt + 2 < nk) load(kt + 2);
        }
        __syncthreads();
    }
    store_tile64(C + g * Mp * Np, Np, tm * kMT + wm * 32, tn * kMT + wn * 32, lane, acc);
}

// F32 product of one batch slice, read in place: no gather, no padding, no crop.
//
//   C[g][m][n] = sum_k A'[g][m][k] B'[g][n][k], A' stored [M, K] (row stride lda) or, A_MN, [K, M]; B'
//   stored [N, K] or, B_MN, [K, N]; any extents, 4-byte alignment.
//
// What bounds it is the F32 matrix rate (256 flop per clock and CU, 157 TFLOP/s): a 128x128 tile takes
// 2048 matrix clocks per 16 k against 16 KB of operands, so the loads only have to stay ahead.
// Tiles travel by global->LDS loads, whose range check zero-fills past the matrix, into a ring of NS
// stages of 16 k: 16-byte loads where an operand's rows are aligned, else 4-byte ones, of which the 64
// per 128x128 stage take the memory pipeline longer (~40 clocks each) than the MFMAs take. A K-major operand is staged as 64-byte rows of 16 k (16-byte chunks XOR (row /
// 4) % 4, so that 16 rows at one chunk lie in distinct banks), an MN-major one as rows of the tile's
// columns (column XOR 16 (k / 4), so that the four 16-lane groups of a read lie in distinct banks). An
// MFMA (16x16x4: half the accumulator traffic per flop of 32x32x2) takes one k per 16-lane group: group
// g contributes k = 4 g + u to MFMA u for A and B alike.
// Measured: 4096^3 1007 us (136 TFLOP/s); [4000, 1024] x [1024, 1000] with its two gradients 228 us, 378 with
// gathered operands and a 64x64 kernel; F32 error against float64 5.7e-7 -> 2.9e-7.
struct F32Args {
    const float* a;
    const float* b;
    float* c;  // [G][M][N], or with splits [splits][G][M][N]
    MatmulBatch ab, bb;
    int m, n, k;
    int lda, ldb;
    int tiles_m, tiles_n;
    int splits, steps_per_split;  // K in steps of 16
};

constexpr int kFK = 16;

__device__ __forceinline__ int64_t batch_offset(const MatmulBatch& mb, int64_t g) {
    int64_t off = 0;
    for (int d = mb.dims - 1; d >= 0; --d) {
        off += g % mb.shape[d] * mb.stride[d];
        g /= mb.shape[d];
    }
    return off;
}

// T: 128x128 (2) or 64x64 (1) tiles, four waves of 32 T x 32 T as 2T x 2T blocks of 16x16.
// VA, VB: 16-byte loads of A, B (16-byte aligned base, row stride a multiple of 4 floats).
template <int T, int NS, bool A_MN, bool B_MN, bool VA, bool VB>
__global__ void __launch_bounds__(kThreads, 2)
matmul_f32_tile(F32Args p) {
    constexpr int W = 64 * T;             // tile edge
    constexpr int kOp = W * kFK;          // floats of one operand's stage
    constexpr int kLoadsA = VA ? T : 4 * T, kLoads = kLoadsA + (VB ? T : 4 * T);  // per wave and stage
    static_assert((NS - 1) * kLoads < 64, "vmcnt range");
    __shared__ __attribute__((aligned(1024))) float ring[NS][2 * kOp];

    const int tiles = p.tiles_m * p.tiles_n, all = tiles * p.splits;
    int bid = blockIdx.x;
    if ((all & 7) == 0) bid = (bid & 7) * (all >> 3) + (bid >> 3);  // XCD-contiguous
    const int split = bid / tiles;
    bid -= split * tiles;
    constexpr int GROUP = 8;
    const int per_group = GROUP * p.tiles_n, first_m = bid / per_group * GROUP;
    const int gsize = min(p.tiles_m - first_m, GROUP);
    const int tm = first_m + bid % per_group % gsize, tn = bid % per_group / gsize;
    const int64_t g = blockIdx.z;
    const i32x4_t ra = buffer_resource(p.a + batch_offset(p.ab, g), (A_MN ? p.k : p.m) * p.lda * 4);
    const i32x4_t rb = buffer_resource(p.b + batch_offset(p.bb, g), (B_MN ? p.k : p.n) * p.ldb * 4);

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wm = wave >> 1, wn = wave & 1, l16 = lane & 15, g4 = lane >> 4;
    const int first = split * p.steps_per_split;
    const int nk = min((p.k + kFK - 1) / kFK - first, p.steps_per_split);

    // K-major 4-byte load q = wave + 4 d: rows 4 q .. 4 q + 3, whose XOR term is q % 4 = wave
    const int kk = (((lane & 15) >> 2) ^ wave) << 2 | (lane & 3);
    auto load = [&](const i32x4_t& r, float* dst, bool mn, bool vec, int row0, int ld, int step, int d) __attribute__((always_inline)) {
        const int q = wave + 4 * d;
        int off;
        if (mn) {  // k-rows of W columns
            const int per = vec ? 256 : 64, at = per * q + (vec ? 4 * lane : lane);
            const int k = at / W, pos = at % W;
            off = ((step * kFK + k) * ld + row0 + (pos ^ ((k >> 2) << 4))) * 4;
        } else if (vec) {  // 16 rows of four chunks
            const int k = step * kFK + (((lane & 3) ^ (lane >> 4)) << 2);
            off = k < p.k ? ((row0 + 16 * q + (lane >> 2)) * ld + k) * 4 : static_cast<int>(0x80000000u);
        } else {
            const int k = step * kFK + kk;
            off = k < p.k ? ((row0 + 4 * q + (lane >> 4)) * ld + k) * 4 : static_cast<int>(0x80000000u);
        }
        if (vec) load_lds16(r, lds_address(reinterpret_cast<const uint16_t*>(dst + 256 * q)), off, 0);
        else load_lds4(r, lds_address(reinterpret_cast<const uint16_t*>(dst + 64 * q)), off, 0);
    };
    auto fetch_one = [&](int slot, int step, int d) __attribute__((always_inline)) {
        if (d < kLoadsA) load(ra, ring[slot], A_MN, VA, tm * W, p.lda, step, d);
        else load(rb, ring[slot] + kOp, B_MN, VB, tn * W, p.ldb, step, d - kLoadsA);
    };
    auto fetch = [&](int slot, int step) __attribute__((always_inline)) {
#pragma unroll
        for (int d = 0; d < kLoads; ++d) fetch_one(slot, step, d);
    };
    // k = 4 g4 .. 4 g4 + 3 of row (column) `row` of a stage
    auto frag = [&](const float* t, bool mn, int row) __attribute__((always_inline)) {
        if (!mn) return *reinterpret_cast<const f32x4_t*>(t + row * kFK + ((g4 ^ ((row >> 2) & 3)) << 2));
        f32x4_t v;
#pragma unroll
        for (int u = 0; u < 4; ++u) v[u] = t[(4 * g4 + u) * W + (row ^ (g4 << 4))];
        return v;
    };

    // Two levels of accumulators: `acc` sums 256 k, then joins `sum`, so the error of a long contraction
    // grows with its number of blocks, not of products.
    constexpr int B = 2 * T;  // 16x16 blocks per wave and direction
    f32x4_t acc[B][B], sum[B][B];
    auto clear = [&](f32x4_t (&x)[B][B]) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < B; ++i)
#pragma unroll
            for (int j = 0; j < B; ++j) x[i][j] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
    };
    auto join = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < B; ++i)
#pragma unroll
            for (int j = 0; j < B; ++j)
#pragma unroll
                for (int e = 0; e < 4; ++e) sum[i][j][e] += acc[i][j][e];
    };
    clear(acc);
    clear(sum);

    // The MFMAs of a step run while the next step's operands are read. The barrier before them (step s + 1
    // landed, every read of step s done) frees the slot of step s for step s + NS. Past the last step
    // the loads repeat it.
    const int last = first + nk - 1;
    f32x4_t fa[2][B], fb[2][B];
    auto read_one = [&](int slot, auto buf, int f) __attribute__((always_inline)) {
        constexpr int N = decltype(buf)::value;
        if (f < B) fa[N][f] = frag(ring[slot], A_MN, 16 * (B * wm + f) + l16);
        else fb[N][f - B] = frag(ring[slot] + kOp, B_MN, 16 * (B * wn + f - B) + l16);
    };
    auto landed = [&](auto left) __attribute__((always_inline)) {
        constexpr int kLeft = decltype(left)::value;
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_waitcnt((kLeft & 15) | ((kLeft >> 4) << 14) | (7 << 4) | (0 << 8));
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };
    auto step = [&](int s, auto buf) __attribute__((always_inline)) {
        constexpr int N = decltype(buf)::value;
        landed(std::integral_constant<int, (NS - 2) * kLoads>{});
        // the next step's operand reads and the loads spread between the MFMAs (issue is in order)
        const int slot = s % NS, next = (s + 1) % NS, ahead = min(first + s + NS, last);
        constexpr int kMfma = 4 * B * B, kMem = 2 * B + kLoads;
#pragma unroll
        for (int e = 0; e < kMfma; ++e) {
            const int u = e / (B * B), i = e / B % B, j = e % B;
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(fb[N][j][u], fa[N][i][u], acc[i][j], 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int f = e * kMem / kMfma; f < (e + 1) * kMem / kMfma; ++f) {
                if (f < 2 * B) read_one(next, std::integral_constant<int, N ^ 1>{}, f);
                else fetch_one(slot, ahead, f - 2 * B);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        if ((s & 15) == 15) {
            join();
            clear(acc);
        }
    };
#pragma unroll
    for (int u = 0; u < NS; ++u) fetch(u, min(first + u, last));
    landed(std::integral_constant<int, (NS - 1) * kLoads>{});
#pragma unroll
    for (int f = 0; f < 2 * B; ++f) read_one(0, std::integral_constant<int, 0>{}, f);
    for (int s = 0; s < nk; s += 2) {
        step(s, std::integral_constant<int, 0>{});
        if (s + 1 < nk) step(s + 1, std::integral_constant<int, 1>{});
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // no load may still be writing LDS at exit
    join();

    float* c = p.c + (static_cast<int64_t>(split) * gridDim.z + g) * p.m * p.n;
    const bool vec = (p.n & 3) == 0 && (reinterpret_cast<uintptr_t>(p.c) & 15) == 0;
#pragma unroll
    for (int i = 0; i < B; ++i) {
        const int m = tm * W + 16 * (B * wm + i) + l16;
        if (m >= p.m) continue;
        float* row = c + static_cast<int64_t>(m) * p.n;
#pragma unroll
        for (int j = 0; j < B; ++j) {
            const int n = tn * W + 16 * (B * wn + j) + 4 * g4;
            if (vec && n < p.n) {
                *reinterpret_cast<f32x4_t*>(row + n) = sum[i][j];
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (n + e < p.n) row[n + e] = sum[i][j][e];
            }
        }
    }
}

// out = the sum over the splits, in order, of the partial planes [splits][total].
__global__ void __launch_bounds__(256)
sum_planes(const float* __restrict__ partial, float* __restrict__ out, int splits, int64_t total) {
    for (int64_t i = flat_begin(256); i < total; i += flat_stride(256)) {
        float sum = partial[i];
        for (int s = 1; s < splits; ++s) sum += partial[s * total + i];
        out[i] = sum;
    }
}

template <typename T> __device__ __forceinline__ T to_elem(float x);
template <> __device__ __forceinline__ float to_elem<float>(float x) { return x; }
template <> __device__ __forceinline__ _Float16 to_elem<_Float16>(float x) { return static_cast<_Float16>(x); }
template <> __device__ __forceinline__ uint16_t to_elem<uint16_t>(float x) { return f32_to_bf16(x); }  // BF16 RNE

// out[go][r][c] = sum over the output batches g that broadcast onto batch go of src[g][r][c], in
// increasing g, for r < rows, c < cols; src is [G, R, C] F32 (G = the output batch count), out
// [count of the operand's batch, rows, cols]. op_shape is the operand's batch shape aligned to the
// output's (1 along a dim it broadcasts), so with no broadcast dim this is a crop and a conversion.
template <typename T>
__global__ void __launch_bounds__(256)
reduce_batches(const float* __restrict__ src, T* __restrict__ out, MatmulBatch ob, MatmulBatch op, int64_t rows,
               int64_t cols, int64_t R, int64_t C) {
    const int64_t plane = rows * cols, total = plane * op.count;
    int64_t ostride[4], reps = 1, st = 1;
    for (int d = ob.dims - 1; d >= 0; --d) {
        ostride[d] = st;
        st *= ob.shape[d];
        if (op.shape[d] == 1) reps *= ob.shape[d];
    }
    for (int64_t i = flat_begin(256); i < total; i += flat_stride(256)) {
        const int64_t go = i / plane, rc = i - go * plane;
        const int64_t r = rc / cols, c = rc - r * cols;
        int64_t base = 0, rest = go;
        for (int d = ob.dims - 1; d >= 0; --d) {
            const int64_t idx = rest % op.shape[d];
            rest /= op.shape[d];
            base += idx * ostride[d];
        }
        float sum = 0.0f;
        for (int64_t rep = 0; rep < reps; ++rep) {  // the broadcast dims' indices, lexicographic
            int64_t g = base, q = rep;
            for (int d = ob.dims - 1; d >= 0; --d)
                if (op.shape[d] == 1) {
                    g += (q % ob.shape[d]) * ostride[d];
                    q /= ob.shape[d];
                }
            sum += src[(g * R + r) * C + c];
        }
        out[i] = to_elem<T>(sum);
    }
}

int64_t round_up(int64_t x, int64_t q) { return (x + q - 1) / q * q; }

// Padded extents of an NT product X [rows, K] Y [cols, K]^T: whole kernel tiles and K steps.
struct Padded {
    int64_t M, N, K;
};
Padded padded(int dtype, int64_t m, int64_t n, int64_t k) {
    const int64_t kq = dtype == 0 ? kF32K : dtype == 1 ? kF16K : 16;
    const int64_t mq = dtype == 27 ? 16 : kMT;
    return {round_up(m, mq), round_up(n, mq), round_up(k, kq)};
}

size_t round256(size_t x) { return (x + 255) & ~size_t(255); }

// One gathered operand: the [rows, cols] matrices of src (row stride ld, or transposed: element
// (r, c) at c * ld + r) over the output batches, strides in b.
struct Gather {
    const void* src;
    MatmulBatch b;
    int64_t rows, cols, ld;
    int transpose;
};

template <typename T>
void gather(const Gather& x, void* dst, int64_t R, int64_t C, hipStream_t st) {
    hipLaunchKernelGGL((gather_pad<T>), dim3(flat_blocks(x.b.count * R * C, 256)), dim3(256), 0, st,
                       static_cast<const T*>(x.src), static_cast<T*>(dst), x.b, x.rows, x.cols, x.ld, x.transpose, R,
                       C);
}

size_t product_bytes(int dtype, int64_t G, const Padded& p, bool out_f32) {
    const size_t es = dtype == 0 ? 4 : 2, eo = out_f32 ? 4 : es;
    return round256(G * p.M * p.K * es) + round256(G * p.N * p.K * es) + round256(G * p.M * p.N * eo);
}

// C'[g] = X[g] Y[g]^T for the output batches g, X [rows M, K] and Y [cols N, K] gathered into the
// workspace, zero-padded to p; C' [G, p.M, p.N] in F32 (out_f32) or the dtype, at *c (the
// workspace's third piece).
hipError_t product(int dtype, int64_t G, const Gather& x, const Gather& y, const Padded& p, bool out_f32,
                   void* workspace, void** c, int num_cus, hipStream_t st) {
    const size_t es = dtype == 0 ? 4 : 2;
    char* ws = static_cast<char*>(workspace);
    void* xp = ws;
    void* yp = ws + round256(G * p.M * p.K * es);
    void* cp = static_cast<char*>(yp) + round256(G * p.N * p.K * es);
    *c = cp;
    if (dtype == 0) {
        gather<float>(x, xp, p.M, p.K, st);
        gather<float>(y, yp, p.N, p.K, st);
    } else {
        gather<uint16_t>(x, xp, p.M, p.K, st);  // F16 and BF16 move as 16-bit words
        gather<uint16_t>(y, yp, p.N, p.K, st);
    }
    const size_t eo = out_f32 ? 4 : es;
    const int tiles_n = static_cast<int>(p.N / kMT);
    for (int64_t g0 = 0; g0 < G; g0 += 4096) {  // at most 4096 batches per launch
        const int64_t gc = G - g0 < 4096 ? G - g0 : 4096;
        const char* xg = static_cast<const char*>(xp) + g0 * p.M * p.K * es;
        const char* yg = static_cast<const char*>(yp) + g0 * p.N * p.K * es;
        char* cg = static_cast<char*>(cp) + g0 * p.M * p.N * eo;
        const dim3 grid(static_cast<unsigned>((p.M / kMT) * tiles_n), 1, static_cast<unsigned>(gc));
        if (dtype == 0) {
            hipLaunchKernelGGL(matmul_f32_nt, grid, dim3(kThreads), 0, st, reinterpret_cast<const float*>(xg),
                               reinterpret_cast<const float*>(yg), reinterpret_cast<float*>(cg), tiles_n, p.M, p.N, p.K);
        } else if (dtype == 1) {
            if (out_f32)
                hipLaunchKernelGGL((matmul_f16_nt<float>), grid, dim3(kThreads), 0, st,
                                   reinterpret_cast<const _Float16*>(xg), reinterpret_cast<const _Float16*>(yg),
                                   reinterpret_cast<float*>(cg), tiles_n, p.M, p.N, p.K);
            else
                hipLaunchKernelGGL((matmul_f16_nt<_Float16>), grid, dim3(kThreads), 0, st,
                                   reinterpret_cast<const _Float16*>(xg), reinterpret_cast<const _Float16*>(yg),
                                   reinterpret_cast<_Float16*>(cg), tiles_n, p.M, p.N, p.K);
        } else {
            // NT operands need no transposition, so the GEMM takes no workspace
            hipError_t e = gemm_bf16(xg, yg, cg, out_f32 ? 0 : 1, gc, p.M, p.N, p.K, 0, 1, nullptr, 0, num_cus, st);
            if (e != hipSuccess) return e;
        }
    }
    return hipGetLastError();
}

MatmulBatch packed_batch(const MatmulBatch& shape, int64_t plane) {  // a contiguous [G, ...] operand
    MatmulBatch b = shape;
    int64_t st = plane;
    for (int d = shape.dims - 1; d >= 0; --d) {
        b.stride[d] = st;
        st *= shape.shape[d];
    }
    return b;
}

MatmulBatch operand_shape(const MatmulBatch& out, const MatmulBatch& op) {  // 1 along broadcast dims
    MatmulBatch b = out;
    for (int d = 0; d < out.dims; ++d) b.shape[d] = op.stride[d] == 0 ? 1 : out.shape[d];
    b.count = 1;
    for (int d = 0; d < out.dims; ++d) b.count *= b.shape[d];
    return b;
}

hipError_t zero_fill(void* p, int64_t bytes, hipStream_t st) {
    if (bytes <= 0) return hipSuccess;
    hipLaunchKernelGGL(zero_u8, dim3(flat_blocks(bytes, 256)), dim3(256), 0, st, static_cast<unsigned char*>(p), bytes);
    return hipGetLastError();
}

template <typename T>
void reduce(const float* c, void* out, const MatmulBatch& ob, const MatmulBatch& op, int64_t rows, int64_t cols,
            int64_t R, int64_t C, hipStream_t st) {
    hipLaunchKernelGGL((reduce_batches<T>), dim3(flat_blocks(op.count * rows * cols, 256)), dim3(256), 0, st, c,
                       static_cast<T*>(out), ob, op, rows, cols, R, C);
}

void reduce_any(int dtype, const float* c, void* out, const MatmulBatch& ob, const MatmulBatch& op, int64_t rows,
                int64_t cols, int64_t R, int64_t C, hipStream_t st) {
    if (dtype == 0) reduce<float>(c, out, ob, op, rows, cols, R, C, st);
    else if (dtype == 1) reduce<_Float16>(c, out, ob, op, rows, cols, R, C, st);
    else reduce<uint16_t>(c, out, ob, op, rows, cols, R, C, st);
}

size_t matmul_gathered_bytes(const MatmulSpec& s) {
    return product_bytes(s.dtype, s.batch.count, padded(s.dtype, s.m, s.n, s.k), false);
}
size_t matmul_gathered_backward_bytes(const MatmulSpec& s) {
    const Padded pa = padded(s.dtype, s.m, s.k, s.n), pb = padded(s.dtype, s.k, s.n, s.m);
    return std::max(product_bytes(s.dtype, s.batch.count, pa, true), product_bytes(s.dtype, s.batch.count, pb, true));
}

// ---- F32 products read in place (matmul_f32_tile)

// One F32 product: the operands' storage and batch strides, C [G][m][n] packed.
struct F32Product {
    const float* a;
    const float* b;
    MatmulBatch ab, bb;
    int64_t m, n, k, lda, ldb;
    bool a_mn, b_mn;
    bool folded = false;  // the batch has joined M or K: C is the whole result
};

// Each operand slice and its padded tile edge within 32-bit byte offsets.
bool f32_fits(const F32Product& x) {
    auto fits = [](int64_t rows, int64_t ld) { return (rows + 128) * ld * 4 < (int64_t{1} << 31); };
    return fits(x.a_mn ? x.k : x.m, x.lda) && fits(x.b_mn ? x.k : x.n, x.ldb) && x.ab.count <= 65535 &&
           x.m <= INT32_MAX - 128 && x.n <= INT32_MAX - 128;
}

struct F32Choice {
    bool big;  // 128x128 tiles
    int splits;
};
// The tile and K split (at least 8 steps of 16 k each, partial planes of at most 64 MB) of least
// estimated time: a 128x128 workgroup takes ~0.95 us a step; 64x64 ones 0.26 us each, but at least 0.42
// when alone on their CU; a split adds a launch and its planes' traffic.
F32Choice f32_choose(const F32Product& x, int num_cus, size_t ws_bytes) {
    const int64_t steps = (x.k + kFK - 1) / kFK, plane = x.ab.count * x.m * x.n * 4;
    F32Choice best{false, 1};
    float best_us = INFINITY;
    for (bool big : {true, false}) {
        const int64_t w = big ? 128 : 64, tiles = ((x.m + w - 1) / w) * ((x.n + w - 1) / w) * x.ab.count;
        for (int splits = 1; splits <= 16; ++splits) {
            if (splits > 1 && (tiles * splits > 4 * num_cus || steps < 8 * splits || plane * splits > (int64_t{64} << 20) ||
                               static_cast<size_t>(plane * splits) > ws_bytes))
                break;
            const int64_t rounds = (tiles * splits + num_cus - 1) / num_cus, per = (steps + splits - 1) / splits;
            float us = big ? rounds * per * 0.95f : per * fmaxf(rounds * 0.26f, 0.42f);
            if (splits > 1) us += 4.0f + plane * (splits + 1) * 2.5e-7f;
            if (us < best_us) best_us = us, best = F32Choice{big, splits};
        }
    }
    return best;
}
size_t f32_bytes(const F32Product& x, int num_cus) {
    const F32Choice c = f32_choose(x, num_cus, SIZE_MAX);
    return c.splits > 1 ? round256(static_cast<size_t>(x.ab.count * x.m * x.n) * 4 * c.splits) : 0;
}

template <int T, bool A_MN, bool B_MN>
void f32_launch_mn(const F32Args& p, bool va, bool vb, const dim3& grid, hipStream_t st) {
    if (va && vb) hipLaunchKernelGGL((matmul_f32_tile<T, 4, A_MN, B_MN, true, true>), grid, dim3(kThreads), 0, st, p);
    else if (va) hipLaunchKernelGGL((matmul_f32_tile<T, 4, A_MN, B_MN, true, false>), grid, dim3(kThreads), 0, st, p);
    else if (vb) hipLaunchKernelGGL((matmul_f32_tile<T, 4, A_MN, B_MN, false, true>), grid, dim3(kThreads), 0, st, p);
    else hipLaunchKernelGGL((matmul_f32_tile<T, 4, A_MN, B_MN, false, false>), grid, dim3(kThreads), 0, st, p);
}
template <int T>
void f32_launch(const F32Args& p, bool a_mn, bool b_mn, bool va, bool vb, const dim3& grid, hipStream_t st) {
    if (a_mn && b_mn) f32_launch_mn<T, true, true>(p, va, vb, grid, st);
    else if (b_mn) f32_launch_mn<T, false, true>(p, va, vb, grid, st);
    else f32_launch_mn<T, false, false>(p, va, vb, grid, st);  // no product reads only A MN-major
}

// 16-byte loads: every row of every batch slice 16-byte aligned.
bool f32_vec(const float* x, const MatmulBatch& b, int64_t ld) {
    if (reinterpret_cast<uintptr_t>(x) % 16 != 0 || ld % 4 != 0) return false;
    for (int d = 0; d < b.dims; ++d)
        if (b.stride[d] % 4 != 0) return false;
    return true;
}

void f32_product(const F32Product& x, float* out, void* workspace, size_t ws_bytes, int num_cus, hipStream_t st) {
    const F32Choice c = f32_choose(x, num_cus, ws_bytes);
    F32Args p{};
    p.a = x.a, p.b = x.b, p.ab = x.ab, p.bb = x.bb;
    p.m = static_cast<int>(x.m), p.n = static_cast<int>(x.n), p.k = static_cast<int>(x.k);
    p.lda = static_cast<int>(x.lda), p.ldb = static_cast<int>(x.ldb);
    const int w = c.big ? 128 : 64, steps = (p.k + kFK - 1) / kFK;
    p.tiles_m = (p.m + w - 1) / w, p.tiles_n = (p.n + w - 1) / w;
    p.steps_per_split = (steps + c.splits - 1) / c.splits;
    p.splits = (steps + p.steps_per_split - 1) / p.steps_per_split;
    p.c = p.splits > 1 ? static_cast<float*>(workspace) : out;
    const dim3 grid(static_cast<unsigned>(p.tiles_m * p.tiles_n * p.splits), 1, static_cast<unsigned>(x.ab.count));
    const bool va = f32_vec(x.a, x.ab, x.lda), vb = f32_vec(x.b, x.bb, x.ldb);
    if (c.big) f32_launch<2>(p, x.a_mn, x.b_mn, va, vb, grid, st);
    else f32_launch<1>(p, x.a_mn, x.b_mn, va, vb, grid, st);
    if (p.splits > 1) {
        const int64_t total = x.ab.count * x.m * x.n;
        hipLaunchKernelGGL(sum_planes, dim3(flat_blocks(total, 256)), dim3(256), 0, st, p.c, out, p.splits, total);
    }
}

bool is_shared(const MatmulBatch& b) {  // every batch reads the same matrix
    for (int d = 0; d < b.dims; ++d)
        if (b.shape[d] > 1 && b.stride[d] != 0) return false;
    return true;
}
bool is_packed(const MatmulBatch& b, int64_t plane) {  // a contiguous [G, plane] operand
    int64_t st = plane;
    for (int d = b.dims - 1; d >= 0; --d) {
        if (b.shape[d] > 1 && b.stride[d] != st) return false;
        st *= b.shape[d];
    }
    return true;
}

// The three F32 products of a spec: out = A B, dA = dY B^T, dB = A^T dY. With one B for a packed batch
// of A the batch joins M (dB: the contraction), so B is read once and dB needs no sum over batches.
F32Product f32_forward(const MatmulSpec& s, const float* a, const float* b) {
    F32Product x{a, b, s.a_batch, s.b_batch, s.m, s.n, s.k, s.k, s.n, false, true};
    if (is_shared(s.b_batch) && is_packed(s.a_batch, s.m * s.k)) x.m *= s.batch.count, x.ab = x.bb = MatmulBatch{}, x.folded = true;
    return x;
}
F32Product f32_grad_a(const MatmulSpec& s, const float* dy, const float* b) {
    F32Product x{dy, b, packed_batch(s.batch, s.m * s.n), s.b_batch, s.m, s.k, s.n, s.n, s.n, false, false};
    if (is_shared(s.b_batch) && is_packed(s.a_batch, s.m * s.k)) x.m *= s.batch.count, x.ab = x.bb = MatmulBatch{}, x.folded = true;
    return x;
}
F32Product f32_grad_b(const MatmulSpec& s, const float* a, const float* dy) {
    F32Product x{a, dy, s.a_batch, packed_batch(s.batch, s.m * s.n), s.k, s.n, s.m, s.k, s.n, true, true};
    if (is_shared(s.b_batch) && is_packed(s.a_batch, s.m * s.k)) x.k *= s.batch.count, x.ab = x.bb = MatmulBatch{}, x.folded = true;
    return x;
}

// Bytes of an operand gradient's batch slices, which are summed over the batches the operand broadcasts
// along (0: the product is the gradient).
size_t f32_slice_bytes(const F32Product& x, const MatmulBatch& op) {
    return x.folded || x.ab.count == op.count ? 0 : round256(static_cast<size_t>(x.ab.count * x.m * x.n) * 4);
}

}  // namespace

Scratch matmul_workspace(const MatmulSpec& s, int num_cus) {
    if (s.dtype == 0) {
        const F32Product x = f32_forward(s, nullptr, nullptr);
        if (f32_fits(x)) return {0, f32_bytes(x, num_cus)};
    }
    const size_t bytes = matmul_gathered_bytes(s);
    return {bytes, bytes};
}

Scratch matmul_backward_workspace(const MatmulSpec& s, int num_cus) {
    if (s.dtype == 0) {
        const F32Product xa = f32_grad_a(s, nullptr, nullptr), xb = f32_grad_b(s, nullptr, nullptr);
        if (f32_fits(xa) && f32_fits(xb)) {
            const MatmulBatch oa = operand_shape(s.batch, s.a_batch), ob = operand_shape(s.batch, s.b_batch);
            const size_t na = f32_slice_bytes(xa, oa), nb = f32_slice_bytes(xb, ob);
            return {std::max(na, nb), std::max(na + f32_bytes(xa, num_cus), nb + f32_bytes(xb, num_cus))};
        }
    }
    const size_t bytes = matmul_gathered_backward_bytes(s);
    return {bytes, bytes};
}

int matmul_f32_route(const MatmulSpec& s, int which, size_t ws_bytes, int num_cus) {
    if (s.dtype != 0 || s.batch.count * s.m * s.n * s.k == 0) return -1;
    const F32Product xa = f32_grad_a(s, nullptr, nullptr), xb = f32_grad_b(s, nullptr, nullptr);
    const F32Product x = which == 0 ? f32_forward(s, nullptr, nullptr) : (which == 1 ? xa : xb);
    if (which == 0 ? !f32_fits(x) : !f32_fits(xa) || !f32_fits(xb)) return -1;
    const size_t slices = which == 0 ? 0 : f32_slice_bytes(x, operand_shape(s.batch, which == 1 ? s.a_batch : s.b_batch));
    const F32Choice c = f32_choose(x, num_cus, ws_bytes > slices ? ws_bytes - slices : 0);
    const int64_t steps = (x.k + kFK - 1) / kFK, per = (steps + c.splits - 1) / c.splits;
    return (c.big ? 128 : 64) + 1024 * static_cast<int>((steps + per - 1) / per);
}

hipError_t matmul(const MatmulSpec& s, const void* a, const void* b, void* out, void* workspace, size_t ws_bytes,
                  int num_cus, hipStream_t st) {
    const int64_t G = s.batch.count;
    const size_t es = s.dtype == 0 ? 4 : 2;
    if (G * s.m * s.n == 0) return hipSuccess;
    if (s.k == 0) return zero_fill(out, G * s.m * s.n * static_cast<int64_t>(es), st);  // an empty contraction
    if (s.dtype == 0) {
        const F32Product f = f32_forward(s, static_cast<const float*>(a), static_cast<const float*>(b));
        if (f32_fits(f)) {
            f32_product(f, static_cast<float*>(out), workspace, ws_bytes, num_cus, st);
            return hipGetLastError();
        }
    }
    const Padded p = padded(s.dtype, s.m, s.n, s.k);
    const Gather x{a, s.a_batch, s.m, s.k, s.k, 0}, y{b, s.b_batch, s.n, s.k, s.n, 1};
    void* c = nullptr;
    hipError_t e = product(s.dtype, G, x, y, p, false, workspace, &c, num_cus, st);
    if (e != hipSuccess) return e;
    if (s.dtype == 0)
        hipLaunchKernelGGL((crop<float>), dim3(flat_blocks(G * s.m * s.n, 256)), dim3(256), 0, st,
                           static_cast<const float*>(c), static_cast<float*>(out), G, s.m, s.n, p.M, p.N);
    else
        hipLaunchKernelGGL((crop<uint16_t>), dim3(flat_blocks(G * s.m * s.n, 256)), dim3(256), 0, st,
                           static_cast<const uint16_t*>(c), static_cast<uint16_t*>(out), G, s.m, s.n, p.M, p.N);
    return hipGetLastError();
}

hipError_t matmul_backward(const MatmulSpec& s, const void* a, const void* b, const void* dy, void* da, void* db,
                           void* workspace, size_t ws_bytes, int num_cus, hipStream_t st) {
    const int64_t G = s.batch.count;
    const size_t es = s.dtype == 0 ? 4 : 2;
    const MatmulBatch oa = operand_shape(s.batch, s.a_batch), obb = operand_shape(s.batch, s.b_batch);
    const MatmulBatch dyb = packed_batch(s.batch, s.m * s.n);
    hipError_t e;
    if (G * s.m * s.n == 0) {  // no output elements: both gradients are zero
        if ((e = zero_fill(da, oa.count * s.m * s.k * static_cast<int64_t>(es), st)) != hipSuccess) return e;
        return zero_fill(db, obb.count * s.k * s.n * static_cast<int64_t>(es), st);
    }
    if (s.k == 0) return hipSuccess;  // dA [.., M, 0] and dB [.., 0, N] hold nothing
    if (s.dtype == 0) {
        const F32Product xa = f32_grad_a(s, static_cast<const float*>(dy), static_cast<const float*>(b));
        const F32Product xb = f32_grad_b(s, static_cast<const float*>(a), static_cast<const float*>(dy));
        if (f32_fits(xa) && f32_fits(xb)) {
            auto grad = [&](const F32Product& x, const MatmulBatch& op, void* out) {
                const size_t bytes = f32_slice_bytes(x, op);
                if (bytes == 0) {
                    f32_product(x, static_cast<float*>(out), workspace, ws_bytes, num_cus, st);
                    return;
                }
                float* slices = static_cast<float*>(workspace);  // summed over the broadcast batches
                f32_product(x, slices, static_cast<char*>(workspace) + bytes, ws_bytes - bytes, num_cus, st);
                reduce<float>(slices, out, s.batch, op, x.m, x.n, x.m, x.n, st);
            };
            grad(xa, oa, da);
            grad(xb, obb, db);
            return hipGetLastError();
        }
    }
    void* c = nullptr;
    // dA[g] = dY[g] B[g]^T: X = dY [M, N], Y = B as [K, N]; then summed over A's broadcast batches
    {
        const Padded p = padded(s.dtype, s.m, s.k, s.n);
        const Gather x{dy, dyb, s.m, s.n, s.n, 0}, y{b, s.b_batch, s.k, s.n, s.n, 0};
        if ((e = product(s.dtype, G, x, y, p, true, workspace, &c, num_cus, st)) != hipSuccess) return e;
        reduce_any(s.dtype, static_cast<const float*>(c), da, s.batch, oa, s.m, s.k, p.M, p.N, st);
    }
    // dB[g] = A[g]^T dY[g]: X = A^T [K, M], Y = dY^T [N, M]; then summed over B's broadcast batches
    {
        const Padded p = padded(s.dtype, s.k, s.n, s.m);
        const Gather x{a, s.a_batch, s.k, s.m, s.k, 1}, y{dy, dyb, s.n, s.m, s.n, 1};
        if ((e = product(s.dtype, G, x, y, p, true, workspace, &c, num_cus, st)) != hipSuccess) return e;
        reduce_any(s.dtype, static_cast<const float*>(c), db, s.batch, obb, s.k, s.n, p.M, p.N, st);
    }
    return hipGetLastError();
}

}  // namespace hk
