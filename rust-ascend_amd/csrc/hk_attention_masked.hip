// hk_attention_masked.hip — the materialized attention's score passes on 16 query rows a workgroup
// (additive F32 mask, any head and value width), for key counts whose scores fit the registers.
//
// Semantics (reference: src/nn/attention.rs:10-67): S = bf16(Q) bf16(K)^T in F32, S * scale (+ mask),
// P = softmax (F32), O = bf16(P) bf16(V); the gradient recomputes P: dP = bf16(dO) bf16(V)^T,
// dS = P (dP - sum(P dP)), dQ = bf16(scale dS) bf16(K). dK and dV are products of the BF16 P and dS
// that the backward pass writes.
//
// A GEMM per score matrix and a row pass over them wrote and read 4 bytes a score two (forward) or
// five (backward) times; here a score exists only as an accumulator, so what is left is the mask's 4
// bytes (and the backward's 2 + 2 bytes of P and dS, 4 of a mask gradient). 32 heads of 1040 x 1056
// scores, D = Dv = 64: forward 126 -> 55 us, backward 285 -> 140 (92 of them this kernel; the mask and
// the stores would take 26 and 52 at 5.5 TB/s). What bounds them besides is the address unit (16 clocks
// for a 1 KB operand load, 36 of them per wave and 32 columns) and the arithmetic of 20 instructions a
// score, both overlapped with the traffic by two workgroups on a CU.
// Layout: the four waves of a workgroup take the 32-key blocks in turn, for the same 16 query rows.
// S^T = K Q^T on 16x16x32 MFMAs: a lane's accumulators are one query (lane & 15) and, with the keys
// of a block dealt to the two tiles' rows in fours, the 8 consecutive keys 8 (lane >> 4): whole
// cache lines of the mask, 16-byte stores of P and dS, and P^T or dS^T packed to BF16 is at once the
// B operand of the product that follows. K and V come in fragment order (pack_operands; a copy that the
// rounding to BF16 makes anyway), from L2 straight into operands: every workgroup of a KV head passes
// over them, so a head's workgroups share an XCD.
#include "hk_common.hpp"
#include "hk_kernels.hpp"

#include <type_traits>

namespace hk {

namespace {

constexpr int kRowsPerWg = 16;
constexpr int kMaxBlocks = 9;   // 32-key blocks a wave holds: 72 registers of scores, of dP and of operands each
constexpr int kChunk = 128;     // output columns summed over the waves at a time
constexpr int kPastEnd = 0x7ffffff0;  // a byte offset past every buffer: loads of it return 0
constexpr float kLog2e = 1.4426950408889634f, kLog2eLow = 1.925963033500e-8f;  // log2(e) = their sum
constexpr float kLn2 = 0.6931471805599453f;

struct MaskedArgs {
    const uint16_t* q;     // [groups][rows][d]
    const uint16_t* k;     // K as score fragments
    const uint16_t* v;     // backward: V as score fragments
    const uint16_t* dout;  // backward: [groups][rows][dv]
    const uint16_t* xt;    // V (forward) or K (backward) as transposed fragments
    const float* mask;     // [groups][rows][n] or null
    uint16_t* p;           // backward: bf16(P) and bf16(scale dS) [groups][rows][n]
    uint16_t* ds;
    float* dmask;          // backward: dS in F32, or null
    void* out;             // O [groups][rows][dv] (forward) or dQ [groups][rows][d] (backward)
    float scale;
    int out_bf16, rows, n, d, dv;
};

__device__ __forceinline__ u32x4_t load16(__amdgpu_buffer_rsrc_t r, int off) {
    return __builtin_bit_cast(u32x4_t, __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 0));
}
__device__ __forceinline__ __amdgpu_buffer_rsrc_t resource(const void* p, int64_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, static_cast<int>(bytes), kBufferConfig);
}

// A wave's operand registers: two 16-byte loads for each of its key blocks. Every phase consumes a block's
// pair and at once reloads it with what the wave needs next (the next columns, the mask, the next
// matrix), so all of them are in flight while the others are used.
template <int MAXB>
using Pairs = u32x4_t[MAXB][2];

// The operand loads of a score product: 32-column step ks of the query rows, and of the keys' fragments.
struct ScoreLoads {
    __amdgpu_buffer_rsrc_t queries, keys;
    int width, steps, first, stride, query_off, col;
    __device__ __forceinline__ ScoreLoads(const uint16_t* q, const uint16_t* k, int64_t group, int n, int w, int waves,
                                          int wave, int lane)
        : queries(resource(q, static_cast<int64_t>(kRowsPerWg) * w * 2)), width(w), steps((w + 31) / 32) {
        const int64_t bytes = static_cast<int64_t>(n) * steps * 64;
        keys = resource(reinterpret_cast<const char*>(k) + group * bytes, bytes);
        first = wave * steps * 2048 + lane * 16;
        stride = waves * steps * 2048;
        col = 8 * (lane >> 4);
        query_off = (lane & 15) * w * 2 + col * 2;
    }
    __device__ __forceinline__ u32x4_t query(int ks) const {
        return load16(queries, ks * 32 + col < width ? query_off + ks * 64 : kPastEnd);
    }
    __device__ __forceinline__ u32x4_t key(int ks, int b, int t) const {  // past the last block: 0
        return load16(keys, first + b * stride + ks * 2048 + t * 1024);
    }
};

// acc[b] += the product of a score's column step held in f, f[b] = next(b, tile)
template <int MAXB, class Next>
__device__ __forceinline__ void score_step(f32x4_t (&acc)[MAXB][2], u32x4_t q, Pairs<MAXB>& f, Next&& next) {
#pragma unroll
    for (int b = 0; b < MAXB; ++b) {
#pragma unroll
        for (int t = 0; t < 2; ++t)
            acc[b][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, f[b][t]),
                                                                __builtin_bit_cast(bf16x8_t, q), acc[b][t], 0, 0, 0);
#pragma unroll
        for (int t = 0; t < 2; ++t) f[b][t] = next(b, t);
        __builtin_amdgcn_sched_barrier(0);
    }
}

// The scores of every column step; q and f hold step 0, f ends with `after`'s loads.
template <int MAXB, class After>
__device__ __forceinline__ void scores(const ScoreLoads& l, f32x4_t (&acc)[MAXB][2], u32x4_t q, Pairs<MAXB>& f, After&& after) {
#pragma unroll
    for (int b = 0; b < MAXB; ++b) acc[b][0] = acc[b][1] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
    for (int ks = 1; ks < l.steps; ++ks) {
        const u32x4_t qn = l.query(ks);
        score_step<MAXB>(acc, q, f, [&](int b, int t) { return l.key(ks, b, t); });
        q = qn;
    }
    score_step<MAXB>(acc, q, f, after);
}

// A query's maximum or sum over its lanes (lane, lane ^ 16, ^ 32, ^ 48) of every wave.
template <bool MAX, int W>
__device__ __forceinline__ float over_waves(float v, float (*scratch)[16], int wave, int lane) {
#pragma unroll
    for (int s = 16; s < 64; s *= 2) {
        const float o = __shfl_xor(v, s);
        v = MAX ? fmaxf(v, o) : v + o;
    }
    if (lane < 16) scratch[wave][lane] = v;
    __syncthreads();
    v = scratch[0][lane & 15];
#pragma unroll
    for (int w = 1; w < W; ++w) v = MAX ? fmaxf(v, scratch[w][lane & 15]) : v + scratch[w][lane & 15];
    return v;
}

// Between the order of a row block in memory (16 rows; consecutive lanes take consecutive 16 bytes of a
// row) and a lane's 8 keys of one query, through the wave's own LDS: with 16 lanes on 16 rows a memory
// access takes 64 clocks of the address unit instead of 16. 16-byte slots are exchanged within a row so
// that 16 lanes meet all banks both ways. F32 blocks: 32 keys, 8 slots a row; BF16 blocks: 4 slots.
__device__ __forceinline__ void wave_fence() {  // LDS accesses of a wave execute in order
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}
__device__ __forceinline__ int f32_slot(int row, int c) { return (row * 8 + (c ^ (row >> 1 & 7))) * 4; }
__device__ __forceinline__ int bf16_slot(int row, int c) { return (row * 4 + (c ^ (row >> 2))) * 4; }

constexpr int kBatch = 4;  // blocks in a wave's LDS at a time

// e^x for x <= 0 within an ulp or two: 2^t of the rounded product t = x log2(e), whose rounding (up to |t| / 2 ulps of
// the result: 2e-6 of it at x = -60) is taken back in first order. Where t is -inf (x as well, or near the type's lowest
// value) the remainder is a NaN or infinite, which the median bounds, and r is 0; x = NaN makes r one. For dMask, the
// one result that holds the weights in F32; where they only go on in BF16 (2^-9) the plain power is the same.
__device__ __forceinline__ float exp_f32(float x) {
    const float t = x * kLog2e;
    const float rest = __builtin_amdgcn_fmed3f(fmaf(x, kLog2eLow, fmaf(x, kLog2e, -t)), -1.0f, 1.0f);
    const float r = __builtin_amdgcn_exp2f(t);
    return fmaf(r * rest, kLn2, r);
}

// f[b]: rows lane / 8 (+ 8) in memory order -> query r, keys 8 g + 4 t
template <int MAXB>
__device__ __forceinline__ void rows_to_queries(Pairs<MAXB>& f, uint32_t* lds, int lane) {
#pragma unroll
    for (int b0 = 0; b0 < MAXB; b0 += kBatch) {
#pragma unroll
        for (int b = b0; b < MAXB && b < b0 + kBatch; ++b)
#pragma unroll
            for (int t = 0; t < 2; ++t)
                *reinterpret_cast<u32x4_t*>(lds + (b - b0) * 512 + f32_slot(8 * t + (lane >> 3), lane & 7)) = f[b][t];
        wave_fence();
#pragma unroll
        for (int b = b0; b < MAXB && b < b0 + kBatch; ++b)
#pragma unroll
            for (int t = 0; t < 2; ++t)
                f[b][t] = *reinterpret_cast<const u32x4_t*>(lds + (b - b0) * 512 + f32_slot(lane & 15, 2 * (lane >> 4) + t));
        wave_fence();
    }
}

// x[b]: query r, keys 8 g..8 g + 7 -> row lane / 4, keys 8 (lane & 3)..
template <int MAXB>
__device__ __forceinline__ void store_rows(const u32x4_t (&x)[MAXB], uint16_t* out, int64_t row0, int n, int first, int stride,
                                           uint32_t* lds, int lane) {
    const int row = lane >> 2, key = first + 8 * (lane & 3);
    uint16_t* p = out + (row0 + row) * n + key;
#pragma unroll
    for (int b0 = 0; b0 < MAXB; b0 += 2 * kBatch) {
#pragma unroll
        for (int b = b0; b < MAXB && b < b0 + 2 * kBatch; ++b)
            *reinterpret_cast<u32x4_t*>(lds + (b - b0) * 256 + bf16_slot(lane & 15, lane >> 4)) = x[b];
        wave_fence();
#pragma unroll
        for (int b = b0; b < MAXB && b < b0 + 2 * kBatch; ++b) {
            const u32x4_t v = *reinterpret_cast<const u32x4_t*>(lds + (b - b0) * 256 + bf16_slot(row, lane & 3));
            if (key + b * stride < n) *reinterpret_cast<u32x4_t*>(p + b * stride) = v;
        }
        wave_fence();
    }
}

template <int MAXB, int W, bool BWD>
__global__ void __launch_bounds__(64 * W) __attribute__((amdgpu_waves_per_eu(MAXB <= 4 ? 4 : 2)))
masked_attention(MaskedArgs a) {
    __shared__ float stat[3][W][16];
    __shared__ float part[W][kRowsPerWg][kChunk + 4];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int r = lane & 15, g = lane >> 4;
    const int row_blocks = a.rows / kRowsPerWg;
    const int logical = xcd_logical();
    const int64_t group = logical / row_blocks;
    const int64_t row0 = group * a.rows + (logical % row_blocks) * kRowsPerWg;  // of all groups
    const int n = a.n, key0 = wave * 32 + 8 * g;  // this lane's keys: key0 + 32 W b + 0..7

    const ScoreLoads qk(a.q + row0 * a.d, a.k, group, n, a.d, W, wave, lane);
    const ScoreLoads dv(BWD ? a.dout + row0 * a.dv : a.q, BWD ? a.v : a.k, group, n, a.dv, W, wave, lane);
    const auto rm = resource(a.mask ? a.mask + row0 * n : nullptr, a.mask ? static_cast<int64_t>(kRowsPerWg) * n * 4 : 0);
    const int width = BWD ? a.d : a.dv;  // of the product that follows
    const auto rx = resource(a.xt + group * n * width, static_cast<int64_t>(n) * width * 2);
    const int x_block = width * 64, x_first = wave * x_block + lane * 16;
    auto load_x = [&](int c, int b, int t) __attribute__((always_inline)) {  // columns c + 16 t; past the last block: 0
        return load16(rx, x_first + b * (W * x_block) + c * 64 + t * 1024);
    };

    Pairs<MAXB> f;
    const u32x4_t q0 = qk.query(0);
#pragma unroll
    for (int b = 0; b < MAXB; ++b) f[b][0] = qk.key(0, b, 0), f[b][1] = qk.key(0, b, 1);
    f32x4_t s[MAXB][2];
    uint32_t* const own = reinterpret_cast<uint32_t*>(&part[wave][0][0]);
    static_assert(sizeof(part[0]) >= kBatch * 2048, "a wave's blocks in LDS");
    const int mask_at = ((lane >> 3) * n + wave * 32 + 4 * (lane & 7)) * 4;
    scores<MAXB>(qk, s, q0, f, [&](int b, int t) { return load16(rm, mask_at + b * (W * 128) + t * 32 * n); });
    rows_to_queries<MAXB>(f, own, lane);

    // x = S * scale + mask (no mask loads 0); blocks past the last key never win the maximum and add 0
    const u32x4_t d0 = BWD ? dv.query(0) : q0;
    float m = -INFINITY;
#pragma unroll
    for (int b = 0; b < MAXB; ++b) {
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            const f32x4_t k = __builtin_bit_cast(f32x4_t, f[b][t]);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const float x = s[b][t][e] * a.scale + k[e];
                s[b][t][e] = key0 + 32 * W * b < n ? x : -INFINITY;
                m = fmaxf(m, s[b][t][e]);
            }
            f[b][t] = BWD ? dv.key(0, b, t) : load_x(0, b, t);
        }
        __builtin_amdgcn_sched_barrier(0);
    }
    m = over_waves<true, W>(m, stat[0], wave, lane);

    f32x4_t dp[BWD ? MAXB : 1][2];
    if constexpr (BWD) scores<MAXB>(dv, dp, d0, f, [&](int b, int t) { return f[b][t]; });  // no registers for K^T yet
    // The sums join a tile's four terms before the running sum: with one term at a time its rounding (72 terms a
    // lane) showed in every weight of the row, dMask 1-4% further from float64 than by the row kernels.
    float sum = 0.0f, dot = 0.0f;
    auto weigh = [&](auto exact) __attribute__((always_inline)) {
#pragma unroll
        for (int b = 0; b < MAXB; ++b)
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                f32x4_t& w = s[b][t];
#pragma unroll
                for (int e = 0; e < 4; ++e) w[e] = decltype(exact)::value ? exp_f32(w[e] - m) : __builtin_amdgcn_exp2f((w[e] - m) * kLog2e);
                sum += (w[0] + w[1]) + (w[2] + w[3]);
                if constexpr (BWD) dot += (w[0] * dp[b][t][0] + w[1] * dp[b][t][1]) + (w[2] * dp[b][t][2] + w[3] * dp[b][t][3]);
            }
    };
    if (BWD && a.dmask != nullptr) weigh(std::true_type{});
    else weigh(std::false_type{});
    const float inv = 1.0f / over_waves<false, W>(sum, stat[1], wave, lane);
    if constexpr (BWD) dot = over_waves<false, W>(dot, stat[2], wave, lane) * inv;

    // P and, in the backward, scale dS: packed to BF16, 8 keys a lane
    u32x4_t x[MAXB];
#pragma unroll
    for (int b = 0; b < MAXB; ++b)
#pragma unroll
        for (int t = 0; t < 2; ++t) {
#pragma unroll
            for (int e = 0; e < 4; ++e) s[b][t][e] *= inv;
            x[b][2 * t] = pack_bf16x2(s[b][t][0], s[b][t][1]);
            x[b][2 * t + 1] = pack_bf16x2(s[b][t][2], s[b][t][3]);
        }
    if constexpr (BWD) {
        store_rows<MAXB>(x, a.p, row0, n, wave * 32, W * 32, own, lane);
#pragma unroll
        for (int b = 0; b < MAXB; ++b) {
            const bool in = key0 + 32 * W * b < n;
            const int64_t at = (row0 + r) * n + key0 + 32 * W * b;
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                f32x4_t d;
#pragma unroll
                for (int e = 0; e < 4; ++e) d[e] = s[b][t][e] * (dp[b][t][e] - dot);
                if (a.dmask != nullptr && in) *reinterpret_cast<f32x4_t*>(a.dmask + at + 4 * t) = d;
#pragma unroll
                for (int e = 0; e < 4; ++e) d[e] *= a.scale;
                x[b][2 * t] = pack_bf16x2(d[0], d[1]);
                x[b][2 * t + 1] = pack_bf16x2(d[2], d[3]);
                f[b][t] = load_x(0, b, t);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        store_rows<MAXB>(x, a.ds, row0, n, wave * 32, W * 32, own, lane);
    }

    // O^T = V^T P^T or dQ^T = K^T dS^T: each wave over its own keys, then the waves' sums in wave order
    for (int c0 = 0; c0 < width; c0 += kChunk) {
        const int cols = min(kChunk, width - c0);
        if (c0 > 0) __syncthreads();  // the last chunk's sums are read
        for (int c = 0; c < cols; c += 32) {
            f32x4_t acc[2] = {{0.0f, 0.0f, 0.0f, 0.0f}, {0.0f, 0.0f, 0.0f, 0.0f}};
#pragma unroll
            for (int b = 0; b < MAXB; ++b) {
#pragma unroll
                for (int t = 0; t < 2; ++t) {
                    acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, f[b][t]),
                                                                     __builtin_bit_cast(bf16x8_t, x[b]), acc[t], 0, 0, 0);
                    f[b][t] = load_x(c0 + c + 32, b, t);  // past the last column: never used
                }
                __builtin_amdgcn_sched_barrier(0);
            }
#pragma unroll
            for (int t = 0; t < 2; ++t)
                if (c + 16 * t < cols) *reinterpret_cast<f32x4_t*>(&part[wave][r][c + 16 * t + 4 * g]) = acc[t];
        }
        __syncthreads();
        for (int i = threadIdx.x; i < kRowsPerWg * (cols / 4); i += 64 * W) {
            const int row = i / (cols / 4), c = i % (cols / 4) * 4;
            f32x4_t o = *reinterpret_cast<const f32x4_t*>(&part[0][row][c]);
#pragma unroll
            for (int w = 1; w < W; ++w) o += *reinterpret_cast<const f32x4_t*>(&part[w][row][c]);
            const int64_t at = (row0 + row) * width + c0 + c;
            if (a.out_bf16)
                *reinterpret_cast<u32x2_t*>(static_cast<uint16_t*>(a.out) + at) =
                    u32x2_t{pack_bf16x2(o[0], o[1]), pack_bf16x2(o[2], o[3])};
            else
                *reinterpret_cast<f32x4_t*>(static_cast<float*>(a.out) + at) = o;
        }
    }
}

// K or V [groups][n][w] as the 1 KB fragments that a wave loads an MFMA operand by (16 bytes a lane; read
// row by row, each load would touch 16 lines):
//   score fragments [n / 32][ceil(w / 32)][2]: tile t, lane (r, g): key 8 (r >> 2) + 4 t + (r & 3) of the
//   block, columns 8 g..8 g + 7 of the step (0 past w)
//   transposed fragments [n / 32][w / 16]: lane (r, g): column r of the tile, keys 8 g..8 g + 7
constexpr int kPackCols = 128;
struct PackArgs {
    hk::PackJob job[3];
    int last[3];  // column blocks up to and with the job
    int n;
};

template <class T>
__device__ __forceinline__ void pack_load(const PackJob& j, int64_t row, int c, uint16_t* out) {
    float v[8];
    load8(static_cast<const T*>(j.in) + row * j.w + c, v);
    store8(out, v);
}

__global__ void __launch_bounds__(256)
pack_operands(PackArgs a) {
    __shared__ __attribute__((aligned(16))) uint16_t tile[32][kPackCols + 8];
    const int cb = blockIdx.y, which = cb < a.last[0] ? 0 : (cb < a.last[1] ? 1 : 2);
    const PackJob j = a.job[which];
    const int c0 = (cb - (which ? a.last[which - 1] : 0)) * kPackCols;
    const int64_t group = blockIdx.z;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const int key = i * 16 + (threadIdx.x >> 4), c = (threadIdx.x & 15) * 8;
        const int64_t row = group * a.n + blockIdx.x * 32 + key;
        if (c0 + c >= j.w) *reinterpret_cast<u32x4_t*>(&tile[key][c]) = u32x4_t{0, 0, 0, 0};
        else if (j.bf16) pack_load<uint16_t>(j, row, c0 + c, &tile[key][c]);
        else pack_load<float>(j, row, c0 + c, &tile[key][c]);
    }
    __syncthreads();
    const int steps = (j.w + 31) / 32, tiles = j.w / 16;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const int f = i * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
        if (!j.transposed) {
            const int step = c0 / 32 + (f >> 1), t = f & 1;
            if (step < steps)
                *reinterpret_cast<u32x4_t*>(j.out + (((group * (a.n / 32) + blockIdx.x) * steps + step) * 2 + t) * 512 + lane * 8) =
                    *reinterpret_cast<const u32x4_t*>(&tile[8 * (r >> 2) + 4 * t + (r & 3)][(f >> 1) * 32 + 8 * g]);
        } else if (c0 / 16 + f < tiles) {
            u32x4_t w;
#pragma unroll
            for (int e = 0; e < 4; ++e)
                w[e] = tile[8 * g + 2 * e][16 * f + r] | static_cast<uint32_t>(tile[8 * g + 2 * e + 1][16 * f + r]) << 16;
            *reinterpret_cast<u32x4_t*>(j.out + ((group * (a.n / 32) + blockIdx.x) * tiles + c0 / 16 + f) * 512 + lane * 8) = w;
        }
    }
}

// Four waves up to the key blocks that they can hold, then eight (past 2304 keys neither can).
template <int W, bool BWD, int B>
void launch_blocks(int blocks, unsigned grid, const MaskedArgs& a, hipStream_t s) {
    if constexpr (B < kMaxBlocks) {
        if (blocks > B) return launch_blocks<W, BWD, B + 1>(blocks, grid, a, s);
    }
    hipLaunchKernelGGL((masked_attention<B, W, BWD>), dim3(grid), dim3(64 * W), 0, s, a);
}
template <bool BWD>
void launch(int64_t groups, const MaskedArgs& a, hipStream_t s) {
    const unsigned grid = static_cast<unsigned>(groups * (a.rows / kRowsPerWg));
    const int blocks = a.n / 32;
    if (blocks <= 4 * kMaxBlocks) launch_blocks<4, BWD, 1>((blocks + 3) / 4, grid, a, s);
    else launch_blocks<8, BWD, kMaxBlocks / 2>((blocks + 7) / 8, grid, a, s);
}

}  // namespace

// Up to the keys whose scores eight waves hold. A workgroup passes over K and V for 16 query rows, a GEMM
// for 128 or more, so wide heads belong to the GEMMs: at the size above D = Dv = 256 takes 135 and 320 us
// (forward, backward) here and 183 and 391 there, 512 takes 248 and 538 here and 252 and 530 there.
bool masked_attention_applies(int64_t groups, int64_t rows, int64_t n, int64_t d, int64_t dv) {
    return d + dv <= 768 && n <= 32 * 8 * kMaxBlocks && n % 32 == 0 && rows % kRowsPerWg == 0 && d % 16 == 0 && dv % 16 == 0 &&
           groups <= 65535 && groups * (rows / kRowsPerWg) < (int64_t{1} << 30);
}

hipError_t masked_attention_forward(const void* q, const void* k, const void* vt, const float* mask, float scale, void* o,
                                    bool out_bf16, int64_t groups, int64_t rows, int64_t n, int64_t d, int64_t dv,
                                    hipStream_t s) {
    MaskedArgs a{};
    a.q = static_cast<const uint16_t*>(q);
    a.k = static_cast<const uint16_t*>(k);
    a.xt = static_cast<const uint16_t*>(vt);
    a.mask = mask;
    a.scale = scale;
    a.out = o;
    a.out_bf16 = out_bf16;
    a.rows = static_cast<int>(rows);
    a.n = static_cast<int>(n);
    a.d = static_cast<int>(d);
    a.dv = static_cast<int>(dv);
    launch<false>(groups, a, s);
    return hipGetLastError();
}

hipError_t masked_attention_backward(const void* q, const void* k, const void* v, const void* kt, const void* dout,
                                     const float* mask, float scale, void* p, void* ds, float* dmask, void* dq,
                                     bool dq_bf16, int64_t groups, int64_t rows, int64_t n, int64_t d, int64_t dv,
                                     hipStream_t s) {
    MaskedArgs a{};
    a.q = static_cast<const uint16_t*>(q);
    a.k = static_cast<const uint16_t*>(k);
    a.v = static_cast<const uint16_t*>(v);
    a.dout = static_cast<const uint16_t*>(dout);
    a.xt = static_cast<const uint16_t*>(kt);
    a.mask = mask;
    a.scale = scale;
    a.p = static_cast<uint16_t*>(p);
    a.ds = static_cast<uint16_t*>(ds);
    a.dmask = dmask;
    a.out = dq;
    a.out_bf16 = dq_bf16;
    a.rows = static_cast<int>(rows);
    a.n = static_cast<int>(n);
    a.d = static_cast<int>(d);
    a.dv = static_cast<int>(dv);
    launch<true>(groups, a, s);
    return hipGetLastError();
}

size_t packed_bytes(const PackJob& j, int64_t groups, int64_t n) {
    return static_cast<size_t>(groups * n) * (j.transposed ? j.w : (j.w + 31) / 32 * 32) * 2;
}

hipError_t pack_attention_operands(const PackJob* jobs, int count, int64_t groups, int64_t n, hipStream_t s) {
    PackArgs a{};
    int blocks = 0;
    for (int i = 0; i < 3; ++i) {
        if (i < count) {
            a.job[i] = jobs[i];
            blocks += (jobs[i].w + kPackCols - 1) / kPackCols;
        }
        a.last[i] = blocks;
    }
    a.n = static_cast<int>(n);
    hipLaunchKernelGGL(pack_operands, dim3(static_cast<unsigned>(n / 32), static_cast<unsigned>(blocks),
                       static_cast<unsigned>(groups)), dim3(256), 0, s, a);
    return hipGetLastError();
}

}  // namespace hk
