// hk_gemm_mid.hpp — device code of the BF16 GEMM for grids that 256x256 tiles cannot fill (gfx950).
//
// The 256x256 tile kernel (hk_gemm_device.hpp) runs one workgroup per CU; a product with fewer
// such tiles than CUs leaves the chip idle. This kernel covers those: smaller tiles, K split over
// several workgroups when even those are too few, and the same in-place reading of every
// transpose, so no operand is transposed through memory first.
#pragma once

#include <type_traits>

#include "hk_common.hpp"
#include "hk_gemm_device.hpp"

namespace hk {

namespace {

// Output tiles of (16 WM NI) x (16 WN NJ) by four wavefronts in a WM x WN arrangement, each owning
// NI x NJ v_mfma_f32_16x16x32_bf16 tiles. K stages of 64 in a ring of NS LDS slots filled straight
// from global memory; a stage is two k-slices of 32. The mid-stage barrier (all reads of the
// stage's slot done, stage s + 1 landed) frees the slot, which the loads of stage s + NS then fill
// during the stage's second slice, so every load has NS - 1 stages to land.
//
// K-major operands are staged in 128-byte k-rows (16-byte chunk XOR (row / 2) % 8); MN-major ones
// in 64 k-rows of W = BM or BN columns, 64-byte blocks XORed with the k-row (k-row % 4 for rows of
// 256 bytes or more, (k-row / 2) % 2 for 128-byte rows), so that the four k-rows of a 16-lane
// transposing read lie in distinct 64-byte bank groups; read by two ds_read_b64_tr_b16 each.
//
// The last stage may be partial (K % 8 == 0): 16-byte chunks past K take an out-of-range offset and
// k-rows past K lie past the operand, so both read as zero.
//
// What bounds it: at 128x128 the L2 (64 B per CU and clock for the loads of a stage against 512 MFMA
// cycles), below that the length of the K loop per workgroup, and for a few rows against a large
// weight the stream of that weight from HBM, which needs ~100 KB of loads in flight per CU: hence the
// deep rings and two workgroups per CU. Measured (us, back to back on rotating operands, against the
// 32x32x16 kernel with 32-deep stages and transposing passes that this replaced):
//   2000 x 4096 x 4096 NT F32 81 -> 60, NN 109 -> 64;  2000 x 5632 x 2048 NT 63 -> 42;
//   2000 x 2048 x 5632 NN 75 -> 51;  512 x 3072 x 2048 NT 17 -> 13;  2048 x 2048 x 512 TN 30 -> 12;
//   16 x 4096 x 14336 NT 60 -> 24 (4 splits; 5.6 TB/s in the product itself).
//
// K split: workgroup column `split` takes stages [split * per, ...), writing its F32 partial tile
// to plane `split` of the workspace; splitk_reduce adds the planes in order.
struct MidArgs : GemmEpiArgs {
    int splits;           // K splits (1: none)
    int stages_per_split; // K stages of 64 per split
    float* partial;       // [splits][batch][m][n] F32 when splits > 1
};

template <int W>
__device__ __forceinline__ int mn_block_xor(int krow) {
    return W >= 128 ? (krow & 3) : ((krow >> 1) & 1);
}

constexpr int kMidStageElems(int bm, int bn) {  // BF16 per slot: whole 1 KB loads, the same count per wave
    return ((bm + bn) / 8 + 3) / 4 * 4 * 512;
}

template <int WM, int WN, int NI, int NJ, int NS, bool A_MN, bool B_MN, bool OUT_BF16, int EPI, int PER_CU>
__global__ void __launch_bounds__(256, PER_CU)
gemm_mid_kernel(MidArgs p) {
    static_assert(WM * WN == 4, "four waves");
    constexpr int BM = 16 * WM * NI, BN = 16 * WN * NJ;
    static_assert((!A_MN || BM == 64 || BM == 128 || BM == 256) && (!B_MN || BN == 64 || BN == 128 || BN == 256),
                  "MN-major rows of 128, 256 or 512 bytes");
    constexpr int kLoadsA = BM / 8, kLoadsAll = (BM + BN) / 8;  // 1 KB loads per stage
    constexpr int kLoads = (kLoadsAll + 3) / 4;                 // per wave (the last may be a dummy)
    constexpr int kStage = kMidStageElems(BM, BN);
    constexpr int kReads = NI + NJ, kMfma = NI * NJ;
    static_assert((NS - 2) * kLoads < 64, "vmcnt range");
    __shared__ __attribute__((aligned(1024))) uint16_t ring[NS][kStage];

    // XCD-contiguous ranges of (split, tile), bands of 8 tile rows within a split; where the grid is no multiple
    // of 8, only for the two to eight row tiles of one matrix, which in dispatch order lie on different XCDs
    // and each read their column tile of the weight into its own L2 (64 x 8112 x 4096 NT, 254 tiles of 32x64:
    // 36 us, 19 in this order; one row tile, many or a batch lose up to 30% by it: 5 x 704 x 208 x 2032 14, 18).
    const int tiles = p.tiles_m * p.tiles_n, all = tiles * p.splits;
    int bid = blockIdx.x;
    if ((all & 7) == 0) bid = (bid & 7) * (all >> 3) + (bid >> 3);
    else if (p.tiles_m > 1 && p.tiles_m <= 8 && gridDim.z == 1) bid = xcd_logical();
    const int split = bid / tiles;
    bid -= split * tiles;
    constexpr int GROUP = 8;
    const int per_group = GROUP * p.tiles_n;
    const int first_m = (bid / per_group) * GROUP;
    const int gsize = min(p.tiles_m - first_m, GROUP);
    const int tm = first_m + (bid % per_group) % gsize;
    const int tn = (bid % per_group) / gsize;
    const int64_t g = blockIdx.z;
    const uint16_t* A = p.a + g * static_cast<int64_t>(p.m) * p.k;
    const uint16_t* B = weight_slice(p, tm * BM, g);
    const int s_first = split * p.stages_per_split;
    const int nk = min((p.k + kPK - 1) / kPK - s_first, p.stages_per_split);

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wm = wave / WN, wn = wave % WN;
    const int l16 = lane & 15, lg = lane >> 4;

    const i32x4_t ra = buffer_resource(A, p.m * p.k * 2);
    const i32x4_t rb = buffer_resource(B, p.n * p.k * 2);
    // K-major load q of a stage fills rows 8 q .. 8 q + 7 of A (q < BM / 8) or B; q % 2 = wave % 2
    const int r_in = lane >> 3;
    const int src_chunk = (lane & 7) ^ ((4 * (wave & 1) + (r_in >> 1)) & 7);
    const int voff = (r_in * p.k + src_chunk * 8) * 2;
    // MN-major load q fills 512 / W k-rows; lane l takes 16-byte position l % (W / 8) of k-row l / (W / 8)
    auto mn_off = [&](int q, int kt, int cols, int col0, auto w) __attribute__((always_inline)) {
        constexpr int W = decltype(w)::value;
        constexpr int kPos = W / 8;  // 16-byte positions per k-row
        const int krow = q * (512 / W) + lane / kPos, pos = lane % kPos;
        const int c = (((pos >> 2) ^ mn_block_xor<W>(krow)) << 2) | (pos & 3);
        return ((kt * kPK + krow) * cols + col0 + c * 8) * 2;
    };
    auto dload = [&](uint32_t slot, int kt, int d) __attribute__((always_inline)) {
        const int q = wave + 4 * d;  // wave-uniform
        const uint32_t dst = slot + q * 1024;
        if (4 * d + 3 < kLoadsA || (4 * d < kLoadsA && q < kLoadsA)) {
            if constexpr (A_MN)
                load_lds16(ra, dst, mn_off(q, kt, p.m, tm * BM, std::integral_constant<int, BM>{}), 0);
            else
                load_lds16(ra, dst,
                           kt * kPK + src_chunk * 8 < p.k ? voff + (tm * BM + 8 * q) * p.k * 2 + kt * kPK * 2 : kOutOfRange, 0);
        } else {
            const int qb = q - kLoadsA;
            const bool real = 4 * d + 3 < kLoadsAll || q < kLoadsAll;
            if constexpr (B_MN)
                load_lds16(rb, dst, real ? mn_off(qb, kt, p.n, tn * BN, std::integral_constant<int, BN>{}) : kOutOfRange, 0);
            else
                load_lds16(rb, dst,
                           real && kt * kPK + src_chunk * 8 < p.k ? voff + (tn * BN + 8 * qb) * p.k * 2 + kt * kPK * 2
                                                                  : kOutOfRange, 0);
        }
    };

    const int tr_i = lane & 15;
    auto read_tr = [&](const uint16_t* stage, int k0, int col0, auto w) __attribute__((always_inline)) {
        constexpr int W = decltype(w)::value;
        // k0 % 8 == 0, so the XOR term of k-row k0 + i / 4 (and of the row 4 further) is that of i / 4
        const int kr = tr_i >> 2;
        const uint16_t* at = stage + (k0 + kr) * W + ((((col0 >> 5) ^ mn_block_xor<W>(kr)) << 5) | (col0 & 31)) + 4 * (tr_i & 3);
        const v4i16_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4i16_t*)(at));
        const v4i16_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4i16_t*)(at + 4 * W));
        typedef short v8i16_t __attribute__((ext_vector_type(8)));
        const v8i16_t v = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
        return __builtin_bit_cast(bf16x8_t, v);
    };
    bf16x8_t fa[2][NI], fb[2][NJ];
    auto read1 = [&](const uint16_t* slot, int ks, int buf, int f) __attribute__((always_inline)) {
        const int c = 4 * ks + lg;
        if (f < NI) {
            if constexpr (A_MN) fa[buf][f] = read_tr(slot, 8 * c, 16 * (NI * wm + f), std::integral_constant<int, BM>{});
            else fa[buf][f] = *reinterpret_cast<const bf16x8_t*>(slot + swz64(16 * (NI * wm + f) + l16, c));
        } else {
            if constexpr (B_MN)
                fb[buf][f - NI] = read_tr(slot + BM * kPK, 8 * c, 16 * (NJ * wn + f - NI), std::integral_constant<int, BN>{});
            else
                fb[buf][f - NI] = *reinterpret_cast<const bf16x8_t*>(slot + BM * kPK + swz64(16 * (NJ * wn + f - NI) + l16, c));
        }
    };

    f32x4_t acc[NI][NJ];
#pragma unroll
    for (int i = 0; i < NI; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j) acc[i][j] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};

    // The MFMAs of one slice (fragments in buffer `cur`) with the reads of the next slice's fragments
    // and, with LOADS, a stage's loads spread evenly between them.
    auto slice = [&](int cur, const uint16_t* next_slot, int next_ks, bool loads, uint32_t load_slot, int kt) __attribute__((always_inline)) {
#pragma unroll
        for (int e = 0; e < kMfma; ++e) {
            const int i = e / NJ, j = e % NJ;
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fb[cur][j], fa[cur][i], acc[i][j], 0, 0, 0);
            phase_fence();
#pragma unroll
            for (int f = e * kReads / kMfma; f < (e + 1) * kReads / kMfma; ++f) read1(next_slot, next_ks, cur ^ 1, f);
            if (loads) {
#pragma unroll
                for (int d = e * kLoads / kMfma; d < (e + 1) * kLoads / kMfma; ++d) dload(load_slot, kt, d);
            }
            phase_fence();
        }
    };

    // Past the last stage the loads repeat it into slots that are no longer read, so every stage
    // issues the same number and the wait counts hold.
    const int last = s_first + nk - 1;
#pragma unroll
    for (int u = 0; u < NS; ++u)
#pragma unroll
        for (int d = 0; d < kLoads; ++d) dload(lds_address(ring[u]), min(s_first + u, last), d);
    stage_barrier<(NS - 1) * kLoads>();
#pragma unroll
    for (int f = 0; f < kReads; ++f) read1(ring[0], 0, 0, f);

    int s = 0;
    do {  // nk >= 1
#pragma unroll
        for (int u = 0; u < NS; ++u) {
            if (u == 0 || s + u < nk) {
                slice(0, ring[u], 1, false, 0, 0);
                stage_barrier<(NS - 2) * kLoads>();  // stage s + u + 1 landed; every read of slot u done
                slice(1, ring[(u + 1) % NS], 0, true, lds_address(ring[u]), min(s_first + s + u + NS, last));
            }
        }
        s += NS;
    } while (s < nk);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // no load may still be writing LDS at exit

    const int m0 = tm * BM + 16 * NI * wm + l16, n0 = tn * BN + 16 * NJ * wn;
    if constexpr (EPI == kEpiQkvRope) {
        static_assert(NJ == 8 && OUT_BF16, "the fused QKV epilogue needs 128-column wave blocks");
        store_qkv_rope<NI>(p, acc, m0, n0, lg);
        return;
    } else if constexpr (EPI != kEpiPlain) {
        constexpr int kAhead = epi_reads<EPI>() ? (NI < 4 ? NI : 4) : 1;
        EpiRowIn<EPI, NJ> in[kAhead];
        if constexpr (epi_reads<EPI>()) {
#pragma unroll
            for (int i = 0; i < kAhead; ++i) load_fused_row<EPI, NJ>(p, in[i], g, m0 + 16 * i, n0, lg);
        }
#pragma unroll
        for (int i = 0; i < NI; ++i) {
            if (m0 + 16 * i < p.m) store_fused_row<EPI, NJ>(p, acc[i], in[i % kAhead], g, m0 + 16 * i, n0, lg);
            if constexpr (epi_reads<EPI>()) {
                if (i + kAhead < NI) load_fused_row<EPI, NJ>(p, in[i % kAhead], g, m0 + 16 * (i + kAhead), n0, lg);
            }
        }
        return;
    }
    if constexpr (!OUT_BF16) {
        if (p.crop_n != 0) {  // never split
#pragma unroll
            for (int i = 0; i < NI; ++i)
#pragma unroll
                for (int j = 0; j < NJ; ++j) store_cropped(p, g, m0 + 16 * i, n0 + 16 * j + 4 * lg, acc[i][j]);
            return;
        }
    }
    // partial planes: [split][batch][m][n] F32
    const int64_t plane = p.splits > 1 ? static_cast<int64_t>(split) * gridDim.z + g : g;
#pragma unroll
    for (int i = 0; i < NI; ++i) {
        const int m = m0 + 16 * i;
        if (m >= p.m) continue;
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
            const int n = n0 + 16 * j + 4 * lg;
            if (n >= p.n) continue;
            const int64_t off = (plane * p.m + m) * static_cast<int64_t>(p.n) + n;
            if constexpr (OUT_BF16) {
                u32x2_t w = {pack_bf16x2(acc[i][j][0], acc[i][j][1]), pack_bf16x2(acc[i][j][2], acc[i][j][3])};
                *reinterpret_cast<u32x2_t*>(static_cast<uint16_t*>(p.c) + off) = w;
            } else {
                *reinterpret_cast<f32x4_t*>((p.splits > 1 ? p.partial : out_f32(p, p.g_split != 0 ? static_cast<int>(g) : m)) + off) = acc[i][j];
            }
        }
    }
}

// out = sum over the splits, in order, of the F32 partial planes [splits][total] (total % 4 == 0).
template <bool OUT_BF16>
__global__ void __launch_bounds__(256)
splitk_reduce(const float* __restrict__ partial, void* __restrict__ out, int splits, int64_t total) {
    for (int64_t i = flat_begin(256); i < total / 4; i += flat_stride(256)) {
        f32x4_t sum = *reinterpret_cast<const f32x4_t*>(partial + 4 * i);
        for (int s = 1; s < splits; ++s) {
            const f32x4_t v = *reinterpret_cast<const f32x4_t*>(partial + s * total + 4 * i);
#pragma unroll
            for (int e = 0; e < 4; ++e) sum[e] += v[e];
        }
        if constexpr (OUT_BF16)
            reinterpret_cast<u32x2_t*>(out)[i] = u32x2_t{pack_bf16x2(sum[0], sum[1]), pack_bf16x2(sum[2], sum[3])};
        else
            reinterpret_cast<f32x4_t*>(out)[i] = sum;
    }
}

}  // namespace

}  // namespace hk
