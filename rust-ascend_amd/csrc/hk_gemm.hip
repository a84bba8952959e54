// hk_gemm.hip — BF16 GEMM with FP32 accumulation for gfx950 (MI355X).
//
// Semantics (reference rust-ascend-kernels/src/kernel.rs:5-76, ascend.rs:22-68):
//   C[g, i, j] = sum_k A'[g, i, k] * B'[g, k, j]  with FP32 accumulation,
//   C stored as BF16 (round to nearest even) or F32. A' is A ([M,K]) or A^T (A stored
//   [K,M]); B' is B ([K,N]) or B^T (B stored [N,K]). Batched operands are contiguous
//   [G, ...] with strides M*K, N*K, M*N (ascend.rs:88-114).
//
// Design (MI355X-first, not a translation of the reference's 64x64 Ascend tiles):
//   * Large problems (at least one 256x256 tile per CU, K % 64 == 0), every transpose read in
//     place -> gemm_nt_m16_kernel: four wavefronts of 128x128 with 16x16x32 MFMAs and
//     global->LDS loads; a K-contiguous operand (A [M,K], B [N,K]) is staged in 128-byte k-rows
//     and read with 16-byte LDS reads, an MN-contiguous one (A stored [K,M] or B stored [K,N]) in
//     512-byte rows of 256 columns and read with transposing LDS reads.
//   * Smaller problems -> gemm_mid_kernel (hk_gemm_mid.hpp): tiles from 256x128 down to 32x64 with
//     the same MFMAs, in-place transposes and global->LDS loads, K split over workgroups where
//     even those tiles are too few; pick_gemm estimates each shape's time per tile and split.
//   * Operands past 32-bit byte offsets or off 16-byte alignment -> gemm_nt_kernel: MN-contiguous
//     operands are first transposed into the workspace, then four wavefronts (2x2) compute a
//     BMxBN output tile (256, 128 or 64) of v_mfma_f32_32x32x16_bf16.
//   * gemm_nt_kernel's K loop in steps of BK = 64: A and B slices are prefetched from HBM into registers one
//     step ahead, written to a double-buffered LDS tile (rows of 64 BF16 = 128 B, 16-byte
//     chunks XOR-swizzled by row%8 so both the row-contiguous writes and the 32-row
//     fragment reads are bank-conflict-free), one barrier per step.
//   * MFMA operand order is swapped (B tile as the MFMA "A" operand) so each lane ends with
//     4 consecutive output columns per register group: 8-byte BF16 / 16-byte F32 stores.
//   * Tile order: blocks are remapped so each of the 8 XCDs (blockIdx % 8) receives a
//     contiguous range of tiles, then grouped in 8-tile-row bands, so tiles that share A/B
//     slices run on the same XCD's L2.
#include "hk_common.hpp"
#include "hk_gemm_device.hpp"
#include "hk_gemm_mid.hpp"
#include "hk_kernels.hpp"

namespace hk {

namespace {

constexpr int kBK = 64;
constexpr int kThreads = 256;

__device__ __forceinline__ int swz(int row, int chunk) { return row * kBK + ((chunk ^ (row & 7)) << 3); }

template <int BM, int BN, bool OUT_BF16>
__global__ void __launch_bounds__(kThreads)
gemm_nt_kernel(GemmArgs p) {
    constexpr int TI = BM / 64;          // 32x32 tiles per wave along M
    constexpr int TJ = BN / 64;          // along N
    constexpr int A_LOADS = BM * 8 / kThreads;  // 16-byte chunks per thread per K step
    constexpr int B_LOADS = BN * 8 / kThreads;
    __shared__ __attribute__((aligned(16))) uint16_t lds[2][(BM + BN) * kBK];

    // ---- tile coordinates: XCD-contiguous ranges, then 8-row grouped order
    const int tiles = p.tiles_m * p.tiles_n;
    int bid = blockIdx.x;
    if ((tiles & 7) == 0) bid = (bid & 7) * (tiles >> 3) + (bid >> 3);
    constexpr int GROUP = 8;
    const int per_group = GROUP * p.tiles_n;
    const int first_m = (bid / per_group) * GROUP;
    const int gsize = min(p.tiles_m - first_m, GROUP);
    const int tm = first_m + (bid % per_group) % gsize;
    const int tn = (bid % per_group) / gsize;
    const int64_t g = blockIdx.z;

    const uint16_t* A = p.a + g * static_cast<int64_t>(p.m) * p.k;
    const uint16_t* B = weight_slice(p, tm * BM, g);

    const int t = threadIdx.x;
    const int lane = t & 63;
    const int wave = t >> 6;
    const int wm = wave >> 1, wn = wave & 1;
    const int lr = lane & 31, lk = lane >> 5;

    // ---- global -> register prefetch assignment
    const int lcol = t & 7;   // 16-byte chunk within the 64-wide K slice
    const int lrow = t >> 3;  // 0..31, plus 32*i
    const uint16_t* a_src[A_LOADS];
    const uint16_t* b_src[B_LOADS];
#pragma unroll
    for (int i = 0; i < A_LOADS; ++i) {
        int r = tm * BM + lrow + 32 * i;
        r = r < p.m ? r : p.m - 1;  // rows past M read a valid row; their outputs are not stored
        a_src[i] = A + static_cast<int64_t>(r) * p.k + lcol * 8;
    }
#pragma unroll
    for (int i = 0; i < B_LOADS; ++i) {
        int r = tn * BN + lrow + 32 * i;
        r = r < p.n ? r : p.n - 1;
        b_src[i] = B + static_cast<int64_t>(r) * p.k + lcol * 8;
    }
    u32x4_t ra[A_LOADS], rb[B_LOADS];
    auto load_global = [&](int kt) {
        const int kk = kt * kBK + lcol * 8;
        const bool in = kk < p.k;  // K % 16 == 0: a 16-byte chunk is wholly in or out
#pragma unroll
        for (int i = 0; i < A_LOADS; ++i)
            ra[i] = in ? *reinterpret_cast<const u32x4_t*>(a_src[i] + kt * kBK) : u32x4_t{0, 0, 0, 0};
#pragma unroll
        for (int i = 0; i < B_LOADS; ++i)
            rb[i] = in ? *reinterpret_cast<const u32x4_t*>(b_src[i] + kt * kBK) : u32x4_t{0, 0, 0, 0};
    };
    auto store_lds = [&](int buf) {
        uint16_t* la = lds[buf];
        uint16_t* lb = lds[buf] + BM * kBK;
#pragma unroll
        for (int i = 0; i < A_LOADS; ++i)
            *reinterpret_cast<u32x4_t*>(la + swz(lrow + 32 * i, lcol)) = ra[i];
#pragma unroll
        for (int i = 0; i < B_LOADS; ++i)
            *reinterpret_cast<u32x4_t*>(lb + swz(lrow + 32 * i, lcol)) = rb[i];
    };

    f32x16_t acc[TI][TJ];
#pragma unroll
    for (int i = 0; i < TI; ++i)
#pragma unroll
        for (int j = 0; j < TJ; ++j)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.0f;

    const int nk = (p.k + kBK - 1) / kBK;
    load_global(0);
    store_lds(0);
    if (nk > 1) load_global(1);
    __syncthreads();

    for (int kt = 0; kt < nk; ++kt) {
        const int cur = kt & 1;
        const uint16_t* la = lds[cur];
        const uint16_t* lb = lds[cur] + BM * kBK;
#pragma unroll
        for (int ks = 0; ks < kBK / 16; ++ks) {
            const int chunk = ks * 2 + lk;
            bf16x8_t af[TI], bfr[TJ];
#pragma unroll
            for (int i = 0; i < TI; ++i)
                af[i] = *reinterpret_cast<const bf16x8_t*>(la + swz(wm * (BM / 2) + i * 32 + lr, chunk));
#pragma unroll
            for (int j = 0; j < TJ; ++j)
                bfr[j] = *reinterpret_cast<const bf16x8_t*>(lb + swz(wn * (BN / 2) + j * 32 + lr, chunk));
#pragma unroll
            for (int i = 0; i < TI; ++i)
#pragma unroll
                for (int j = 0; j < TJ; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(bfr[j], af[i], acc[i][j], 0, 0, 0);
        }
        if (kt + 1 < nk) {
            store_lds(cur ^ 1);
            if (kt + 2 < nk) load_global(kt + 2);
        }
        __syncthreads();
    }

    // ---- epilogue: lane holds C[m = .. + lr][n = .. + 8*grp + 4*lk + 0..3]
#pragma unroll
    for (int i = 0; i < TI; ++i) {
        const int m = tm * BM + wm * (BM / 2) + i * 32 + lr;
        if (m >= p.m) continue;
#pragma unroll
        for (int j = 0; j < TJ; ++j) {
#pragma unroll
            for (int grp = 0; grp < 4; ++grp) {
                const int n = tn * BN + wn * (BN / 2) + j * 32 + grp * 8 + lk * 4;
                if (n >= p.n) continue;
                const int64_t off = (g * p.m + m) * static_cast<int64_t>(p.n) + n;
                if constexpr (OUT_BF16) {
                    u32x2_t w = {pack_bf16x2(acc[i][j][grp * 4 + 0], acc[i][j][grp * 4 + 1]),
                                 pack_bf16x2(acc[i][j][grp * 4 + 2], acc[i][j][grp * 4 + 3])};
                    *reinterpret_cast<u32x2_t*>(static_cast<uint16_t*>(p.c) + off) = w;
                } else {
                    f32x4_t w = {acc[i][j][grp * 4 + 0], acc[i][j][grp * 4 + 1], acc[i][j][grp * 4 + 2],
                                 acc[i][j][grp * 4 + 3]};
                    *reinterpret_cast<f32x4_t*>(static_cast<float*>(p.c) + off) = w;
                }
            }
        }
    }
}

// out[g][c][r] = in[g][r][c] for BF16, 64x64 tiles through LDS (padded rows).
__global__ void __launch_bounds__(256)
transpose_bf16(const uint16_t* __restrict__ in, uint16_t* __restrict__ out, int64_t rows, int64_t cols) {
    __shared__ uint16_t tile[64][66];
    const int64_t g = blockIdx.z;
    const int64_t r0 = static_cast<int64_t>(blockIdx.y) * 64, c0 = static_cast<int64_t>(blockIdx.x) * 64;
    const uint16_t* src = in + g * rows * cols;
    uint16_t* dst = out + g * rows * cols;
    const int tx = threadIdx.x & 63, ty = threadIdx.x >> 6;
    for (int i = ty; i < 64; i += 4) {
        const int64_t r = r0 + i, c = c0 + tx;
        if (r < rows && c < cols) tile[i][tx] = src[r * cols + c];
    }
    __syncthreads();
    for (int i = ty; i < 64; i += 4) {
        const int64_t c = c0 + i, r = r0 + tx;
        if (r < rows && c < cols) dst[c * rows + r] = tile[tx][i];
    }
}

// Output tile width: 256 (NJ = 8) or 192 (NJ = 6) for a grid of `batch` x M/256 x N/(32 NJ) tiles
// on num_cus CUs, whichever takes fewer rounds of workgroups times the time of one tile. Measured
// on MI355X with each width forced: a part-empty last round costs nearly a full one, and a narrow
// tile takes ~1.1-1.15x the square tile's time per flop, so a round costs 80 (square) or 69
// (192-wide): narrow tiles are taken only when they save a whole round. C3's shapes fill whole
// rounds of square tiles and stay square; C5's 4096 x 6144 QKV projection (384 square tiles, 1.5
// rounds) runs 512 narrow tiles in 2 rounds (alone 168 -> 151 us; 180 -> 175 us inside the layer).
// 224-wide tiles (NJ = 7) for the 896-tile 4096 x 14336 outputs gained 1-4% alone and nothing
// inside the layer, so they are not built.
int pick_tile_nj(int64_t batch, int64_t m, int64_t n, int num_cus) {
    const int64_t tiles_m = (m + kPPTile - 1) / kPPTile;
    auto cost = [&](int nj, int per_round) {
        const int64_t tiles = tiles_m * ((n + 32 * nj - 1) / (32 * nj)) * batch;
        return (tiles + num_cus - 1) / num_cus * per_round;
    };
    return cost(6, 69) < cost(8, 80) ? 6 : 8;
}

template <bool OUT_BF16, int NJ>
void launch_pp_nj(const GemmArgs& p, const dim3& grid, bool a_mn, bool b_mn, hipStream_t s) {
    if (a_mn && b_mn) hipLaunchKernelGGL((gemm_nt_m16_kernel<OUT_BF16, true, true, false, NJ>), grid, dim3(kW4Threads), 0, s, p);
    else if (a_mn) hipLaunchKernelGGL((gemm_nt_m16_kernel<OUT_BF16, true, false, false, NJ>), grid, dim3(kW4Threads), 0, s, p);
    else if (b_mn) hipLaunchKernelGGL((gemm_nt_m16_kernel<OUT_BF16, false, true, false, NJ>), grid, dim3(kW4Threads), 0, s, p);
    else hipLaunchKernelGGL((gemm_nt_m16_kernel<OUT_BF16, false, false, false, NJ>), grid, dim3(kW4Threads), 0, s, p);
}

// nj: 8, or 6 for 192-wide tiles (whole K stages only: the KTAIL variants are square).
template <bool OUT_BF16>
void launch_pp(const GemmArgs& a, int64_t batch, bool a_mn, bool b_mn, int nj, hipStream_t s) {
    GemmArgs p = a;
    p.tiles_m = (p.m + kPPTile - 1) / kPPTile;
    p.tiles_n = (p.n + 32 * nj - 1) / (32 * nj);
    const dim3 grid(static_cast<unsigned>(p.tiles_m * p.tiles_n), 1, static_cast<unsigned>(batch));
    // Square tile grids run bands of 4 M-tile rows per XCD; other grids bands of 8 N-tile
    // columns, so an XCD's L2 holds a narrow slice of B (Llama projections 8192x4096->14336
    // and 8192x14336->4096: 1.40 -> 1.49 and 1.38 -> 1.47 PFLOP/s; 8192^3 keeps 1.54 with
    // M bands vs 1.50 with N bands).
    p.band_n = p.tiles_m == p.tiles_n ? 0 : 8;
    if (p.k % kPK != 0) {
        if (a_mn && b_mn) hipLaunchKernelGGL((gemm_nt_m16_kernel<OUT_BF16, true, true, true>), grid, dim3(kW4Threads), 0, s, p);
        else if (a_mn) hipLaunchKernelGGL((gemm_nt_m16_kernel<OUT_BF16, true, false, true>), grid, dim3(kW4Threads), 0, s, p);
        else if (b_mn) hipLaunchKernelGGL((gemm_nt_m16_kernel<OUT_BF16, false, true, true>), grid, dim3(kW4Threads), 0, s, p);
        else hipLaunchKernelGGL((gemm_nt_m16_kernel<OUT_BF16, false, false, true>), grid, dim3(kW4Threads), 0, s, p);
        return;
    }
    if (nj == 6) launch_pp_nj<OUT_BF16, 6>(p, grid, a_mn, b_mn, s);
    else launch_pp_nj<OUT_BF16, 8>(p, grid, a_mn, b_mn, s);
}

template <int BM, int BN>
void launch_nt(const GemmArgs& a, int64_t batch, bool out_bf16, hipStream_t s) {
    GemmArgs p = a;
    p.tiles_m = (p.m + BM - 1) / BM;
    p.tiles_n = (p.n + BN - 1) / BN;
    const dim3 grid(static_cast<unsigned>(p.tiles_m * p.tiles_n), 1, static_cast<unsigned>(batch));
    if (out_bf16) hipLaunchKernelGGL((gemm_nt_kernel<BM, BN, true>), grid, dim3(kThreads), 0, s, p);
    else hipLaunchKernelGGL((gemm_nt_kernel<BM, BN, false>), grid, dim3(kThreads), 0, s, p);
}

// Output tile of 256, 128 or 64: the largest whose grid still fills the CUs.
void launch_nt_sized(const GemmArgs& p, int64_t batch, bool out_bf16, int num_cus, hipStream_t s) {
    const int64_t m = p.m, n = p.n;
    const int64_t t256 = ((m + 255) / 256) * ((n + 255) / 256) * batch;
    const int64_t t128 = ((m + 127) / 128) * ((n + 127) / 128) * batch;
    if (t256 >= num_cus) launch_nt<256, 256>(p, batch, out_bf16, s);
    else if (t128 >= num_cus) launch_nt<128, 128>(p, batch, out_bf16, s);
    else launch_nt<64, 64>(p, batch, out_bf16, s);
}

// The tile shapes a product may run on. `per_cu` workgroups share a CU; a stage of 64 k costs `k1` us
// and a tile's start and end `t1` us with one workgroup on the CU, `k2` and `t2` (per pair) with two;
// each further round of a single-workgroup shape costs t2 besides its stages. The figures are a
// least-squares fit on MI355X to measured (shape, tile, split) times over 120 shapes (M 16-5600,
// N 64-14000, K 64-14000, batches 1-32, every transpose). The choice they lead to is on average
// 3.3% slower than the best measured one (40% at worst); the rule it replaces (the largest of 256, 128
// and 64 whose grid fills the CUs, after a transposing pass) was on average 113% slower.
enum GemmTile { kT256, kT256x192, kT256x128, kT128, kT128Pair, kT64x128, kT128x64, kT64, kT32x64, kTiles };
struct TileCost {
    int bm, bn, per_cu, slots;  // slots: K stages in the LDS ring
    float k1, t1, k2, t2;
};
constexpr TileCost kTileCost[kTiles] = {
    {256, 256, 1, 2, 1.232f, 6.44f, 0.0f, 1.08f},  {256, 192, 1, 2, 0.922f, 5.32f, 0.0f, 8.67f},
    {256, 128, 1, 3, 0.715f, 3.72f, 0.0f, 3.67f},  {128, 128, 1, 4, 0.447f, 2.96f, 0.0f, 3.72f},
    {128, 128, 2, 2, 0.658f, 1.88f, 0.915f, 3.42f}, {64, 128, 2, 3, 0.314f, 1.44f, 0.625f, 3.12f},
    {128, 64, 2, 3, 0.279f, 1.63f, 0.644f, 2.74f},  {64, 64, 2, 4, 0.191f, 1.02f, 0.421f, 2.21f},
    {32, 64, 2, 6, 0.142f, 0.94f, 0.393f, 1.55f},
};

struct GemmChoice {
    int tile = kT64;
    int splits = 1;
    float us = 0.0f;
};

// Estimated time (us) of the product on one tile shape with K cut into `splits`.
float tile_time(const TileCost& t, int64_t batch, int64_t m, int64_t n, int64_t k, bool out_bf16, int splits,
                int num_cus) {
    const int64_t nk = (k + kPK - 1) / kPK, per = (nk + splits - 1) / splits;
    const int64_t wgs = ((m + t.bm - 1) / t.bm) * ((n + t.bn - 1) / t.bn) * batch * splits;
    const int64_t rounds = (wgs + num_cus - 1) / num_cus;
    float us = t.per_cu == 1 ? rounds * per * t.k1 + t.t1 + (rounds - 1) * t.t2
                             : (rounds / 2) * (per * t.k2 + t.t2) + (rounds % 2) * (per * t.k1 + t.t1);
    const float out = static_cast<float>(batch) * m * n;
    const float bytes = static_cast<float>(batch) * (m + n) * k * 2 + out * (splits > 1 ? 4 * splits : out_bf16 ? 2 : 4);
    us = fmaxf(us, bytes * (bytes > 64e6f ? 1.8e-7f : 2.8e-7f));  // 5.5 TB/s; short streams reach 3.5
    if (bytes > 64e6f) {
        // operands past the caches arrive at the rate that the loads in flight allow over a round trip
        // of 2.5 us (16 x 6336 x 12208: 99 workgroups 55 us, 198 36 us)
        const int64_t resident = wgs < num_cus * t.per_cu ? wgs : num_cus * t.per_cu;
        us = fmaxf(us, bytes * 2.5f / (static_cast<float>(resident) * (t.slots - 1) * (t.bm + t.bn) * (2 * kPK)));
    }
    if (splits > 1) us += 1.9f + out * 4 * (splits + 0.5f) * 2.4e-7f;  // the reducing launch, the planes
    return us;
}

constexpr int64_t kMaxSplitBytes = int64_t{64} << 20;  // F32 partial planes of a K split

// An operand slice (K rounded up to a stage) below 2^31 bytes, and unsigned 32-bit offsets up to the
// end of its last 256-row tile.
bool fits_32bit(int64_t rows, int64_t k) {
    const int64_t k64 = (k + kPK - 1) / kPK * kPK;
    return rows * k64 * 2 < (int64_t{1} << 31) && (rows + 255) / 256 * 256 * k64 * 2 < (int64_t{1} << 32);
}
// The kernels that read every transpose in place (buffer loads of 16 bytes): K % 8 == 0 and 16-byte
// aligned operands. Callers' M and N are multiples of 16, so MN-major rows are aligned too.
bool in_place_applies(int64_t m, int64_t n, int64_t k, bool aligned) {
    return aligned && k > 0 && k % 8 == 0 && fits_32bit(m, k) && fits_32bit(n, k);
}

// The tile shape and K split of least estimated time whose partial planes fit ws_bytes. An MN-major
// A needs tiles of at least 64 rows; 192-wide tiles take whole K stages.
GemmChoice pick_gemm(int64_t batch, int64_t m, int64_t n, int64_t k, bool a_mn, bool out_bf16, size_t ws_bytes,
                     int num_cus) {
    GemmChoice best;
    best.us = INFINITY;
    const int64_t nk = (k + kPK - 1) / kPK;
    for (int t = 0; t < kTiles; ++t) {
        const TileCost& c = kTileCost[t];
        if ((a_mn && c.bm < 64) || (t == kT256x192 && k % kPK != 0)) continue;
        const int64_t tiles = ((m + c.bm - 1) / c.bm) * ((n + c.bn - 1) / c.bn) * batch;
        for (int splits : {1, 2, 3, 4, 6, 8, 12, 16}) {
            // K is split only where the tiles leave CUs idle, into at least two stages each
            const int64_t planes = batch * m * n * 4 * splits;
            if (splits > 1 && (t <= kT256x192 || tiles >= 2 * num_cus || tiles * splits > 4 * num_cus ||
                               nk < 2 * splits || planes > kMaxSplitBytes || static_cast<size_t>(planes) > ws_bytes))
                break;
            const float us = tile_time(c, batch, m, n, k, out_bf16, splits, num_cus);
            if (us < best.us) best = GemmChoice{t, splits, us};
        }
    }
    return best;
}

// The choice for a product: full grids of 256x256 tiles (at least one per CU, at most a fifth of
// them past the output's edges) keep the 256-wide kernels; the rest take pick_gemm's.
GemmChoice choose_gemm(int64_t batch, int64_t m, int64_t n, int64_t k, bool a_mn, bool out_bf16, size_t ws_bytes,
                       int num_cus) {
    const int64_t tiles = ((m + kPPTile - 1) / kPPTile) * ((n + kPPTile - 1) / kPPTile) * batch;
    if (tiles >= num_cus && 5 * batch * m * n >= 4 * tiles * kPPTile * kPPTile) {
        GemmChoice c;
        c.tile = k % kPK == 0 && pick_tile_nj(batch, m, n, num_cus) == 6 ? kT256x192 : kT256;
        return c;
    }
    // One row tile against a weight past the caches, whose column tiles of 64 alone fill 3/4 of the CUs or more, in one
    // round: its stream is what counts, and a split only adds its planes and a launch. The estimates tie there, with
    // errors either way. 64 x 14336 x 4096: 25.6 us unsplit on rotating weights, 20.0 on one, 29.0 and 24.5 with K
    // in two on 128x128; 32 x 12320 x 11488: 65 and 58 against 72 and 63.
    const int64_t columns = (n + 63) / 64;
    if (batch == 1 && m <= 64 && n * k * 2 > 64000000 && 4 * columns >= 3 * num_cus && columns <= num_cus) {
        GemmChoice c;
        c.tile = m <= 32 && !a_mn ? kT32x64 : kT64;
        c.us = tile_time(kTileCost[c.tile], batch, m, n, k, out_bf16, 1, num_cus);
        return c;
    }
    return pick_gemm(batch, m, n, k, a_mn, out_bf16, ws_bytes, num_cus);
}

template <int WM, int WN, int NI, int NJ, int NS, int PER_CU, bool OUT_BF16>
void launch_mid_as(MidArgs& p, int64_t batch, bool a_mn, bool b_mn, hipStream_t s) {
    constexpr int BM = 16 * WM * NI, BN = 16 * WN * NJ;
    p.tiles_m = (p.m + BM - 1) / BM;
    p.tiles_n = (p.n + BN - 1) / BN;
    const dim3 grid(static_cast<unsigned>(p.tiles_m * p.tiles_n * p.splits), 1, static_cast<unsigned>(batch));
    if constexpr (BM >= 64) {
        if (a_mn && b_mn) {
            hipLaunchKernelGGL((gemm_mid_kernel<WM, WN, NI, NJ, NS, true, true, OUT_BF16, kEpiPlain, PER_CU>), grid,
                               dim3(kThreads), 0, s, p);
            return;
        }
        if (a_mn) {
            hipLaunchKernelGGL((gemm_mid_kernel<WM, WN, NI, NJ, NS, true, false, OUT_BF16, kEpiPlain, PER_CU>), grid,
                               dim3(kThreads), 0, s, p);
            return;
        }
    }
    if (b_mn)
        hipLaunchKernelGGL((gemm_mid_kernel<WM, WN, NI, NJ, NS, false, true, OUT_BF16, kEpiPlain, PER_CU>), grid,
                           dim3(kThreads), 0, s, p);
    else
        hipLaunchKernelGGL((gemm_mid_kernel<WM, WN, NI, NJ, NS, false, false, OUT_BF16, kEpiPlain, PER_CU>), grid,
                           dim3(kThreads), 0, s, p);
}

template <int WM, int WN, int NI, int NJ, int NS, int PER_CU>
void launch_mid(MidArgs& p, int64_t batch, bool out_bf16, bool a_mn, bool b_mn, hipStream_t s) {
    if (out_bf16 && p.splits == 1) launch_mid_as<WM, WN, NI, NJ, NS, PER_CU, true>(p, batch, a_mn, b_mn, s);
    else launch_mid_as<WM, WN, NI, NJ, NS, PER_CU, false>(p, batch, a_mn, b_mn, s);
}

void set_splits(MidArgs& p, int splits) {
    const int nk = (p.k + kPK - 1) / kPK;
    p.stages_per_split = (nk + splits - 1) / splits;
    p.splits = (nk + p.stages_per_split - 1) / p.stages_per_split;  // every split holds a stage
}

void launch_choice(const GemmChoice& c, const GemmArgs& a, int64_t batch, bool out_bf16, bool a_mn, bool b_mn,
                   void* workspace, hipStream_t s) {
    if (c.tile == kT256 || c.tile == kT256x192) {
        const int nj = c.tile == kT256 ? 8 : 6;
        if (out_bf16) launch_pp<true>(a, batch, a_mn, b_mn, nj, s);
        else launch_pp<false>(a, batch, a_mn, b_mn, nj, s);
        return;
    }
    MidArgs p{};
    static_cast<GemmArgs&>(p) = a;
    set_splits(p, c.splits);
    p.partial = static_cast<float*>(workspace);
    switch (c.tile) {
        case kT256x128: launch_mid<2, 2, 8, 4, 3, 1>(p, batch, out_bf16, a_mn, b_mn, s); break;
        case kT128: launch_mid<2, 2, 4, 4, 4, 1>(p, batch, out_bf16, a_mn, b_mn, s); break;
        case kT128Pair: launch_mid<2, 2, 4, 4, 2, 2>(p, batch, out_bf16, a_mn, b_mn, s); break;
        case kT64x128: launch_mid<2, 2, 2, 4, 3, 2>(p, batch, out_bf16, a_mn, b_mn, s); break;
        case kT128x64: launch_mid<2, 2, 4, 2, 3, 2>(p, batch, out_bf16, a_mn, b_mn, s); break;
        case kT64: launch_mid<2, 2, 2, 2, 4, 2>(p, batch, out_bf16, a_mn, b_mn, s); break;
        default: launch_mid<1, 4, 2, 1, 6, 2>(p, batch, out_bf16, a_mn, b_mn, s); break;
    }
    if (p.splits == 1) return;
    const int64_t total = batch * p.m * p.n;
    const dim3 grid(flat_blocks(total / 4, 256));
    if (out_bf16) hipLaunchKernelGGL((splitk_reduce<true>), grid, dim3(256), 0, s, p.partial, p.c, p.splits, total);
    else hipLaunchKernelGGL((splitk_reduce<false>), grid, dim3(256), 0, s, p.partial, p.c, p.splits, total);
}

size_t round256(size_t x) { return (x + 255) & ~size_t(255); }

}  // namespace

Scratch gemm_workspace(int64_t batch, int64_t m, int64_t n, int64_t k, int ta, int tb, bool out_bf16, bool aligned,
                             int num_cus) {
    Scratch w;
    if (in_place_applies(m, n, k, aligned)) {
        const GemmChoice c = choose_gemm(batch, m, n, k, ta != 0, out_bf16, SIZE_MAX, num_cus);
        if (c.splits > 1) w.want = static_cast<size_t>(batch * m * n) * 4 * c.splits;
        return w;
    }
    if (ta) w.need += round256(static_cast<size_t>(batch * m * k) * 2);
    if (!tb) w.need += round256(static_cast<size_t>(batch * n * k) * 2);
    w.want = w.need;
    return w;
}

hipError_t gemm_bf16(const void* a, const void* b, void* c, int out_bf16, int64_t batch, int64_t m, int64_t n,
                     int64_t k, int ta, int tb, void* workspace, size_t ws_bytes, int num_cus, hipStream_t s) {
    GemmArgs p{};
    p.a = static_cast<const uint16_t*>(a);
    p.b = static_cast<const uint16_t*>(b);
    p.c = c;
    p.m = static_cast<int>(m);
    p.n = static_cast<int>(n);
    p.k = static_cast<int>(k);
    if (in_place_applies(m, n, k, aligned16({a, b, c}))) {
        const GemmChoice ch = choose_gemm(batch, m, n, k, ta != 0, out_bf16 != 0, ws_bytes, num_cus);
        launch_choice(ch, p, batch, out_bf16 != 0, ta != 0, tb == 0, workspace, s);
        return hipGetLastError();
    }
    char* ws = static_cast<char*>(workspace);
    if (ta) {  // A stored [K,M] -> [M,K]
        uint16_t* t = reinterpret_cast<uint16_t*>(ws);
        hipLaunchKernelGGL(transpose_bf16, dim3((unsigned)((m + 63) / 64), (unsigned)((k + 63) / 64), (unsigned)batch),
                           dim3(256), 0, s, p.a, t, k, m);
        p.a = t;
        ws += round256(static_cast<size_t>(batch * m * k) * 2);
    }
    if (!tb) {  // B stored [K,N] -> [N,K]
        uint16_t* t = reinterpret_cast<uint16_t*>(ws);
        hipLaunchKernelGGL(transpose_bf16, dim3((unsigned)((n + 63) / 64), (unsigned)((k + 63) / 64), (unsigned)batch),
                           dim3(256), 0, s, p.b, t, k, n);
        p.b = t;
    }
    launch_nt_sized(p, batch, out_bf16 != 0, num_cus, s);
    return hipGetLastError();
}

hipError_t gemm_bf16_two_outputs(const void* a, const void* b, float* c, float* c2, int64_t m_split, int64_t m, int64_t n,
                                 int64_t k, int ta, int tb, int num_cus, hipStream_t s) {
    if (!in_place_applies(m, n, k, aligned16({a, b, c, c2})) || m_split % 16 != 0) return hipErrorInvalidValue;
    GemmArgs p{};
    p.a = static_cast<const uint16_t*>(a);
    p.b = static_cast<const uint16_t*>(b);
    p.c = c;
    p.c2 = reinterpret_cast<void*>(reinterpret_cast<uintptr_t>(c2) - static_cast<uintptr_t>(m_split * n) * sizeof(float));
    p.m_split = static_cast<int>(m_split);
    p.m = static_cast<int>(m);
    p.n = static_cast<int>(n);
    p.k = static_cast<int>(k);
    launch_choice(choose_gemm(1, m, n, k, ta != 0, false, 0, num_cus), p, 1, false, ta != 0, tb == 0, nullptr, s);
    return hipGetLastError();
}

bool gemm_bf16_pair(const void* a, const void* b, float* c, float* c2, int64_t batch, int64_t m, int64_t n, int64_t k,
                    int ta, int tb, int num_cus, hipStream_t s, hipError_t* e) {
    if (!in_place_applies(m, n, k, aligned16({a, b, c, c2}))) return false;
    const GemmChoice ch = choose_gemm(2 * batch, m, n, k, ta != 0, false, 0, num_cus);
    if (ch.tile <= kT256x192) return false;
    GemmArgs p{};
    p.a = static_cast<const uint16_t*>(a);
    p.b = static_cast<const uint16_t*>(b);
    p.c = c;
    p.c2 = reinterpret_cast<void*>(reinterpret_cast<uintptr_t>(c2) - static_cast<uintptr_t>(batch * m * n) * sizeof(float));
    p.m_split = p.g_split = static_cast<int>(batch);
    p.m = static_cast<int>(m);
    p.n = static_cast<int>(n);
    p.k = static_cast<int>(k);
    launch_choice(ch, p, 2 * batch, false, ta != 0, tb == 0, nullptr, s);
    *e = hipGetLastError();
    return true;
}

bool gemm_bf16_cropped(const void* a, const void* b, float* c, int64_t batch, int64_t m, int64_t n, int64_t k, int ta,
                       int tb, int64_t rows, int64_t cols, size_t ws_bytes, int num_cus, hipStream_t s, hipError_t* e) {
    if (!in_place_applies(m, n, k, aligned16({a, b}))) return false;
    const GemmChoice ch = choose_gemm(batch, m, n, k, ta != 0, false, ws_bytes, num_cus);
    if (ch.splits > 1 || ch.tile <= kT256x192) return false;
    GemmArgs p{};
    p.a = static_cast<const uint16_t*>(a);
    p.b = static_cast<const uint16_t*>(b);
    p.c = c;
    p.m = static_cast<int>(m);
    p.n = static_cast<int>(n);
    p.k = static_cast<int>(k);
    p.crop_m = static_cast<int>(rows);
    p.crop_n = static_cast<int>(cols);
    launch_choice(ch, p, batch, false, ta != 0, tb == 0, nullptr, s);
    *e = hipGetLastError();
    return true;
}

int gemm_route(int64_t batch, int64_t m, int64_t n, int64_t k, int ta, bool out_bf16, size_t ws_bytes, int num_cus) {
    if (!in_place_applies(m, n, k, true)) return -1;
    const GemmChoice c = choose_gemm(batch, m, n, k, ta != 0, out_bf16, ws_bytes, num_cus);
    MidArgs p{};
    p.k = static_cast<int>(k);
    set_splits(p, c.splits);
    return c.tile + 256 * p.splits;
}

bool gemm_reads_in_place(int64_t m, int64_t n, int64_t k) { return in_place_applies(m, n, k, true); }

bool epi_applies(int64_t m, int64_t n, int64_t k) {
    const int64_t k64 = (k + kPK - 1) / kPK * kPK;
    return m > 0 && n > 0 && k > 0 && k % 8 == 0 && m * k64 * 2 < (int64_t{1} << 31) &&
           n * k64 * 2 < (int64_t{1} << 31);
}

bool qkv_rope_applies(int64_t tokens, int64_t hidden, int64_t width) {
    return width % 128 == 0 && epi_applies(tokens, width, hidden);
}

namespace {
// The tile of a fused-epilogue product (K is never split: the epilogue needs the whole sum): the
// 256x256 kernel for full grids as choose_gemm has it, else the least estimated time of those built.
// The products of a 512-token layer of hidden 2048 made 16-88 workgroups of 256x256; with these tiles
// its two residual projections take 46 us instead of 187, gate/up 44 (66; 50 on 128x128 pairs), the SwiGLU backward 28 (66)
// and the QKV projection 20 (63).
int pick_epi_tile(int64_t m, int64_t n, int64_t k, std::initializer_list<int> built, int num_cus) {
    const GemmChoice full = choose_gemm(1, m, n, k, false, true, 0, num_cus);
    if (full.us == 0.0f) return kT256;  // a full grid (not estimated)
    int best = kT256;
    float us = tile_time(kTileCost[kT256], 1, m, n, k, true, 1, num_cus);
    for (int t : built) {
        const float e = tile_time(kTileCost[t], 1, m, n, k, true, 1, num_cus);
        if (e < us) us = e, best = t;
    }
    return best;
}

template <int EPI>
int epi_tile(int64_t m, int64_t n, int64_t k, int num_cus) {
    if constexpr (EPI == kEpiQkvRope) return pick_epi_tile(m, n, k, {kT128Pair, kT64x128}, num_cus);
    else return pick_epi_tile(m, n, k, {kT256x128, kT128Pair, kT64x128, kT64}, num_cus);
}

template <int WM, int WN, int NI, int NJ, int NS, int PER_CU, int EPI, bool B_MN>
void launch_epi_mid(const GemmEpiArgs& a, hipStream_t s) {
    MidArgs p{};
    static_cast<GemmEpiArgs&>(p) = a;
    set_splits(p, 1);
    p.tiles_m = (p.m + 16 * WM * NI - 1) / (16 * WM * NI);
    p.tiles_n = (p.n + 16 * WN * NJ - 1) / (16 * WN * NJ);
    const dim3 grid(static_cast<unsigned>(p.tiles_m * p.tiles_n));
    hipLaunchKernelGGL((gemm_mid_kernel<WM, WN, NI, NJ, NS, false, B_MN, true, EPI, PER_CU>), grid, dim3(kThreads), 0, s, p);
}

// A fused-epilogue GEMM over p.m x p.n outputs (256x256 tiles, bands of 8 N-tiles per XCD unless
// the tile grid is square, as launch_pp chooses; smaller tiles below a full grid). The QKV epilogue
// needs a whole 128-column head per wave, so its smaller tiles stack the four waves along M.
template <int EPI, bool B_MN>
hipError_t launch_epi(GemmEpiArgs p, int num_cus, hipStream_t s) {
    if constexpr (EPI == kEpiQkvRope) {
        switch (epi_tile<EPI>(p.m, p.n, p.k, num_cus)) {
            case kT128Pair: launch_epi_mid<4, 1, 2, 8, 2, 2, EPI, B_MN>(p, s); return hipGetLastError();
            case kT64x128: launch_epi_mid<4, 1, 1, 8, 3, 2, EPI, B_MN>(p, s); return hipGetLastError();
            default: break;
        }
    } else {
        switch (epi_tile<EPI>(p.m, p.n, p.k, num_cus)) {
            case kT256x128: launch_epi_mid<2, 2, 8, 4, 3, 1, EPI, B_MN>(p, s); return hipGetLastError();
            case kT128Pair: launch_epi_mid<2, 2, 4, 4, 2, 2, EPI, B_MN>(p, s); return hipGetLastError();
            case kT64x128: launch_epi_mid<2, 2, 2, 4, 3, 2, EPI, B_MN>(p, s); return hipGetLastError();
            case kT64: launch_epi_mid<2, 2, 2, 2, 4, 2, EPI, B_MN>(p, s); return hipGetLastError();
            default: break;
        }
    }
    p.tiles_m = (p.m + kPPTile - 1) / kPPTile;
    p.tiles_n = (p.n + kPPTile - 1) / kPPTile;
    p.band_n = p.tiles_m == p.tiles_n ? 0 : 8;
    const dim3 grid(static_cast<unsigned>(p.tiles_m * p.tiles_n));
    if (p.k % kPK != 0) hipLaunchKernelGGL((gemm_epi_kernel<EPI, B_MN, true>), grid, dim3(kW4Threads), 0, s, p);
    else hipLaunchKernelGGL((gemm_epi_kernel<EPI, B_MN, false>), grid, dim3(kW4Threads), 0, s, p);
    return hipGetLastError();
}

GemmEpiArgs epi_args(const void* a, const void* b, void* c, int64_t m, int64_t n, int64_t k) {
    GemmEpiArgs p{};
    p.a = static_cast<const uint16_t*>(a);
    p.b = static_cast<const uint16_t*>(b);
    p.c = c;
    p.m = static_cast<int>(m);
    p.n = static_cast<int>(n);
    p.k = static_cast<int>(k);
    return p;
}
}  // namespace

int epilogue_route(int64_t m, int64_t n, int64_t k, bool qkv_rope, int num_cus) {
    if (!epi_applies(m, n, k)) return -1;
    return qkv_rope ? epi_tile<kEpiQkvRope>(m, n, k, num_cus) : epi_tile<kEpiResidual>(m, n, k, num_cus);
}

hipError_t gemm_qkv_rope(const void* x, const void* w, int64_t tokens, int64_t hidden, int64_t seq, int64_t hq,
                         int64_t hkv, const float* cos_t, const float* sin_t, int layout, void* q, void* k, void* v,
                         int num_cus, hipStream_t s) {
    GemmEpiArgs p = epi_args(x, w, nullptr, tokens, (hq + 2 * hkv) * 128, hidden);
    p.qkv = QkvRopeOut{static_cast<uint16_t*>(q), static_cast<uint16_t*>(k), static_cast<uint16_t*>(v), cos_t, sin_t,
                       static_cast<int>(seq), static_cast<int>(hq), static_cast<int>(hkv), layout};
    return launch_epi<kEpiQkvRope, false>(p, num_cus, s);
}

hipError_t gemm_residual(const void* x, const void* w, const void* res, void* y, int64_t m, int64_t n, int64_t k,
                         int num_cus, hipStream_t s) {
    GemmEpiArgs p = epi_args(x, w, y, m, n, k);
    p.res = static_cast<const uint16_t*>(res);
    return launch_epi<kEpiResidual, false>(p, num_cus, s);
}

hipError_t gemm_swiglu(const void* x, const void* w_gu, void* gate, void* up, void* act, int64_t m, int64_t f,
                       int64_t k, int num_cus, hipStream_t s) {
    GemmEpiArgs p = epi_args(x, w_gu, nullptr, m, 2 * f, k);
    p.gate = static_cast<uint16_t*>(gate);
    p.up = static_cast<uint16_t*>(up);
    p.act = static_cast<uint16_t*>(act);
    return launch_epi<kEpiSwiglu, false>(p, num_cus, s);
}

hipError_t gemm_swiglu_backward(const void* dy, const void* wd, const void* gate, const void* up, void* dgu, int64_t m,
                                int64_t f, int64_t k, int num_cus, hipStream_t s) {
    GemmEpiArgs p = epi_args(dy, wd, nullptr, m, f, k);
    p.gate = const_cast<uint16_t*>(static_cast<const uint16_t*>(gate));
    p.up = const_cast<uint16_t*>(static_cast<const uint16_t*>(up));
    p.dgu = static_cast<uint16_t*>(dgu);
    return launch_epi<kEpiSwigluBwd, true>(p, num_cus, s);
}

hipError_t gemm_bf16_grouped_nt(const void* a, const void* w, void* c, int out_bf16, int64_t m, int64_t n, int64_t k,
                                const int32_t* block_group, int num_cus, hipStream_t s) {
    GemmArgs p{};
    p.a = static_cast<const uint16_t*>(a);
    p.b = static_cast<const uint16_t*>(w);
    p.c = c;
    p.m = static_cast<int>(m);
    p.n = static_cast<int>(n);
    p.k = static_cast<int>(k);
    p.block_group = block_group;
    if (in_place_applies(m, n, k, aligned16({a, w, c})))
        launch_choice(choose_gemm(1, m, n, k, false, out_bf16 != 0, 0, num_cus), p, 1, out_bf16 != 0, false, false, nullptr, s);
    else
        launch_nt_sized(p, 1, out_bf16 != 0, num_cus, s);
    return hipGetLastError();
}

}  // namespace hk
