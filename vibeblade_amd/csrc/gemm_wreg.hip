// GEMM for 17 to 256 activation rows on the register-decoding tile of
// wreg_core.hpp: Y (M x N) = X W^T, W in Q4_K / Q5_K / Q6_K / Q8_0.
//
// Three launches: X packed in fragment order (rounded to fp16, as every
// batched kernel takes its activations), the products, and with K splits the
// sum of the partial products in a fixed order.  A workgroup multiplies 128
// columns by all the rows, its two K groups of four waves take half of its
// super-blocks each; K is split between workgroups until the CUs are filled
// (one 512-thread workgroup per CU: 160 KB of LDS).
//
// Why: every weight is decoded once, by the wave that owns its column, while
// the tiled kernel decodes it once per 64-128 rows through LDS and the K-split
// kernel once per 16-64 rows.  The weight loads and the decode bound it; see
// the rule in gemm_wreg_shape for both sides.
#include "wreg_core.hpp"
#include "vb_internal.hpp"
#include "../../include/vbhip.h"

namespace vb {
namespace {

using wreg::BUF_U4;

// Grid (blocks of 16 rows, K / 256); rows past M are zeros.  A wave reads 64
// (fp32: 128) contiguous bytes of 16 rows per load and writes 256-byte runs.
template <int XT>
__global__ void __launch_bounds__(256) wreg_pack_kernel(const void* __restrict__ X, int M, int K, int q6,
                                                        uint4* __restrict__ xf) {
    const int blk = static_cast<int>(blockIdx.x), sb = static_cast<int>(blockIdx.y), nsb = K >> 8;
    uint4* dst = xf + (static_cast<int64_t>(blk) * nsb + sb) * 512;
#pragma unroll
    for (int q = 0; q < 2; q++) {
        const int id = static_cast<int>(threadIdx.x) + 256 * q;
        const int row = (id >> 2) & 15, piece = (id & 3) + 4 * (id >> 6);
        uint4 v = make_uint4(0, 0, 0, 0);
        if (16 * blk + row < M) {
            const int64_t at = static_cast<int64_t>(16 * blk + row) * K + 256 * sb + 8 * piece;
            v = x8_f16<XT>(X, at);
        }
        int g, m, e;
        wreg::k_slot(8 * piece, q6 != 0, g, m, e);
        dst[m * 64 + g * 16 + row] = v;
    }
}

template <int TYPE, int MB>
__global__ void __launch_bounds__(512) gemm_wreg_kernel(const uint8_t* __restrict__ w, uint32_t wbytes, uint32_t rb,
                                                        const uint8_t* __restrict__ xf, float* __restrict__ out, int M,
                                                        int N, int nsb, int ntile, int ks, int mt, int bpt) {
    __shared__ u32x4 b0[2 * BUF_U4];
    __shared__ u32x4 b1[2 * BUF_U4];
    // Workgroups go to the eight XCDs round robin; each XCD takes a contiguous
    // eighth of the split-major order, so that it reads the packed rows of one
    // or two K splits only, and the row tiles of a column tile share its weights.
    const int lin = static_cast<int>(blockIdx.x), items = ntile * ks * mt, per = (items + 7) >> 3;
    const int item = (lin & 7) * per + (lin >> 3);
    if ((lin >> 3) >= per || item >= items) return;
    const int z = item / (ntile * mt), rest = item - z * ntile * mt;
    const int col = rest / mt, blk0 = (rest - col * mt) * bpt, n0 = col * 128;
    const int lane = static_cast<int>(threadIdx.x) & 63, j = lane & 15, g = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
    const int wn = wave & 3, kw = wave >> 2;
    // this split's super-blocks, halved between the K groups
    const int s0 = z * nsb / ks, len = (z + 1) * nsb / ks - s0, half = (len + 1) >> 1;
    const int nc = n0 + 32 * wn + j;  // column of fragment 0; fragment 1 is 16 on
    const uint32_t ro0 = static_cast<uint32_t>(nc < N ? nc : N - 1) * rb;
    const uint32_t ro1 = static_cast<uint32_t>(nc + 16 < N ? nc + 16 : N - 1) * rb;
    const int left = ((M + 15) >> 4) - blk0, nblk = left < bpt ? left : bpt;
    const __amdgpu_buffer_rsrc_t ws = make_rsrc(w, wbytes);
    const __amdgpu_buffer_rsrc_t xs = make_rsrc(xf + static_cast<int64_t>(blk0) * nsb * 8192,
                                                static_cast<uint32_t>(nblk * nsb) * 8192u);
    float4_t acc[MB][2];
#pragma unroll
    for (int b = 0; b < MB; b++) acc[b][0] = acc[b][1] = float4_t{0.f, 0.f, 0.f, 0.f};
    wreg::mainloop<TYPE, MB>(acc, ws, ws, ro0, ro1, xs, nblk, nsb, kw ? s0 + half : s0, kw ? len - half : half, half,
                             b0 + kw * BUF_U4, b1 + kw * BUF_U4, wn);
    // K group kw finishes fragment kw: the other group's sums of it come
    // through LDS (group 0's of fragment 1 in b0, group 1's of fragment 0 in b1)
    float4_t* put = reinterpret_cast<float4_t*>(kw ? b1 : b0) + (wn * MB) * 64 + lane;
    const float4_t* get = reinterpret_cast<const float4_t*>(kw ? b0 : b1) + (wn * MB) * 64 + lane;
#pragma unroll
    for (int b = 0; b < MB; b++) put[b * 64] = acc[b][kw ? 0 : 1];
    __syncthreads();
    const int n = nc + 16 * kw;
    if (n >= N) return;
    float* o = out + static_cast<int64_t>(z) * M * N + n;
#pragma unroll
    for (int b = 0; b < MB; b++) {
        const float4_t mine = acc[b][kw ? 1 : 0], oth = get[b * 64];
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int m = 16 * (blk0 + b) + 4 * g + r;
            if (b < nblk && m < M) o[static_cast<int64_t>(m) * N] = kw ? oth[r] + mine[r] : mine[r] + oth[r];
        }
    }
}

// K splits: as many as one workgroup per CU takes, at least four super-blocks
// each (two per K group).
int wreg_ksplit(int64_t N, int64_t K) {
    const int64_t tiles = (N + 127) / 128, nsb = K / 256;
    int64_t ks = num_cus() / tiles;
    if (ks > nsb / 4) ks = nsb / 4;
    return static_cast<int>(ks < 1 ? 1 : ks);
}

// Row tiles: what the CUs still have room for, at least four blocks each.
int wreg_rowtiles(int64_t M, int64_t N, int64_t ks) {
    const int64_t items = (N + 127) / 128 * ks, nblk = (M + 15) / 16;
    int64_t mt = num_cus() / items;
    if (mt > (nblk + 3) / 4) mt = (nblk + 3) / 4;
    return static_cast<int>(mt < 1 ? 1 : mt);
}

int64_t wreg_packed_bytes(int64_t M, int64_t K) { return (M + 15) / 16 * 16 * K * 2; }

}  // namespace

// Where this kernel leads: the smallest K, in super-blocks, from which it does
// at every K measured (0: not taken), by the rows of X (kWregRows) and the
// columns (kWregCols; the last entry beyond).
//
// Measured on MI355X over 68000 calls (each type and X; 11 to 19 values of M;
// N from 16 to 151936, K from 2048 to 28672, on a grid and at random; weights
// not in cache) against the skinny, K-split or tiled kernel that the call ran
// on before, the packing and the sum of the splits included.  No call that the
// table takes ran below 0.97 of the other kernel's rate; they gain 2.05 in the
// geometric mean; the ones left out are 1.09 in the mean and 0.63 at the worst.
// Some of both, us other / this one:
//   fp16 X            M = 17       32           64           128          256
//   Q4_K 4096x14336   29.5 / 21.9  35.2 / 22.3  62.8 / 25.8  77.3 / 33.8  78.7 / 49.2
//   Q6_K 4096x14336   29.8 / 28.5  38.7 / 28.8  61.5 / 32.4  90.1 / 43.2  86.0 / 68.3
//   Q8_0 8192x8192    43.6 / 30.3  56.0 / 29.7  89.8 / 33.1  58.1 / 41.3  74.1 / 63.5
//   Q4_K 4096x4096                              21.6 / 17.4  23.6 / 20.4
//   Q5_K 14336x4096   26.7 / 25.5  29.6 / 26.2  38.0 / 29.6  39.4 / 38.1  62.8 / 66.8
//   Q5_K 32768x2048                             40.8 / 27.5  43.4 / 34.6  47.9 / 62.7
//   fp32 X (the other kernels convert it in every column tile)
//   Q4_K 4096x14336   44.6 / 22.3  63.1 / 23.0  112 / 26.3   92.4 / 34.4  93.9 / 50.4
//   Q4_K 14336x4096                             30.4 / 25.0  39.8 / 32.6  55.7 / 48.1
//   Q6_K 4096x4096                              34.4 / 21.8  27.8 / 24.4  36.6 / 29.4
// Why the lines lie there: the packing and the sum of the splits are launches
// of their own, which a small K does not pay for (called eagerly, the three
// launches and the workspace take the host 18.5 us, one launch 11: Q4_K up to 20
// rows begins where the other kernel takes longer than that); up to 64 rows with
// fp16 X the other kernels decode a weight once as well; and above 192 rows the
// tiles of 16 blocks spill 34 / 27 / 11 registers on Q5_K / Q6_K / Q8_0.
constexpr int kWregRows[7] = {20, 32, 40, 64, 128, 192, 256};
constexpr int kWregCols[8] = {511, 2047, 4096, 6144, 8191, 11264, 16384, 32768};
constexpr uint8_t kWregMinSb[4][2][7][9] = {
    {
        { // Q4_K, X fp16
            {39, 39, 39, 39, 39,  0,  0,  0,  0},
            {32, 32, 32, 32, 34,  0,  0,  0,  0},
            {32, 24, 24, 16, 16, 47,  0,  8,  0},
            {32, 16, 16, 16, 16, 32, 32,  8,  8},
            {32, 16, 16, 17, 23, 16, 16,  8,  8},
            {32, 20, 21, 29, 22, 16, 16,  8,  8},
            {32, 20, 39, 20, 22, 16, 21,  8, 10},
        },
        { // X fp32
            {32, 24, 24, 16, 16, 32, 32,  0,  0},
            {32, 16, 16, 16, 16, 32, 32,  0, 32},
            {32, 16, 16, 16, 16, 12, 12,  8,  8},
            {32, 16, 16, 16, 16, 15, 13,  8,  8},
            {32, 16, 16, 16, 16, 12, 12,  8,  8},
            {32, 16, 16, 16, 16, 12, 12,  8,  8},
            {32, 16, 16, 16, 16, 15, 14,  8,  8},
        },
    },
    {
        { // Q5_K, X fp16
            {48, 50, 52, 32, 34, 15, 21, 12,  0},
            {32, 35, 41, 32, 34, 12, 20, 12, 12},
            {32, 31, 32, 16, 16, 12, 12,  8,  8},
            {32, 20, 20, 16, 16, 12, 12,  8,  8},
            {32, 16, 16, 16, 16, 15, 14,  8,  8},
            {32, 20, 20, 20, 22, 12, 13, 10,  8},
            {32, 20, 30, 20, 39, 29,  0,  0,  0},
        },
        { // X fp32
            {32, 32, 32, 32, 34, 12, 13, 12, 12},
            {32, 32, 32, 32, 34, 12, 12, 12, 12},
            {32, 16, 16, 16, 16, 12, 12,  8,  8},
            {32, 16, 16, 16, 16, 12, 12,  8,  8},
            {32, 16, 16, 16, 16, 12, 12,  8,  8},
            {32, 16, 16, 16, 16, 12, 12,  8,  8},
            {32, 16, 27, 16, 16, 12, 23, 42,  0},
        },
    },
    {
        { // Q6_K, X fp16
            {48, 50, 52, 48, 50, 48, 48,  0,  0},
            {48, 48, 48, 48, 50, 48, 48,  0,  0},
            {32, 31, 32, 24, 25, 24, 24,  8,  0},
            {32, 24, 24, 24, 25, 24, 24,  8,  9},
            {32, 16, 16, 20, 22, 16, 16,  8,  8},
            {32, 20, 20, 22, 22, 20, 20, 20, 20},
            {32, 20, 32, 20, 22, 25, 20,  0,  0},
        },
        { // X fp32
            {32, 32, 32, 32, 34, 32, 32,  0,  0},
            {32, 32, 32, 32, 34, 32, 32,  0, 32},
            {32, 16, 16, 16, 16, 12, 12,  8,  8},
            {32, 16, 16, 16, 16, 12, 12,  8,  8},
            {32, 16, 16, 16, 16, 12, 12,  8,  8},
            {32, 16, 16, 16, 16, 12, 12,  8,  8},
            {32, 16, 16, 16, 16, 12, 14, 42,  0},
        },
    },
    {
        { // Q8_0, X fp16
            {48, 50, 47, 32, 34, 15, 14, 12, 16},
            {32, 35, 35, 32, 34, 12, 13, 12, 12},
            {32, 31, 30, 16, 16, 12, 13,  8, 10},
            {32, 20, 20, 16, 16, 12, 12,  8,  8},
            {32, 16, 16, 16, 22, 15, 14,  8,  8},
            {32, 20, 20, 24, 22, 15, 14, 10, 10},
            {32, 20, 30, 20, 27, 25, 21,  0,  0},
        },
        { // X fp32
            {32, 32, 32, 32, 34, 12, 12, 12, 12},
            {32, 32, 32, 32, 34, 12, 12, 12, 12},
            {32, 16, 16, 16, 16, 12, 12,  8,  8},
            {32, 16, 16, 16, 16, 12, 12,  8,  8},
            {32, 16, 16, 16, 16, 12, 12,  8,  8},
            {32, 16, 16, 20, 16, 12, 12,  8,  8},
            {32, 16, 16, 16, 16, 12, 14, 22, 20},
        },
    },
};

bool gemm_wreg_shape(int32_t type, int32_t x_dtype, int64_t M, int64_t N, int64_t K) {
    const int t = type == TYPE_Q4_K ? 0 : (type == TYPE_Q5_K ? 1 : (type == TYPE_Q6_K ? 2 : (type == TYPE_Q8_0 ? 3 : -1)));
    if (t < 0 || K % 256 != 0 || M < 2 || M > 16 * wreg::MB_MAX) return false;
    if (knobs().gemm_wreg_min_m >= 0) return M >= knobs().gemm_wreg_min_m;
    const bool f32 = x_dtype == X_F32;
    // few rows: the conversion of fp32 X alone makes it worth it (M = 8, 4096 x
    // 12288: Q4_K 25.9 / 20.5, Q8_0 32.0 / 28.2)
    if (M < 17) return f32 && M >= 8 && N < 8192 && K >= (type == TYPE_Q6_K ? 14336 : 12288);
    int m = 0, n = 0;
    while (M > kWregRows[m]) m++;
    while (n < 8 && N > kWregCols[n]) n++;
    const int64_t sb = kWregMinSb[t][f32 ? 1 : 0][m][n];
    return sb != 0 && K >= 256 * sb;
}

int64_t gemm_wreg_workspace(int64_t M, int64_t N, int64_t K) {
    const int64_t ks = wreg_ksplit(N, K);
    return wreg_packed_bytes(M, K) + (ks > 1 ? ks * M * N * 4 : 0);
}

int gemm_wreg(const void* w, const void* X, int32_t x_dtype, float* Y, int64_t M, int64_t N, int64_t K, int32_t type,
              void* wsp, hipStream_t st) {
    const uint32_t rb = static_cast<uint32_t>(row_bytes(type, K));
    const uint32_t wbytes = static_cast<uint32_t>((N * rb + 3) & ~int64_t(3));
    const int m = static_cast<int>(M), n = static_cast<int>(N), k = static_cast<int>(K), nsb = k / 256;
    const int ks = wreg_ksplit(N, K), nblk = (m + 15) / 16, ntile = (n + 127) / 128;
    const int mt0 = wreg_rowtiles(M, N, ks), bpt = (nblk + mt0 - 1) / mt0, mt = (nblk + bpt - 1) / bpt;
    const dim3 pg(static_cast<uint32_t>(nblk), static_cast<uint32_t>(nsb));
    uint4* xf = static_cast<uint4*>(wsp);
    if (x_dtype == X_F16) wreg_pack_kernel<X_F16><<<pg, dim3(256), 0, st>>>(X, m, k, type == TYPE_Q6_K, xf);
    else wreg_pack_kernel<X_F32><<<pg, dim3(256), 0, st>>>(X, m, k, type == TYPE_Q6_K, xf);
    if (const int rc = check_launch("vb_gemm"); rc != OK) return rc;
    float* out = ks > 1 ? reinterpret_cast<float*>(static_cast<uint8_t*>(wsp) + wreg_packed_bytes(M, K)) : Y;
    const dim3 grid(static_cast<uint32_t>((ntile * ks * mt + 7) / 8 * 8));
    const uint8_t *wb = static_cast<const uint8_t*>(w), *x8 = static_cast<const uint8_t*>(wsp);
    auto by_rows = [&](auto type_c) {
        constexpr int T = decltype(type_c)::value;
#define VB_WREG(MB) \
    gemm_wreg_kernel<T, MB><<<grid, dim3(512), 0, st>>>(wb, wbytes, rb, x8, out, m, n, nsb, ntile, ks, mt, bpt)
        switch (bpt) {
            case 1: VB_WREG(1); break;
            case 2: VB_WREG(2); break;
            case 3: VB_WREG(3); break;
            case 4: VB_WREG(4); break;
            case 5: VB_WREG(5); break;
            case 6: VB_WREG(6); break;
            case 7: VB_WREG(7); break;
            case 8: VB_WREG(8); break;
            case 9: VB_WREG(9); break;
            case 10: VB_WREG(10); break;
            case 11:
            case 12: VB_WREG(12); break;
            default: VB_WREG(16); break;
        }
#undef VB_WREG
    };
    if (type == TYPE_Q4_K) by_rows(std::integral_constant<int, TYPE_Q4_K>{});
    else if (type == TYPE_Q5_K) by_rows(std::integral_constant<int, TYPE_Q5_K>{});
    else if (type == TYPE_Q6_K) by_rows(std::integral_constant<int, TYPE_Q6_K>{});
    else by_rows(std::integral_constant<int, TYPE_Q8_0>{});
    if (const int rc = check_launch("vb_gemm"); rc != OK) return rc;
    return ks > 1 ? gemm_ksum(out, Y, M * N, ks, st) : OK;
}

}  // namespace vb
