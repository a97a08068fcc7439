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

// Where this kernel leads.  MI355X, us old / this one (the packing and the
// sum of the splits included), old = the skinny, K-split or tiled kernel:
//   fp16 X            M = 17       32         64         128        256
//   Q4_K 4096x14336   29.2 / 21.3  36 / 22    63 / 26    69 / 34    77 / 52
//   Q6_K 4096x14336   29.7 / 27.5  39 / 28    62 / 32    90 / 42    87 / 70
//   Q8_0 4096x14336   37.6 / 29.9             81 / 34    96 / 42    101 / 64
//   Q4_K 8192x8192    19.7 / 21.9             36 / 24    51 / 34    84 / 55
//   Q6_K 4096x8192    17.7 / 21.0             31 / 23    55 / 31    56 / 48
//   Q4_K 4096x4096    11.5 / 13.9  14 / 15    21.3 / 17  24 / 20    26.6 / 27.2
//   Q6_K 4096x4096    10.3 / 17.8  13 / 19    20.3 / 22  27 / 24    28 / 34
//   Q4_K 14336x4096   13.3 / 19.6  16 / 21    26.2 / 24  33.1 / 33  54 / 52
//   Q5_K 14336x4096   26.8 / 25.0             39 / 29    42 / 38    68.0 / 68.4
//   Q4_K 32768x2048   16.7 / 18.2             26 / 21    42 / 32    66 / 51
//   Q4_K 8192x2048     8.1 / 13.5             13.8 / 15  18 / 19    26.6 / 27.6
//   fp32 X (the other kernels convert it in every column tile)
//   Q4_K 4096x14336   44.6 / 21.6             87 / 24    84 / 34    96 / 53
//   Q8_0 4096x14336   58.7 / 30.1            132 / 32   114 / 43   124 / 66
//   Q4_K 4096x4096    16.2 / 13.9             29 / 16    29 / 23    31 / 27
//   Q6_K 14336x4096   31.4 / 27.6             41 / 31    58 / 44    79 / 73
// Below K = 4096 the three launches and the first loads cost more than the
// decode saved, unless N is large.
bool gemm_wreg_shape(int32_t type, int32_t x_dtype, int64_t M, int64_t N, int64_t K) {
    if (type != TYPE_Q4_K && type != TYPE_Q5_K && type != TYPE_Q6_K && type != TYPE_Q8_0) return false;
    if (K % 256 != 0 || M < 2 || M > 16 * wreg::MB_MAX) return false;
    if (knobs().gemm_wreg_min_m >= 0) return M >= knobs().gemm_wreg_min_m;
    const bool q6 = type == TYPE_Q6_K, f32 = x_dtype == X_F32, wide = N >= 8192;
    const bool slow = type == TYPE_Q5_K || type == TYPE_Q8_0;  // no skinny kernel
    if (M < 17) return f32 && K >= 12288 && !wide && M >= 8;
    if (K >= 8192) return M > 32 || f32 || (q6 ? K >= 12288 : !(wide && type == TYPE_Q4_K));
    if (N < 512) return false;  // one to four workgroups per K split
    if (K >= 4096) {
        if (M <= 32) return wide ? slow : f32 && type == TYPE_Q4_K;
        if (M <= 64) return f32 || (N >= 1024 && (q6 ? K >= 6144 : !(wide && type == TYPE_Q4_K)));
        return M <= 128 || f32 || K >= 5120 || (wide && !q6);
    }
    if (K >= 3072 && wide && (slow ? M > 16 : f32 && M > 32)) return true;
    return M > 32 && K >= 2048 && N >= 16384 && (f32 || !q6 || M <= 128);
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
