// Expert-grouped MoE products for prefill-sized batches: the weights of a hit
// expert are read and decoded once per 160 of its slots (wreg_core.hpp), where
// the skinny and K-split expert kernels (moe.hip, gemm_kq.hip) do so once per
// 16.
//
// Three launches after the routing prep: pack (the experts' activation rows,
// gathered into fragment order), gate/up (SwiGLU in the epilogue, the hidden
// rows written straight in the down kernel's fragment order) and down.
//
// An expert's slots fill ceil(count / 16) blocks of 16 rows; its blocks make
// ceil(blocks / 10) tiles of equal size.  The host knows only the slot count,
// so the grids hold the most tiles any routing can give, and every workgroup
// finds its (expert, tile) from the slot offsets with one wave scan;
// workgroups past the last tile end at once.
#include "mfma_q4k.hpp"
#include "tile_index.hpp"
#include "wreg_core.hpp"
#include "vb_internal.hpp"
#include "../../include/vbhip.h"

namespace vb {
namespace {

using wreg::BUF_U4;

// Blocks per tile.  One kernel holds every tile height, so the tallest sets the
// registers of all: bodies of 16 blocks spilled (14 / 46 / 63 / 42 registers in
// gate/up on Q4_K / Q5_K / Q6_K / Q8_0, up to 42 in down), and one tall tile
// left the CUs idle that two of half its height fill.  MI355X, 2 experts of
// 4096 x 14336, slots each, us with tiles of up to 16 / 12 / 10 blocks: Q4_K
// gate/up, Q6_K down 160 280 / 279 / 287, 192 319 / 324 / 281, 208 464 / 291 /
// 290, 256 483 / 317 / 325, 512 627 / 494 / 449; Q8_0, Q5_K 208 547 / - / 313.
constexpr int MB_MAX = 10;

struct WregExperts {
    const uint8_t* p[MOE_KQ_MAX_EXPERTS];
};

// Work item `lin` of the routing's tiles x ncol column tiles (n_exp <= 64
// experts, lane e = expert e): false past the last one, else the row tile and
// its column tile.  A tile past the packed blocks is dropped (moe_wreg_tile).
// Workgroups go to the eight XCDs round robin (lin % 8);
// each XCD takes a contiguous eighth of the tile-major order, so a tile's
// packed rows are read into one or two XCDs' L2 only (down product at 8
// experts, 125 slots each, 4096 x 14336: the rows dealt over all XCDs ran
// 336 us on Q4_K and 411 us on Q6_K, pinned 240 on Q6_K).  With UNIT = 1 tiles are
// single blocks in order (the pack pass).
template <int UNIT>
__device__ __forceinline__ bool find_tile(const int32_t* __restrict__ eoff, const int32_t* __restrict__ elist,
                                          int n_exp, int nslots, int lin, int ncol, MoeTile& t, int& col) {
    const int lane = static_cast<int>(threadIdx.x) & 63;
    const int c = lane < n_exp ? expert_slots(eoff, elist, lane < n_exp ? lane : 0, nslots).count : 0;
    const int nb = (c + 15) >> 4;
    const int nt = UNIT == 1 ? nb : (nb + MB_MAX - 1) / MB_MAX;
    int st = nt, sb = nb;  // inclusive sums
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const int a = __shfl_up(st, o, 64), b = __shfl_up(sb, o, 64);
        if (lane >= o) {
            st += a;
            sb += b;
        }
    }
    int y = lin;
    col = 0;
    if (UNIT != 1) {
        const int items = __builtin_amdgcn_readlane(st, 63) * ncol, per = (items + 7) >> 3;
        const int w = (lin & 7) * per + (lin >> 3);
        if ((lin >> 3) >= per || w >= items) return false;
        y = w / ncol;
        col = w - y * ncol;
    }
    const uint64_t hit = __ballot(y >= st - nt && y < st);
    if (hit == 0) return false;
    const int e = __builtin_ctzll(hit);
    return moe_wreg_tile(e, y - __builtin_amdgcn_readlane(st - nt, e), __builtin_amdgcn_readlane(c, e),
                         __builtin_amdgcn_readlane(sb - nb, e), UNIT == 1 ? 1 : MB_MAX,
                         moe_wreg_blocks(nslots, n_exp), t);
}

// Packed activations: grid (blocks, h / 256), one 16 x 256 block each; rows
// past the expert's slots are zeros.  A wave reads 64 contiguous bytes of 16
// rows per load and writes four 256-byte runs.
__global__ void __launch_bounds__(256) moe_wreg_pack(const _Float16* __restrict__ xh, const int32_t* __restrict__ eoff,
                                                     const int32_t* __restrict__ elist, int n_exp, int nslots, int topk,
                                                     int h, int q6, uint4* __restrict__ xf) {
    MoeTile t;
    int col;
    if (!find_tile<1>(eoff, elist, n_exp, nslots, static_cast<int>(blockIdx.x), 1, t, col)) return;
    const SlotRange slots = expert_slots(eoff, elist, t.e, nslots);
    const int sb = static_cast<int>(blockIdx.y), nsb = h >> 8;
    uint4* dst = xf + (static_cast<int64_t>(t.blk0) * nsb + sb) * 512;
#pragma unroll
    for (int q = 0; q < 2; q++) {
        const int id = static_cast<int>(threadIdx.x) + 256 * q;
        const int row = (id >> 2) & 15, piece = (id & 3) + 4 * (id >> 6);
        uint4 v = make_uint4(0, 0, 0, 0);
        if (row < t.cnt) {
            const int64_t tok = slots[t.m0 + row] / topk;
            v = *reinterpret_cast<const uint4*>(xh + tok * h + 256 * sb + 8 * piece);
        }
        int g, m, e;
        wreg::k_slot(8 * piece, q6 != 0, g, m, e);
        dst[m * 64 + g * 16 + row] = v;
    }
}

// gate/up: 1-D grid of tiles x (i / 64).  Each wave multiplies 16 gate rows
// and the same 16 up rows.
template <int TYPE, int MB>
__device__ __forceinline__ void gate_up_body(const uint8_t* wg, const uint8_t* wu, uint32_t wbytes, const uint8_t* xf,
                                             const MoeTile& t, int h, int i_dim, uint32_t rb, int n0,
                                             int q6_out, _Float16* __restrict__ hf, u32x4* b0, u32x4* b1) {
    const int lane = static_cast<int>(threadIdx.x) & 63, j = lane & 15, g = lane >> 4;
    const int wn = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
    const int nsb = h >> 8;
    const int n = n0 + 16 * wn + j;
    const uint32_t ro = static_cast<uint32_t>(n) * rb;
    const __amdgpu_buffer_rsrc_t xs = make_rsrc(xf + static_cast<int64_t>(t.blk0) * nsb * 8192,
                                                static_cast<uint32_t>(t.nblk * nsb) * 8192u);
    float4_t acc[MB][2];
#pragma unroll
    for (int b = 0; b < MB; b++) acc[b][0] = acc[b][1] = float4_t{0.f, 0.f, 0.f, 0.f};
    wreg::mainloop<TYPE, MB>(acc, make_rsrc(wg, wbytes), make_rsrc(wu, wbytes), ro, ro, xs, t.nblk, nsb, 0, nsb, nsb,
                             b0, b1, wn);
    // silu(gate) up of rows 4 g .. + 3 and column n of each block, as fp16
    // (the down product takes fp16 rows) in the down kernel's fragment order
    int kg, kt, ke;
    wreg::k_slot(n & 255, q6_out != 0, kg, kt, ke);
    const int nsbi = i_dim >> 8;
    _Float16* dst = hf + ((static_cast<int64_t>(t.blk0) * nsbi + (n >> 8)) * 8 + kt) * 512 + (kg * 16 + 4 * g) * 8 + ke;
#pragma unroll
    for (int b = 0; b < MB; b++) {
        if (b < t.nblk)
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const float gv = acc[b][0][r], uv = acc[b][1][r];
            dst[static_cast<int64_t>(b) * nsbi * 4096 + 8 * r] =
                static_cast<_Float16>(gv / (1.0f + __expf(-gv)) * uv);
        }
    }
}

template <int TYPE>
__global__ void __launch_bounds__(256, 2) moe_wreg_gate_up(WregExperts wg, WregExperts wu, uint32_t wbytes,
                                                           const uint8_t* __restrict__ xf,
                                                           const int32_t* __restrict__ eoff,
                                                           const int32_t* __restrict__ elist, int n_exp, int nslots,
                                                           int h, int i_dim, uint32_t rb, int q6_out,
                                                           _Float16* __restrict__ hf) {
    __shared__ u32x4 b0[BUF_U4];
    __shared__ u32x4 b1[BUF_U4];
    MoeTile t;
    int col;
    if (!find_tile<MB_MAX>(eoff, elist, n_exp, nslots, static_cast<int>(blockIdx.x), i_dim / 64, t, col)) return;
    const int n0 = col * 64;
    const uint8_t *pg = wg.p[t.e], *pu = wu.p[t.e];
#define VB_WREG_GU(MB) \
    gate_up_body<TYPE, MB>(pg, pu, wbytes, xf, t, h, i_dim, rb, n0, q6_out, hf, b0, b1)
    switch (t.nblk) {
        case 1:
        case 2: VB_WREG_GU(2); break;
        case 3: VB_WREG_GU(3); break;
        case 4: VB_WREG_GU(4); break;
        case 5: VB_WREG_GU(5); break;
        case 6: VB_WREG_GU(6); break;
        case 7: VB_WREG_GU(7); break;
        case 8: VB_WREG_GU(8); break;
        case 9: VB_WREG_GU(9); break;
        default: VB_WREG_GU(10); break;
    }
#undef VB_WREG_GU
}

// down: 1-D grid of tiles x (h / 128); the workgroup's two K groups take half
// of the super-blocks each (a 4096-row matrix has 32 column tiles only) and
// exchange one column fragment's sums through LDS.
template <int TYPE, int MB>
__device__ __forceinline__ void down_body(const uint8_t* wd, uint32_t wbytes, const uint8_t* hf, const SlotRange& slots,
                                          const MoeTile& t, int h, int i_dim, uint32_t rb, int n0, float* __restrict__ obuf,
                                          const float* __restrict__ rw, int topk, float* __restrict__ yacc, u32x4* b0,
                                          u32x4* b1) {
    const int lane = static_cast<int>(threadIdx.x) & 63, j = lane & 15, g = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
    const int wn = wave & 3, kw = wave >> 2;
    const int nsb = i_dim >> 8, half = (nsb + 1) >> 1;
    const int nc = n0 + 32 * wn + j;  // column of fragment 0; fragment 1 is 16 on
    const __amdgpu_buffer_rsrc_t ws = make_rsrc(wd, wbytes);
    const __amdgpu_buffer_rsrc_t xs = make_rsrc(hf + static_cast<int64_t>(t.blk0) * nsb * 8192,
                                                static_cast<uint32_t>(t.nblk * nsb) * 8192u);
    float4_t acc[MB][2];
#pragma unroll
    for (int b = 0; b < MB; b++) acc[b][0] = acc[b][1] = float4_t{0.f, 0.f, 0.f, 0.f};
    wreg::mainloop<TYPE, MB>(acc, ws, ws, static_cast<uint32_t>(nc) * rb, static_cast<uint32_t>(nc + 16) * rb, xs,
                             t.nblk, nsb, kw ? half : 0, kw ? nsb - half : half, half, b0 + kw * BUF_U4,
                             b1 + kw * BUF_U4, wn);
    // K group kw finishes fragment kw: the other group's sums of it come
    // through LDS (group 0's of fragment 1 in b0, group 1's of fragment 0 in b1)
    float4_t* out = reinterpret_cast<float4_t*>(kw ? b1 : b0) + (wn * MB) * 64 + lane;
    const float4_t* in = reinterpret_cast<const float4_t*>(kw ? b0 : b1) + (wn * MB) * 64 + lane;
#pragma unroll
    for (int b = 0; b < MB; b++) out[b * 64] = acc[b][kw ? 0 : 1];
    __syncthreads();
    const int n = nc + 16 * kw;
#pragma unroll
    for (int b = 0; b < MB; b++) {
        const float4_t mine = acc[b][kw ? 1 : 0], oth = in[b * 64];
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int m = 16 * b + 4 * g + r;
            if (m >= t.cnt) continue;
            const float v = mine[r] + oth[r];
            const int q = slots[t.m0 + m];
            if (yacc)  // at most two additions into zero: the same bits in either order
                unsafeAtomicAdd(yacc + static_cast<int64_t>(q / topk) * h + n, rw[q] * v);
            else
                obuf[static_cast<int64_t>(q) * h + n] = v;
        }
    }
}

template <int TYPE>
__global__ void __launch_bounds__(512) moe_wreg_down(WregExperts wd, uint32_t wbytes, const uint8_t* __restrict__ hf,
                                                     const int32_t* __restrict__ eoff,
                                                     const int32_t* __restrict__ elist, int n_exp, int nslots,
                                                     int h, int i_dim, uint32_t rb, float* __restrict__ obuf,
                                                     const float* __restrict__ rw, int topk, float* __restrict__ yacc) {
    __shared__ u32x4 b0[2 * BUF_U4];
    __shared__ u32x4 b1[2 * BUF_U4];
    MoeTile t;
    int col;
    if (!find_tile<MB_MAX>(eoff, elist, n_exp, nslots, static_cast<int>(blockIdx.x), h / 128, t, col)) return;
    const SlotRange slots = expert_slots(eoff, elist, t.e, nslots);
    const int n0 = col * 128;
    const uint8_t* pd = wd.p[t.e];
#define VB_WREG_DN(MB) down_body<TYPE, MB>(pd, wbytes, hf, slots, t, h, i_dim, rb, n0, obuf, rw, topk, yacc, b0, b1)
    switch (t.nblk) {
        case 1:
        case 2: VB_WREG_DN(2); break;
        case 3: VB_WREG_DN(3); break;
        case 4: VB_WREG_DN(4); break;
        case 5: VB_WREG_DN(5); break;
        case 6: VB_WREG_DN(6); break;
        case 7: VB_WREG_DN(7); break;
        case 8: VB_WREG_DN(8); break;
        case 9: VB_WREG_DN(9); break;
        default: VB_WREG_DN(10); break;
    }
#undef VB_WREG_DN
}

WregExperts experts(const void* const* w, int n) {
    WregExperts e{};
    for (int i = 0; i < n; i++) e.p[i] = static_cast<const uint8_t*>(w[i]);
    return e;
}

}  // namespace

bool moe_wreg_type(int32_t t) { return t == TYPE_Q4_K || t == TYPE_Q5_K || t == TYPE_Q6_K || t == TYPE_Q8_0; }

int moe_wreg(int32_t gu_type, int32_t dn_type, const void* const* wg, const void* const* wu, const void* const* wd,
             int n_exp, const _Float16* xh, int nslots, int topk, int64_t h, int64_t i, const int32_t* eoff,
             const int32_t* elist, void* xf, void* hf, float* obuf, const float* rw, float* yacc, hipStream_t st) {
    const int blocks = moe_wreg_blocks(nslots, n_exp), tiles = moe_wreg_tiles(nslots, n_exp, MB_MAX);
    const int ih = static_cast<int>(h), ii = static_cast<int>(i);
    const uint32_t rb_gu = static_cast<uint32_t>(row_bytes(gu_type, h)), rb_d = static_cast<uint32_t>(row_bytes(dn_type, i));
    const uint32_t wb_gu = static_cast<uint32_t>((i * rb_gu + 3) & ~int64_t(3));
    const uint32_t wb_d = static_cast<uint32_t>((h * rb_d + 3) & ~int64_t(3));
    int rc;
    moe_wreg_pack<<<dim3(static_cast<uint32_t>(blocks), static_cast<uint32_t>(h / 256)), dim3(256), 0, st>>>(
        xh, eoff, elist, n_exp, nslots, topk, ih, gu_type == TYPE_Q6_K, static_cast<uint4*>(xf));
    if ((rc = check_launch("vb_moe_grouped_ffn")) != OK) return rc;
    const WregExperts pg = experts(wg, n_exp), pu = experts(wu, n_exp), pd = experts(wd, n_exp);
    // whole eighths (find_tile)
    const dim3 gg(static_cast<uint32_t>((tiles * (i / 64) + 7) / 8 * 8)), gd(static_cast<uint32_t>((tiles * (h / 128) + 7) / 8 * 8));
    const uint8_t* x8 = static_cast<const uint8_t*>(xf);
    auto gate_up = [&](auto type_c) {
        moe_wreg_gate_up<decltype(type_c)::value><<<gg, dim3(256), 0, st>>>(
            pg, pu, wb_gu, x8, eoff, elist, n_exp, nslots, ih, ii, rb_gu, dn_type == TYPE_Q6_K,
            static_cast<_Float16*>(hf));
    };
    auto down = [&](auto type_c) {
        moe_wreg_down<decltype(type_c)::value><<<gd, dim3(512), 0, st>>>(
            pd, wb_d, static_cast<const uint8_t*>(hf), eoff, elist, n_exp, nslots, ih, ii, rb_d, obuf, rw, topk,
            yacc);
    };
    auto by_type = [](int32_t t, auto&& f) {
        if (t == TYPE_Q4_K) f(std::integral_constant<int, TYPE_Q4_K>{});
        else if (t == TYPE_Q5_K) f(std::integral_constant<int, TYPE_Q5_K>{});
        else if (t == TYPE_Q6_K) f(std::integral_constant<int, TYPE_Q6_K>{});
        else f(std::integral_constant<int, TYPE_Q8_0>{});
    };
    by_type(gu_type, gate_up);
    if ((rc = check_launch("vb_moe_grouped_ffn")) != OK) return rc;
    by_type(dn_type, down);
    return check_launch("vb_moe_grouped_ffn");
}

}  // namespace vb
