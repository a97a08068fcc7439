// GEMM for 2 to 16 activation rows, K <= 4096: weight rows streamed whole.
//
// The other small-batch kernels load a lane's own bytes of 16 weight rows per
// instruction, which touches 16 to 32 cache lines for 1 KB and holds the
// stream at 2.6 TB/s.  Here 16 rows, which lie back to back in the tensor, are
// loaded as one linear image (1 KB contiguous per instruction), a group of
// rows ahead of the arithmetic, and go through registers into LDS, where the
// lanes pick their bytes.  (LDS DMA would save the registers, but the compiler
// then waits for all of it before each of these reads.)
//
// One persistent workgroup of eight waves per CU walks over the groups of 16
// rows.  Each wave owns an eighth of K for all of them: its activation
// fragments stay in registers for the whole launch (K <= 4096: 16 fragments).
// Per group a wave decodes and multiplies its share, and the eight partial
// 16 x 16 products meet in LDS; they are summed, in wave order, and stored in
// the next group's turn, so a group costs one barrier.
//
// MI355X, M = 5, fp16 X: Q6_K 128256 x 4096 (431 MB) 168 us on the K-split
// kernel, 83 here (5.2 TB/s).  The decode and the LDS round trip beside one
// group's loads in flight bound it.  Q4_K stays on its skinny kernel
// (gemm_skinny.hip): 83 us against 89 at 128256 x 4096, 11 against 16 at 14336.
#include "kq_types.hpp"
#include "tile_index.hpp"
#include "vb_internal.hpp"
#include "../../include/vbhip.h"

namespace vb {
namespace {

constexpr int ROWS_WAVES = 8;
constexpr int ROWS_STEPS = 4;       // 128-element steps per wave, at most
constexpr int ROWS_MAX_K = 4096;

constexpr int rows_block_bytes(int type) {  // of 256 elements
    return type == TYPE_Q5_K ? 176 : (type == TYPE_Q6_K ? 210 : 272);
}
// 1 KB pieces per wave and group of 16 rows at K = 4096
constexpr int rows_pieces(int type) { return (16 * 16 * rows_block_bytes(type) + 8191) / 8192; }

__device__ __forceinline__ void rows_barrier() {
    // the wave's LDS stores are done, then everyone's; loads stay in flight
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_waitcnt(0xC07F);
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
}

template <int TYPE, int XT>
__global__ void __launch_bounds__(64 * ROWS_WAVES) gemm_rows_kernel(const uint8_t* __restrict__ w, uint32_t wbytes,
                                                                    const void* __restrict__ X, float* __restrict__ Y,
                                                                    int M, int N, int K, uint32_t rb) {
    using T = Kq<TYPE>;
    // Rows of an even number of 16-byte slots put the 16 rows of a read on few
    // banks and get a slot's gap (rows_pitch; Q8_0 14336 x 4096: 29 us without,
    // 19 with).  Q6_K rows (210 bytes a block) spread by themselves and need
    // not be whole slots.
    constexpr bool WHOLE = TYPE != TYPE_Q6_K;
    constexpr int P = rows_pieces(TYPE), IMG = 16 * rows_block_bytes(TYPE) + 32;  // 16-byte slots
    __shared__ u32x4 b0[IMG];
    __shared__ u32x4 b1[IMG];
    __shared__ float4_t red[2][ROWS_WAVES * 64];
    const int lane = static_cast<int>(threadIdx.x) & 63, j = lane & 15, g = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
    const int ngroups = (N + 15) >> 4, nsteps = K >> 7;
    const int s0 = wave * nsteps / ROWS_WAVES, cnt = (wave + 1) * nsteps / ROWS_WAVES - s0;
    const __amdgpu_buffer_rsrc_t wr = make_rsrc(w, wbytes);
    const KqConsts kc = kq_consts();
    const int first = static_cast<int>(blockIdx.x), stride = static_cast<int>(gridDim.x);

    // rows 16 grp .. + 15; rows and groups past the last read nothing
    u32x4 st[P];
    const uint32_t pitch = WHOLE ? rows_pitch(rb) : rb;
    const uint32_t gap = (pitch - rb) >> 4;
    int at[P];  // the lane's slots in an image; pieces past the rows go to its last one
#pragma unroll
    for (int i = 0; i < P; i++) {
        const uint32_t slot = static_cast<uint32_t>((wave + ROWS_WAVES * i) * 64 + lane);
        at[i] = slot < rb ? static_cast<int>(slot + (WHOLE ? slot / (rb >> 4) * gap : 0u)) : IMG - 1;
    }
    auto fetch = [&](int grp) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < P; i++) {
            const uint32_t slot = static_cast<uint32_t>((wave + ROWS_WAVES * i) * 64 + lane);
            const uint32_t vo = rows_fetch_at(grp, ngroups, slot, rb);
            st[i] = __builtin_amdgcn_raw_buffer_load_b128(wr, static_cast<int>(vo), 0, 2);
        }
    };
    auto put = [&](u32x4* dst) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < P; i++) dst[at[i]] = st[i];
    };
    fetch(first);
    // activation fragments of the wave's steps (rows past M: zeros)
    constexpr int GSTR = T::kBlockLane ? 32 : 8, KSTR = T::kBlockLane ? 8 : 32;
    Frag af[ROWS_STEPS][4];
#pragma unroll
    for (int s = 0; s < ROWS_STEPS; s++)
#pragma unroll
        for (int ks = 0; ks < 4; ks++) {
            uint4 v = make_uint4(0, 0, 0, 0);
            if (s < cnt && j < M) v = x8_f16<XT>(X, static_cast<int64_t>(j) * K + 128 * (s0 + s) + GSTR * g + KSTR * ks);
            af[s][ks].u[0] = v.x;
            af[s][ks].u[1] = v.y;
            af[s][ks].u[2] = v.z;
            af[s][ks].u[3] = v.w;
        }
    // the finished sums of group grp (partial products in red[p]): four waves, one output per thread
    auto finish = [&](int grp, int p) __attribute__((always_inline)) {
        if (wave >= 4) return;
        const int tok = static_cast<int>(threadIdx.x) >> 4, col = static_cast<int>(threadIdx.x) & 15;
        const float* r = reinterpret_cast<const float*>(red[p]) + ((tok >> 2) * 16 + col) * 4 + (tok & 3);
        float s = r[0];
#pragma unroll
        for (int v = 1; v < ROWS_WAVES; v++) s += r[v * 256];
        const int n = 16 * grp + col;
        if (tok < M && n < N) Y[static_cast<int64_t>(tok) * N + n] = s;
    };
    int grp = first, turn = 0;
    auto group = [&](u32x4* cur, u32x4* nxt) __attribute__((always_inline)) {
        rows_barrier();
        if (turn > 0) finish(grp - stride, (turn - 1) & 1);
        float4_t acc[2] = {float4_t{0.f, 0.f, 0.f, 0.f}, float4_t{0.f, 0.f, 0.f, 0.f}};
        const uint8_t* img = reinterpret_cast<const uint8_t*>(cur);
#pragma unroll
        for (int s = 0; s < ROWS_STEPS; s++) {
            if (s < cnt) {
                typename T::Raw raw;
                Frag f[4];
                T::read(img, static_cast<uint32_t>(j) * pitch, s0 + s, g, raw);
                T::decode(raw, static_cast<uint32_t>(j) * pitch, s0 + s, g, kc, f);
#pragma unroll
                for (int ks = 0; ks < 4; ks++) acc[ks & 1] = mfma16x16x32(af[s][ks], f[ks], acc[ks & 1]);
            }
        }
        red[turn & 1][wave * 64 + lane] = acc[0] + acc[1];
        // the next group's rows, loaded during this one's arithmetic, into the
        // image that every wave was done with at the barrier
        __builtin_amdgcn_sched_barrier(0);
        put(nxt);
        fetch(grp + 2 * stride);
        __builtin_amdgcn_sched_barrier(0);
        grp += stride;
        turn++;
    };
    put(b0);
    fetch(grp + stride);
    while (grp < ngroups) {
        group(b0, b1);
        if (grp >= ngroups) break;
        group(b1, b0);
    }
    rows_barrier();
    if (turn > 0) finish(grp - stride, (turn - 1) & 1);
}

}  // namespace

// The rule and what it was measured on: rows_lead (tile_index.hpp).
bool gemm_rows_shape(int32_t type, int64_t M, int64_t N, int64_t K) {
    if (type != TYPE_Q5_K && type != TYPE_Q6_K && type != TYPE_Q8_0) return false;
    if (M < 2 || M > 16 || K % 256 != 0 || K > ROWS_MAX_K || N * row_bytes(type, K) >= (int64_t(1) << 31)) return false;
    if (knobs().gemm_rows_min_n >= 0) return N >= knobs().gemm_rows_min_n;
    return rows_lead(type == TYPE_Q5_K, type == TYPE_Q8_0, N, K);
}

int gemm_rows(const void* w, const void* X, int32_t x_dtype, float* Y, int64_t M, int64_t N, int64_t K, int32_t type,
              hipStream_t st) {
    const uint32_t rb = static_cast<uint32_t>(row_bytes(type, K));
    const uint32_t wbytes = static_cast<uint32_t>((N * rb + 3) & ~int64_t(3));
    const int64_t groups = (N + 15) / 16;
    const dim3 grid(static_cast<uint32_t>(groups < num_cus() ? groups : num_cus())), block(64 * ROWS_WAVES);
    const uint8_t* wb = static_cast<const uint8_t*>(w);
    const int m = static_cast<int>(M), n = static_cast<int>(N), k = static_cast<int>(K);
#define VB_ROWS(T)                                                                              \
    do {                                                                                        \
        if (x_dtype == X_F16) gemm_rows_kernel<T, X_F16><<<grid, block, 0, st>>>(wb, wbytes, X, Y, m, n, k, rb); \
        else gemm_rows_kernel<T, X_F32><<<grid, block, 0, st>>>(wb, wbytes, X, Y, m, n, k, rb); \
    } while (0)
    if (type == TYPE_Q5_K) VB_ROWS(TYPE_Q5_K);
    else if (type == TYPE_Q6_K) VB_ROWS(TYPE_Q6_K);
    else VB_ROWS(TYPE_Q8_0);
#undef VB_ROWS
    return check_launch("vb_gemm");
}

}  // namespace vb
