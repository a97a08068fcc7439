// GEMM tile with the weights decoded straight into B fragments in registers
// and the activations shared through LDS, for 17 to 256 activation rows per
// tile; used by the batched GEMM (gemm_wreg.hip) and the expert-grouped MoE
// products (moe_wreg.hip, up to 160 rows).
//
// Why this shape.  At these row counts a weight serves few enough MFMAs that
// decoding it costs about as much as multiplying it, so each weight is
// decoded exactly once per tile of up to 256 rows, by the one wave that owns
// its column, and never goes through LDS.  A wave owns two 16-column
// fragments and all the tile's rows (MB blocks of 16): one decoded fragment
// feeds MB MFMAs.  The activations, which all waves of a workgroup share,
// come packed in fragment order and land in LDS by DMA, double buffered.  A
// workgroup has four such waves per K group; two workgroups (or two K
// groups) fill a CU, so one wave's decode runs beside another's MFMAs.
//
// What bounds it (MI355X, kernel trace and counters, the GEMM case 100 rows of
// 4096 x 14336 Q4_K, the MoE 8 experts of 4096 x 14336, Q4_K gate/up and Q6_K
// down, 125 slots each): GEMM 23.5 us, gate/up 282 (830 TFLOP/s), down 243.
// The matrix cores are busy 18 / 45 / 23 % of that, a wave waits 40 / 20 / 35 %
// of its life and issues 26 / 33 / 19 %: MFMA, decode and the waits for weights
// come in turn more than beside each other.  No LDS bank conflicts.  Spelling
// out the order of reads, MFMAs and decode took gate/up / down from 300 / 240 to
// 260 / 220.  At 25 to 64 slots per expert the weight loads bound it, at about
// 3 TB/s: a load touches 16 rows.
//
// K order.  Lane group g (lane / 16) of the MFMA takes its own 64 of a
// super-block's 256 elements, so a lane loads whole 16-byte pieces of its
// row and decodes only its own sub-blocks' scales.  MFMA t = 0..7 of a
// super-block multiplies, in lane group g, the 8 elements from k_of(g, t) on:
//   64 g + 32 (t % 2) + 8 (t / 2)                              most types
//   128 (g / 2) + 32 (2 (t / 2 % 2) + t % 2) + 16 (g % 2) + 8 (t / 4)   Q6_K
// (the Q6_K order gives each lane 16 bytes of each of its two ql runs and of
// qh).  Packed activations: block b of 16 rows, super-block sb, MFMA t is 1
// KB at ((b nsb + sb) 8 + t) 1024, lane (i, g) of it X[16 b + i, 256 sb +
// k_of(g, t) .. + 8) in fp16.
#pragma once

#include <type_traits>

#include "mfma_q4k.hpp"
#include "skinny_core.hpp"  // the lane's Q4_K scale selection

namespace vb {
namespace wreg {

constexpr int MB_MAX = 16;            // 16-row blocks per tile
constexpr int BUF_U4 = 40 * 64;       // 16-byte slots of one LDS buffer of one K group (40 KB)

// element of a super-block -> (lane group, MFMA, position in the 8)
__device__ __forceinline__ void k_slot(int w, bool q6, int& g, int& t, int& e) {
    e = w & 7;
    if (q6) {
        g = 2 * (w >> 7) + ((w >> 4) & 1);
        t = 4 * ((w >> 3) & 1) + ((w >> 5) & 3);
    } else {
        g = w >> 6;
        t = 2 * ((w & 31) >> 3) + ((w >> 5) & 1);
    }
}

// Per type: Raw = one lane's bytes of a super-block, load() issues their
// kLoads loads (ro = the weight row's byte offset), prep() the lane's scales,
// frags() the B fragments of MFMAs 2 s and 2 s + 1.
template <int TYPE> struct W;

template <>
struct W<TYPE_Q4_K> {
    static constexpr int kLoads = 3;
    struct Raw {
        u32x4 hd, qa, qb;
    };
    struct Sc {
        half2_t ds[2], nm[2];
    };
    __device__ static __forceinline__ void load(__amdgpu_buffer_rsrc_t r, uint32_t ro, int g, int sb, Raw& v) {
        const uint32_t so = static_cast<uint32_t>(sb) * 144u, qo = ro + 16u + 32u * static_cast<uint32_t>(g);
        v.hd = buf_ld128(r, ro, so);
        v.qa = buf_ld128(r, qo, so);
        v.qb = buf_ld128(r, qo + 16u, so);
    }
    __device__ static __forceinline__ void prep(const Raw& v, uint32_t, int g, int, Sc& sc) {
        skinny::lane_chunk_scales(v.hd, skinny::lane_scale_sel(g), sc.ds, sc.nm);
    }
    template <int S>
    __device__ static __forceinline__ void frags(const Raw& v, const Sc& sc, int, const KqConsts&, Frag& lo, Frag& hi) {
        const uint32_t q[8] = {v.qa.x, v.qa.y, v.qa.z, v.qa.w, v.qb.x, v.qb.y, v.qb.z, v.qb.w};
        q4k_bfrags_cvt(q[2 * S], q[2 * S + 1], sc.ds, sc.nm, lo, hi);
    }
};

// Q5_K: the Q4_K header, qh[32] @16, qs[128] @48
template <>
struct W<TYPE_Q5_K> {
    static constexpr int kLoads = 5;
    struct Raw {
        u32x4 hd, ha, hb, qa, qb;
    };
    struct Sc {
        half2_t ds[2], nm[2];
    };
    __device__ static __forceinline__ void load(__amdgpu_buffer_rsrc_t r, uint32_t ro, int g, int sb, Raw& v) {
        const uint32_t so = static_cast<uint32_t>(sb) * 176u, qo = ro + 48u + 32u * static_cast<uint32_t>(g);
        v.hd = buf_ld128(r, ro, so);
        v.ha = buf_ld128(r, ro + 16u, so);
        v.hb = buf_ld128(r, ro + 32u, so);
        v.qa = buf_ld128(r, qo, so);
        v.qb = buf_ld128(r, qo + 16u, so);
    }
    __device__ static __forceinline__ void prep(const Raw& v, uint32_t, int g, int, Sc& sc) {
        skinny::lane_chunk_scales(v.hd, skinny::lane_scale_sel(g), sc.ds, sc.nm);
    }
    template <int S>
    __device__ static __forceinline__ void frags(const Raw& v, const Sc& sc, int g, const KqConsts& kc, Frag& lo,
                                                 Frag& hi) {
        const uint32_t q[8] = {v.qa.x, v.qa.y, v.qa.z, v.qa.w, v.qb.x, v.qb.y, v.qb.z, v.qb.w};
        const uint32_t h[8] = {v.ha.x, v.ha.y, v.ha.z, v.ha.w, v.hb.x, v.hb.y, v.hb.z, v.hb.w};
        q5k_frags(q[2 * S], q[2 * S + 1], h[2 * S], h[2 * S + 1], static_cast<uint32_t>(g), sc.ds, sc.nm, kc, lo, hi);
    }
};

// Q8_0: lane group g holds blocks 2 g, 2 g + 1 (68 bytes from a dword)
template <>
struct W<TYPE_Q8_0> {
    static constexpr int kLoads = 5;
    struct Raw {
        u32x4 a, b, c, d;
        uint32_t e;
    };
    struct Sc {
        half2_t dd[2];
    };
    __device__ static __forceinline__ void load(__amdgpu_buffer_rsrc_t r, uint32_t ro, int g, int sb, Raw& v) {
        const uint32_t so = static_cast<uint32_t>(sb) * 272u, o = ro + 68u * static_cast<uint32_t>(g);
        v.a = buf_ld128(r, o, so);
        v.b = buf_ld128(r, o + 16u, so);
        v.c = buf_ld128(r, o + 32u, so);
        v.d = buf_ld128(r, o + 48u, so);
        v.e = __builtin_amdgcn_raw_buffer_load_b32(r, static_cast<int>(o + 64u), static_cast<int>(so), 0);
    }
    __device__ static __forceinline__ void prep(const Raw& v, uint32_t, int, int, Sc& sc) {
        const uint32_t d0 = v.a.x & 0xFFFFu, d1 = v.c.x >> 16;  // bytes 0 and 34
        sc.dd[0] = bits2h(d0 | (d0 << 16));
        sc.dd[1] = bits2h(d1 | (d1 << 16));
    }
    template <int S>
    __device__ static __forceinline__ void frags(const Raw& v, const Sc& sc, int, const KqConsts& kc, Frag& lo,
                                                 Frag& hi) {
        const uint32_t w[17] = {v.a.x, v.a.y, v.a.z, v.a.w, v.b.x, v.b.y, v.b.z, v.b.w, v.c.x,
                                v.c.y, v.c.z, v.c.w, v.d.x, v.d.y, v.d.z, v.d.w, v.e};
        const uint32_t qs[4] = {__builtin_amdgcn_alignbyte(w[2 * S + 1], w[2 * S], 2u),
                                __builtin_amdgcn_alignbyte(w[2 * S + 2], w[2 * S + 1], 2u), w[9 + 2 * S],
                                w[10 + 2 * S]};
        const half2_t k1152 = half2_t{static_cast<_Float16>(1152.0f), static_cast<_Float16>(1152.0f)};
#pragma unroll
        for (int b = 0; b < 2; b++) {
            Frag& f = b ? hi : lo;
#pragma unroll
            for (int i = 0; i < 4; i++) {
                // (b ^ 0x80) | 0x6400 is the half 1024 + q + 128 (exact)
                const uint32_t src =
                    __builtin_amdgcn_perm(0u, qs[2 * b + (i >> 1)], (i & 1) ? 0x0C030C02u : 0x0C010C00u);
                f.u[i] = h2bits((bits2h(src ^ kc.x80) - k1152) * sc.dd[b]);
            }
        }
    }
};

// Q6_K: lane group g = 2 h + b takes ql[64 h + 16 b, +16) and ql[64 h + 32 +
// 16 b, +16), qh[32 h + 16 b, +16) and the scales 8 h + 2 q + b of quarters q;
// super-blocks start on even bytes, so each field is read as the dwords from
// its address rounded down to 4 and realigned.
template <>
struct W<TYPE_Q6_K> {
    static constexpr int kLoads = 8;
    struct Raw {
        u32x4 l0, l1, h;
        uint32_t l0e, l1e, he;
        u32x3 sc;
        uint32_t d;
    };
    struct Sc {
        half2_t ds[4];
        uint32_t l0[4], l1[4], h[4];
    };
    __device__ static __forceinline__ void load(__amdgpu_buffer_rsrc_t r, uint32_t ro, int g, int sb, Raw& v) {
        const uint32_t a = (ro + static_cast<uint32_t>(sb) * 210u) & ~3u;
        const uint32_t h = static_cast<uint32_t>(g >> 1), b = static_cast<uint32_t>(g & 1);
        const uint32_t lo = a + 64u * h + 16u * b, ho = a + 128u + 32u * h + 16u * b;
        v.l0 = buf_ld128(r, lo, 0);
        v.l0e = ld32(r, lo + 16u);
        v.l1 = buf_ld128(r, lo + 32u, 0);
        v.l1e = ld32(r, lo + 48u);
        v.h = buf_ld128(r, ho, 0);
        v.he = ld32(r, ho + 16u);
        v.sc = ld96(r, a + 192u + 8u * h);
        v.d = ld32(r, a + 208u);
    }
    __device__ static __forceinline__ void al16(const u32x4& v, uint32_t e, uint32_t s, uint32_t* o) {
        o[0] = __builtin_amdgcn_alignbyte(v.y, v.x, s);
        o[1] = __builtin_amdgcn_alignbyte(v.z, v.y, s);
        o[2] = __builtin_amdgcn_alignbyte(v.w, v.z, s);
        o[3] = __builtin_amdgcn_alignbyte(e, v.w, s);
    }
    __device__ static __forceinline__ void prep(const Raw& v, uint32_t ro, int g, int sb, Sc& sc) {
        const uint32_t s = (ro + static_cast<uint32_t>(sb) * 210u) & 2u;
        uint32_t y[2];
        realign(v.sc, s, y[0], y[1]);
        const float d = f16lo(v.d >> (8u * s));
        const uint32_t sh = 8u * static_cast<uint32_t>(g & 1);
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const int8_t c = static_cast<int8_t>(y[q >> 1] >> (sh + 16u * (q & 1)));
            const _Float16 w = static_cast<_Float16>(d * static_cast<float>(c));
            sc.ds[q] = half2_t{w, w};
        }
        al16(v.l0, v.l0e, s, sc.l0);
        al16(v.l1, v.l1e, s, sc.l1);
        al16(v.h, v.he, s, sc.h);
    }
    template <int S>
    __device__ static __forceinline__ void frags(const Raw&, const Sc& sc, int, const KqConsts& kc, Frag& lo,
                                                 Frag& hi) {
        constexpr int e = S >> 1, p = S & 1;
        q6k_frags(sc.l0 + 2 * e, sc.l1 + 2 * e, sc.h + 2 * e, p, sc.ds[2 * p], sc.ds[2 * p + 1], kc, lo, hi);
    }
};

// MFMAs per LDS stage: a buffer holds MB blocks x ts(MB) MFMAs x 1 KB <= 40 KB
constexpr int ts_of(int mb) { return mb <= 5 ? 8 : (mb <= 10 ? 4 : 2); }

// blocks per group of activation fragments (a divisor of MB)
constexpr int group_of(int mb) { return mb % 4 == 0 ? 4 : (mb % 3 == 0 ? 3 : (mb % 5 == 0 ? 5 : mb)); }

template <int N>
__device__ __forceinline__ void wait_vm_barrier() {
    // the wave's loads up to the last N have landed, then everyone's (a
    // __syncthreads would wait for the weight loads in flight too)
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_waitcnt(0x0F70 | (N & 15) | ((N >> 4) << 14));
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
}

// acc[b][f] += the tile's products over super-blocks [sb0, sb0 + cnt) of the
// row.  w0, w1 / ro0, ro1: matrix and this lane's row (byte offset) of the
// wave's two column fragments.  xs: the tile's packed activations (nblk >= 1
// blocks; blocks past them repeat the last one, into accumulators the caller
// drops).  iters >= cnt, the same in every wave of the workgroup (they share
// the barriers).  b0, b1: the K group's halves of the two LDS buffers, two
// __shared__ objects: the compiler's wait counting for LDS DMA tells objects
// apart, so reading one does not wait for the DMA into the other.  wn = the
// wave's place (0..3) in its K group.
//
// Per stage (ts_of(MB) MFMAs of a super-block): the stage's DMA has landed
// and everyone is done with the other buffer (one barrier), the next stage's
// DMA goes out into that buffer, and with a super-block's first stage the
// weight bytes of the next super-block.
template <int TYPE, int MB>
__device__ __forceinline__ void mainloop(float4_t (&acc)[MB][2], __amdgpu_buffer_rsrc_t w0, __amdgpu_buffer_rsrc_t w1,
                                         uint32_t ro0, uint32_t ro1, __amdgpu_buffer_rsrc_t xs, int nblk, int nsb,
                                         int sb0, int cnt, int iters, u32x4* b0, u32x4* b1, int wn) {
    using WT = W<TYPE>;
    constexpr int TS = ts_of(MB), Q = 8 / TS;  // stages per super-block
    constexpr int NC = MB * TS / 4;            // 1 KB pieces per wave and stage
    static_assert(MB * TS % 4 == 0 && MB * TS * 64 <= BUF_U4, "stage layout");
    const int lane = static_cast<int>(threadIdx.x) & 63, g = lane >> 4;
    const KqConsts kc = kq_consts();
    const int sb_last = nsb - 1;
    auto clamp_sb = [&](int it) __attribute__((always_inline)) -> int {
        const int sb = sb0 + it;
        return sb < sb_last ? sb : sb_last;
    };
    auto stage_in = [&](int it, int q, u32x4* dst) __attribute__((always_inline)) {
        const int sb = clamp_sb(it);
        typedef __attribute__((address_space(3))) void* lds_ptr;
#pragma unroll
        for (int i = 0; i < NC; i++) {
            const int c = wn + 4 * i, blk = c / TS, tt = c % TS;
            const int bc = blk < nblk ? blk : nblk - 1;
            const uint32_t so = static_cast<uint32_t>((bc * nsb + sb) * 8 + q * TS + tt) * 1024u;
            __builtin_amdgcn_raw_ptr_buffer_load_lds(xs, (lds_ptr)(dst + c * 64), 16, 16 * lane,
                                                     static_cast<int>(so), 0, 0);
        }
    };
    typename WT::Raw raw[2][2];
    typename WT::Sc sc[2];
    Frag bf[2][2][2];  // [pair parity][lo / hi][column fragment]
    auto load_w = [&](int it, auto p_c) __attribute__((always_inline)) {
        constexpr int p = decltype(p_c)::value;
        const int sb = clamp_sb(it);
        WT::load(w0, ro0, g, sb, raw[p][0]);
        WT::load(w1, ro1, g, sb, raw[p][1]);
    };
    // column fragment f of pair s, of the super-block in raw[p] (it: its
    // iteration); with the first pair of a super-block its scales
    auto decode = [&](int it, auto p_c, auto s_c, auto f_c) __attribute__((always_inline)) {
        constexpr int p = decltype(p_c)::value, s = decltype(s_c)::value, f = decltype(f_c)::value;
        if constexpr (s == 0) WT::prep(raw[p][f], f ? ro1 : ro0, g, clamp_sb(it), sc[f]);
        WT::template frags<s>(raw[p][f], sc[f], g, kc, bf[s & 1][0][f], bf[s & 1][1][f]);
    };
    // MFMAs 2 s, 2 s + 1 of a super-block, from fragments decoded before.  The
    // activation fragments come in groups of G blocks, a group read ahead of
    // the MFMAs that use it, and the next pair is decoded between the MFMAs of
    // the first two groups (the scheduling groups spell that order out: left
    // to itself the compiler reads one fragment, waits for it and multiplies,
    // and decodes in one run).
    constexpr int G = group_of(MB), NG = 2 * MB / G;
    Frag af[2][G];
    auto read = [&](const u32x4* buf, int tt, int n, Frag* f) __attribute__((always_inline)) {
        const int hl = n / (MB / G), blk = n % (MB / G) * G;
#pragma unroll
        for (int i = 0; i < G; i++) {
            const u32x4 v = buf[((blk + i) * TS + tt + hl) * 64 + lane];
            f[i].u[0] = v.x;
            f[i].u[1] = v.y;
            f[i].u[2] = v.z;
            f[i].u[3] = v.w;
        }
    };
    auto pair = [&](const u32x4* buf, int it, auto p_c, auto s_c) __attribute__((always_inline)) {
        constexpr int p = decltype(p_c)::value, s = decltype(s_c)::value;
        constexpr int tt = (2 * s) % TS;
        constexpr bool last = tt + 2 == TS;  // of the stage: the next pair's buffer is behind the barrier
        constexpr int np = s == 3 ? p ^ 1 : p, ns = (s + 1) & 3;
        if constexpr (tt == 0) {
            read(buf, tt, 0, af[0]);
            __builtin_amdgcn_sched_barrier(0);
        }
        static_assert(NG % 2 == 0, "the group buffers alternate");
#pragma unroll
        for (int n = 0; n < NG; n++) {
            if (n + 1 < NG) read(buf, tt, n + 1, af[(n + 1) & 1]);
            else if (!last) read(buf, tt + 2, 0, af[0]);
            if (n == 0)
                decode(s == 3 ? it + 1 : it, std::integral_constant<int, np>{}, std::integral_constant<int, ns>{},
                       std::integral_constant<int, 0>{});
            if (n == 1)
                decode(s == 3 ? it + 1 : it, std::integral_constant<int, np>{}, std::integral_constant<int, ns>{},
                       std::integral_constant<int, 1>{});
            const int hl = n / (MB / G), blk = n % (MB / G) * G;
#pragma unroll
            for (int i = 0; i < G; i++) {
                acc[blk + i][0] = mfma16x16x32(af[n & 1][i], bf[s & 1][hl][0], acc[blk + i][0]);
                acc[blk + i][1] = mfma16x16x32(af[n & 1][i], bf[s & 1][hl][1], acc[blk + i][1]);
            }
#pragma unroll
            for (int i = 0; i < 2 * G; i++) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);               // an MFMA,
                if (i < G) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);    // a read of the next group,
                if (n < 2) __builtin_amdgcn_sched_group_barrier(0x002, 4, 0);    // a few instructions of the decode
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    auto step = [&](int it, auto p_c) __attribute__((always_inline)) {
        constexpr int p = decltype(p_c)::value;
        auto stage = [&](auto q_c) __attribute__((always_inline)) {
            constexpr int q = decltype(q_c)::value;
            constexpr bool odd = ((Q == 1 ? p : q) & 1) != 0;
            const u32x4* cur = odd ? b1 : b0;
            u32x4* oth = odd ? b0 : b1;
            // loads issued after this stage's DMA: the weight bytes that go
            // out in a super-block's first stage
            wait_vm_barrier<(Q == 1 || q == 1) ? 2 * WT::kLoads : 0>();
            stage_in(q + 1 < Q ? it : it + 1, q + 1 < Q ? q + 1 : 0, oth);
            __builtin_amdgcn_sched_barrier(0);  // the DMA before the weight loads: the wait above counts on it
            if constexpr (q == 0) load_w(it + 1, std::integral_constant<int, p ^ 1>{});
            __builtin_amdgcn_sched_barrier(0);
            if (it < cnt) {
                pair(cur, it, p_c, std::integral_constant<int, q * TS / 2>{});
                if constexpr (TS >= 4) pair(cur, it, p_c, std::integral_constant<int, q * TS / 2 + (TS >= 4 ? 1 : 0)>{});
                if constexpr (TS == 8) {
                    pair(cur, it, p_c, std::integral_constant<int, TS == 8 ? 2 : 0>{});
                    pair(cur, it, p_c, std::integral_constant<int, TS == 8 ? 3 : 0>{});
                }
            }
        };
        stage(std::integral_constant<int, 0>{});
        if constexpr (Q > 1) stage(std::integral_constant<int, (Q > 1 ? 1 : 0)>{});
        if constexpr (Q > 2) {
            stage(std::integral_constant<int, (Q > 2 ? 2 : 0)>{});
            stage(std::integral_constant<int, (Q > 2 ? 3 : 0)>{});
        }
    };
    stage_in(0, 0, b0);
    __builtin_amdgcn_sched_barrier(0);
    load_w(0, std::integral_constant<int, 0>{});
    decode(0, std::integral_constant<int, 0>{}, std::integral_constant<int, 0>{}, std::integral_constant<int, 0>{});
    decode(0, std::integral_constant<int, 0>{}, std::integral_constant<int, 0>{}, std::integral_constant<int, 1>{});
    for (int it = 0; it < iters; it += 2) {
        step(it, std::integral_constant<int, 0>{});
        step(it + 1, std::integral_constant<int, 1>{});
    }
    // every DMA has landed before the buffers are used again or the wave ends
    wait_vm_barrier<0>();
}

}  // namespace wreg
}  // namespace vb
