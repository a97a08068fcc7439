// Weight types of the small-batch kernels: one lane's share of a 128-element
// step of a weight row (16 rows per fragment: lane (j, g) = row j, lane group
// g), read from memory (issue) or from a 16-byte-aligned image of the rows in
// LDS (read, ro = the row's offset in it), and decoded into the step's four B
// fragments (decode).  rowoff = the row's byte offset in the tensor, or any
// offset equal to it modulo 4.
#pragma once

#include "mfma_q4k.hpp"

namespace vb {

template <class V>
__device__ __forceinline__ V lds_at(const uint8_t* p) {
    return *reinterpret_cast<const V*>(p);
}
__device__ __forceinline__ u32x3 lds96(const uint8_t* p) {
    return u32x3{lds_at<uint32_t>(p), lds_at<uint32_t>(p + 4), lds_at<uint32_t>(p + 8)};
}

template <int TYPE> struct Kq;

// Q4_K (cpp/src/dequant.cpp:258-301; header d, dmin, scales[12] @0, qs[128]
// @16, rows 16-byte aligned): a step is half a super-block, chunks c = 2 h
// and 2 h + 1; k-step 2 (c - 2 h) takes the low nibbles of qs bytes
// [32 c + 8 g, +8) (sub-block 2 c), k-step 2 (c - 2 h) + 1 their high
// nibbles (sub-block 2 c + 1).
template <>
struct Kq<TYPE_Q4_K> {
    static constexpr bool kBlockLane = false;
    struct Raw {
        u32x4 hd;
        uint2 q[2];
    };
    __device__ static __forceinline__ void issue(__amdgpu_buffer_rsrc_t w, uint32_t rowoff, int step, int g,
                                                 Raw& r) {
        const uint32_t base = rowoff + static_cast<uint32_t>(step >> 1) * 144u;
        const uint32_t qo = base + 16u + 64u * static_cast<uint32_t>(step & 1) + 8u * static_cast<uint32_t>(g);
        r.hd = buf_ld128(w, base, 0);
#pragma unroll
        for (int c = 0; c < 2; c++) {
            const auto v = __builtin_amdgcn_raw_buffer_load_b64(w, static_cast<int>(qo + 32u * c), 0, 0);
            r.q[c] = make_uint2(v[0], v[1]);
        }
    }
    __device__ static __forceinline__ void decode(const Raw& r, uint32_t, int step, int, const KqConsts&, Frag* f) {
        const uint4 hd = make_uint4(r.hd.x, r.hd.y, r.hd.z, r.hd.w);
#pragma unroll
        for (int c = 0; c < 2; c++) {
            half2_t ds[2], nm[2];
            q4k_chunk_scales(hd, 2 * (step & 1) + c, ds, nm);
            q4k_bfrags_nat(r.q[c].x, r.q[c].y, ds, nm, f[2 * c], f[2 * c + 1]);
        }
    }
};

// Q5_K (super-block of 256, 176 bytes: the Q4_K header d, dmin, scales[12]
// @0, qh[32] @16, qs[128] @48; rows 16-byte aligned): a step is half a
// super-block, chunks c = 2 h and 2 h + 1, as for Q4_K; lane group g also
// takes qh bytes [8 g, +8), whose bits 2 c, 2 c + 1 are the fifth bits of the
// chunk's two sub-blocks (q5k_frags).
template <>
struct Kq<TYPE_Q5_K> {
    static constexpr bool kBlockLane = false;
    struct Raw {
        u32x4 hd;
        uint2 q[2];
        uint2 h;
    };
    __device__ static __forceinline__ void issue(__amdgpu_buffer_rsrc_t w, uint32_t rowoff, int step, int g,
                                                 Raw& r) {
        const uint32_t base = rowoff + static_cast<uint32_t>(step >> 1) * 176u;
        const uint32_t g8 = 8u * static_cast<uint32_t>(g);
        const uint32_t qo = base + 48u + 64u * static_cast<uint32_t>(step & 1) + g8;
        r.hd = buf_ld128(w, base, 0);
#pragma unroll
        for (int c = 0; c < 2; c++) {
            const auto v = __builtin_amdgcn_raw_buffer_load_b64(w, static_cast<int>(qo + 32u * c), 0, 0);
            r.q[c] = make_uint2(v[0], v[1]);
        }
        const auto v = __builtin_amdgcn_raw_buffer_load_b64(w, static_cast<int>(base + 16u + g8), 0, 0);
        r.h = make_uint2(v[0], v[1]);
    }
    __device__ static __forceinline__ void read(const uint8_t* img, uint32_t ro, int step, int g, Raw& r) {
        const uint8_t* b = img + (ro + static_cast<uint32_t>(step >> 1) * 176u);
        r.hd = lds_at<u32x4>(b);
#pragma unroll
        for (int c = 0; c < 2; c++) r.q[c] = lds_at<uint2>(b + 48 + 64 * (step & 1) + 8 * g + 32 * c);
        r.h = lds_at<uint2>(b + 16 + 8 * g);
    }
    __device__ static __forceinline__ void decode(const Raw& r, uint32_t, int step, int, const KqConsts& kc,
                                                  Frag* f) {
        const uint4 hd = make_uint4(r.hd.x, r.hd.y, r.hd.z, r.hd.w);
#pragma unroll
        for (int c = 0; c < 2; c++) {
            const int cc = 2 * (step & 1) + c;
            half2_t ds[2], nm[2];
            q4k_chunk_scales(hd, cc, ds, nm);
            q5k_frags(r.q[c].x, r.q[c].y, r.h.x, r.h.y, static_cast<uint32_t>(cc), ds, nm, kc, f[2 * c],
                      f[2 * c + 1]);
        }
    }
};

// Q6_K in the GGUF layout (the layout of real files and of the known answers
// in tests/test_kquants.py:134-175; cpp/src/dequant.cpp:359-402 gathers the
// elements in another order): super-block of 256 = two halves h of 128
// elements; bytes ql[128] @0, qh[64] @128, int8
// scales[16] @192, fp16 d @208.  In half h, element l + 32 t (l < 32, t < 4)
// is q - 32 with q = (ql[64 h + l + 32 (t & 1)] >> 4 (t >> 1)) & 15 |
// ((qh[32 h + l] >> 2 t) & 3) << 4, scaled by d * scales[8 h + l / 16 + 2 t].
// A step is one half; k-step ks = t, so lane (j, g) needs ql bytes
// [64 h + 8 g, +8) (t = 0, 2) and [64 h + 32 + 8 g, +8) (t = 1, 3), qh bytes
// [32 h + 8 g, +8), the scales 8 h + g / 2 + 2 t and d.
template <>
struct Kq<TYPE_Q6_K> {
    static constexpr bool kBlockLane = false;
    struct Raw {
        u32x3 l0, l1, qh;
        uint32_t sd;  // lane group g: dword g of (scales of the half: 12 bytes from their dword, d's dword)
    };
    // every field offset is a multiple of 4 from the super-block start, so
    // one shift (the start's offset within its dword) serves all of them
    __device__ static __forceinline__ uint32_t shift(uint32_t rowoff, int step) {
        return (rowoff + static_cast<uint32_t>(step >> 1) * 210u) & 3u;
    }
    __device__ static __forceinline__ void issue(__amdgpu_buffer_rsrc_t w, uint32_t rowoff, int step, int g,
                                                 Raw& r) {
        const uint32_t base = (rowoff + static_cast<uint32_t>(step >> 1) * 210u) & ~3u;
        const uint32_t h = static_cast<uint32_t>(step & 1), g8 = 8u * static_cast<uint32_t>(g);
        r.l0 = ld96(w, base + 64u * h + g8);
        r.l1 = ld96(w, base + 64u * h + 32u + g8);
        r.qh = ld96(w, base + 128u + 32u * h + g8);
        // the four lane groups of a row share its scales and d: one dword each
        r.sd = ld32(w, g < 3 ? base + 192u + 8u * h + 4u * static_cast<uint32_t>(g) : base + 208u);
    }
    __device__ static __forceinline__ void read(const uint8_t* img, uint32_t ro, int step, int g, Raw& r) {
        const uint8_t* b = img + ((ro + static_cast<uint32_t>(step >> 1) * 210u) & ~3u);
        const int h = step & 1;
        r.l0 = lds96(b + 64 * h + 8 * g);
        r.l1 = lds96(b + 64 * h + 32 + 8 * g);
        r.qh = lds96(b + 128 + 32 * h + 8 * g);
        r.sd = lds_at<uint32_t>(g < 3 ? b + 192 + 8 * h + 4 * g : b + 208);
    }
    __device__ static __forceinline__ void decode(const Raw& r, uint32_t rowoff, int step, int g, const KqConsts& kc,
                                                  Frag* f) {
        const uint32_t sh = shift(rowoff, step);
        // scale dwords 0-2 and d's dword from lane groups 0-3: the pair's
        // even / odd 16-lane rows, then the lower / upper halves of the wave
        const auto p16 = __builtin_amdgcn_permlane16_swap(r.sd, r.sd, false, false);
        const auto e32 = __builtin_amdgcn_permlane32_swap(p16[0], p16[0], false, false);
        const auto o32 = __builtin_amdgcn_permlane32_swap(p16[1], p16[1], false, false);
        const u32x3 scw = {e32[0], o32[0], e32[1]};
        uint32_t l0[2], l1[2], qh[2], sc[2];
        realign(r.l0, sh, l0[0], l0[1]);
        realign(r.l1, sh, l1[0], l1[1]);
        realign(r.qh, sh, qh[0], qh[1]);
        realign(scw, sh, sc[0], sc[1]);
        const float d = f16lo(o32[1] >> (8u * sh));
        // scale bytes g / 2 + {0, 2, 4, 6} of the half's eight
        const uint32_t P = __builtin_amdgcn_perm(sc[1], sc[0], g >= 2 ? 0x07050301u : 0x06040200u);
        half2_t dsc[4];
#pragma unroll
        for (int t = 0; t < 4; t++) {
            const int8_t s = static_cast<int8_t>((P >> (8 * t)) & 0xFFu);
            const _Float16 v = static_cast<_Float16>(d * static_cast<float>(s));
            dsc[t] = half2_t{v, v};
        }
        const half2_t k1056 = half2_t{static_cast<_Float16>(1056.0f), static_cast<_Float16>(1056.0f)};
#pragma unroll
        for (int dw = 0; dw < 2; dw++) {
            // four 6-bit codes per dword: run t takes nibble t / 2 of l0 (t
            // even) or l1 (t odd) and qh bits 2 t, 2 t + 1, moved to bits 4, 5
            // of the same byte
            uint32_t q[4];
            q[0] = ((qh[dw] << 4) & 0x30303030u) | (l0[dw] & 0x0F0F0F0Fu);
            q[1] = ((qh[dw] << 2) & 0x30303030u) | (l1[dw] & 0x0F0F0F0Fu);
            q[2] = (qh[dw] & 0x30303030u) | ((l0[dw] >> 4) & 0x0F0F0F0Fu);
            q[3] = ((qh[dw] >> 2) & 0x30303030u) | ((l1[dw] >> 4) & 0x0F0F0F0Fu);
#pragma unroll
            for (int t = 0; t < 4; t++) {
                // bytes (0, 1) and (2, 3) into fp16 halves 1024 + q (exact)
                f[t].u[2 * dw] = h2bits((bits2h(__builtin_amdgcn_perm(kc.h64, q[t], 0x07010500u)) - k1056) * dsc[t]);
                f[t].u[2 * dw + 1] =
                    h2bits((bits2h(__builtin_amdgcn_perm(kc.h64, q[t], 0x07030502u)) - k1056) * dsc[t]);
            }
        }
    }
};

// Q8_0 in the GGUF layout (vibeblade/loader.py:129-133,
// cpp/src/cuda_kernels.cu:718-735): blocks of 32 = fp16 d @0, int8 qs[32]
// @2.  A step is four blocks.  Lane group g takes block 4 s + g whole (one
// 34-byte read, one scale) and k-step ks its codes [8 ks, +8): the "block
// per lane group" k order, which the activation fragments follow (kBlockLane).
// Rows are whole dwords (K % 128 == 0: 136-byte steps), so block g starts
// 2 g bytes into a dword modulo 4.
template <>
struct Kq<TYPE_Q8_0> {
    static constexpr bool kBlockLane = true;
    struct Raw {
        u32x3 q[3];  // 36 bytes from the block's dword
    };
    __device__ static __forceinline__ void issue(__amdgpu_buffer_rsrc_t w, uint32_t rowoff, int step, int g,
                                                 Raw& r) {
        const uint32_t a = (rowoff + static_cast<uint32_t>(step) * 136u + 34u * static_cast<uint32_t>(g)) & ~3u;
#pragma unroll
        for (int i = 0; i < 3; i++) r.q[i] = ld96(w, a + 12u * i);
    }
    __device__ static __forceinline__ void read(const uint8_t* img, uint32_t ro, int step, int g, Raw& r) {
        const uint8_t* b = img + ((ro + static_cast<uint32_t>(step) * 136u + 34u * static_cast<uint32_t>(g)) & ~3u);
#pragma unroll
        for (int i = 0; i < 3; i++) r.q[i] = lds96(b + 12 * i);
    }
    __device__ static __forceinline__ void decode(const Raw& r, uint32_t rowoff, int, int g, const KqConsts& kc,
                                                  Frag* f) {
        const uint32_t w[9] = {r.q[0].x, r.q[0].y, r.q[0].z, r.q[1].x, r.q[1].y, r.q[1].z, r.q[2].x, r.q[2].y,
                               r.q[2].z};
        const bool odd = ((rowoff + 2u * static_cast<uint32_t>(g)) & 3u) != 0;  // block at byte 2 of its dword
        // d at bytes [0, 2) or [2, 4); codes at byte 2 (realign by 2) or 4 (dword 1)
        const uint32_t d16 = odd ? (w[0] >> 16) : (w[0] & 0xFFFFu);
        const half2_t dd = bits2h(d16 | (d16 << 16));
        const half2_t k1152 = half2_t{static_cast<_Float16>(1152.0f), static_cast<_Float16>(1152.0f)};
#pragma unroll
        for (int ks = 0; ks < 4; ks++) {
            uint32_t qs[2];
#pragma unroll
            for (int h = 0; h < 2; h++) {
                const int i = 2 * ks + h;
                qs[h] = odd ? w[i + 1] : __builtin_amdgcn_alignbyte(w[i + 1], w[i], 2u);
            }
#pragma unroll
            for (int i = 0; i < 4; i++) {
                // bytes (b0, b1) into the two halves; (b ^ 0x80) | 0x6400 is
                // the half 1024 + q + 128 (exact)
                const uint32_t src = __builtin_amdgcn_perm(0u, qs[i >> 1], (i & 1) ? 0x0C030C02u : 0x0C010C00u);
                f[ks].u[i] = h2bits((bits2h(src ^ kc.x80) - k1152) * dd);
            }
        }
    }
};

// Q4_0 / Q4_1 / Q5_0 / Q5_1 (B32 in mfma_q4k.hpp): as Q8_0, a step is four
// blocks, lane group g takes block 4 s + g whole and k-step ks its codes
// [8 ks, +8) (kBlockLane).  The block (18-24 bytes) is read as the six
// dwords from its start rounded down to 4 (rows are multiples of 8 bytes at
// K % 128 == 0, so 18- and 22-byte blocks start 2 (g % 2) bytes into a
// dword) and realigned.
template <int TYPE>
struct KqB32 {
    static constexpr bool kBlockLane = true;
    using B = B32<TYPE>;
    struct Raw {
        u32x3 q[2];
    };
    __device__ static __forceinline__ void issue(__amdgpu_buffer_rsrc_t w, uint32_t rowoff, int step, int g,
                                                 Raw& r) {
        const uint32_t a = (rowoff + (4u * static_cast<uint32_t>(step) + static_cast<uint32_t>(g)) * B::kBytes) & ~3u;
        r.q[0] = ld96(w, a);
        r.q[1] = ld96(w, a + 12u);
    }
    __device__ static __forceinline__ void decode(const Raw& r, uint32_t rowoff, int, int g, const KqConsts& kc,
                                                  Frag* f) {
        const uint32_t w[6] = {r.q[0].x, r.q[0].y, r.q[0].z, r.q[1].x, r.q[1].y, r.q[1].z};
        const uint32_t sh = (rowoff + static_cast<uint32_t>(g) * B::kBytes) & 3u;  // 0 or 2
#pragma unroll
        for (int ks = 0; ks < 4; ks++) b32_block_frag<TYPE>(w, sh, ks, kc, f[ks]);
    }
};
template <> struct Kq<TYPE_Q4_0> : KqB32<TYPE_Q4_0> {};
template <> struct Kq<TYPE_Q4_1> : KqB32<TYPE_Q4_1> {};
template <> struct Kq<TYPE_Q5_0> : KqB32<TYPE_Q5_0> {};
template <> struct Kq<TYPE_Q5_1> : KqB32<TYPE_Q5_1> {};

}  // namespace vb
