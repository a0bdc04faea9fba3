// Packed weights by lanes: how one lane loads and decodes 64 weights of a 256-element super-block, for the kernels whose
// lanes need whole runs of a row (gemm_skinny.hip: bf16 operands; gemv_few.hip: fp32 operands). Every format's K is in whole
// super-blocks here; the formats of 32-element blocks take eight of them as one. The decode is the block arithmetic of the
// reference (code * (d * sc) - dmin * m and its siblings) in fp32.
#pragma once
#include "common.h"

namespace skh {

typedef __bf16 skn_bf16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 skn_h2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ uint32_t skn_pack(float a, float b) { return __builtin_bit_cast(uint32_t, skn_bf16x2{(__bf16)a, (__bf16)b}); }

// Element offset inside a super-block of the eight elements of step u (0..7) of lane group q (0..3): a lane's 64 weights are
// consecutive, or for Q6_K, whose bytes interleave quarters, eight runs of eight.
template <bool Q6>
__device__ __forceinline__ int skn_elem(int q, int u) {
    return Q6 ? 128 * (q >> 1) + 32 * (u >> 1) + 16 * (q & 1) + 8 * (u & 1) : 64 * q + 8 * u;
}

// Where a decode leaves its eight weights: as four dwords of bf16 pairs (nearest even), or as they are.
struct SknBf16 {
    uint32_t o[4];
    __device__ __forceinline__ void four(int i, float a, float b, float c, float d) { o[2 * i] = skn_pack(a, b); o[2 * i + 1] = skn_pack(c, d); }
};
struct SknF32 {
    float w[8];
    __device__ __forceinline__ void four(int i, float a, float b, float c, float d) { w[4 * i] = a; w[4 * i + 1] = b; w[4 * i + 2] = c; w[4 * i + 3] = d; }
};

// ---------------------------------------------------------------------------------------------- weight formats
// Per format: Raw (the bytes a lane needs of one super-block of one row), load, Scales (worked out once per super-block),
// and decode<U>: the eight weights of step U.
template <int I> __device__ __forceinline__ float skn_byte(uint32_t v) { return ubyte_to_float<I>(v); }
// four codes, one per byte, times scale plus add
template <class O> __device__ __forceinline__ void skn_bytes4(uint32_t v, float scale, float add, O& o, int i) {
    o.four(i, fmaf(skn_byte<0>(v), scale, add), fmaf(skn_byte<1>(v), scale, add), fmaf(skn_byte<2>(v), scale, add), fmaf(skn_byte<3>(v), scale, add));
}
// The four codes of one nibble plane of a dword (PLANE 0: low nibbles, 1: high): masked into 16-bit fields they are the fp16
// subnormals code * 2^-24 (2^-20), which the mixed-precision multiply-add widens exactly; `scale` carries the power of two.
template <int PLANE, class O>
__device__ __forceinline__ void skn_nibbles4(uint32_t c, float scale, float add, O& o, int i) {
    constexpr uint32_t mask = PLANE ? 0x00F000F0u : 0x000F000Fu;
    const skn_h2 b02 = __builtin_bit_cast(skn_h2, c & mask), b13 = __builtin_bit_cast(skn_h2, (c >> 8) & mask);
    o.four(i, fmaf((float)b02.x, scale, add), fmaf((float)b13.x, scale, add), fmaf((float)b02.y, scale, add), fmaf((float)b13.y, scale, add));
}
constexpr float SKN_2P24 = 16777216.0f, SKN_2P20 = 1048576.0f;

// d * sc and dmin * m of sub-blocks 2 q and 2 q + 1 from a K-quant header (ggml get_scale_min_k4)
struct SknK4 { float s0, s1, m0, m1; };
__device__ __forceinline__ SknK4 skn_k4(const uint4& hdr, int q) {
    const float d = half_bits_to_float_fast(hdr.x & 0xFFFFu), dmin = half_bits_to_float_fast(hdr.x >> 16);
    const uint32_t sc_lo = hdr.y & 0x3F3F3F3Fu, mn_lo = hdr.z & 0x3F3F3F3Fu;
    const uint32_t sc_hi = (hdr.w & 0x0F0F0F0Fu) | ((hdr.y >> 2) & 0x30303030u), mn_hi = ((hdr.w >> 4) & 0x0F0F0F0Fu) | ((hdr.z >> 2) & 0x30303030u);
    const int sh = 16 * (q & 1);
    const uint32_t sc = (q < 2 ? sc_lo : sc_hi) >> sh, mn = (q < 2 ? mn_lo : mn_hi) >> sh;
    return SknK4{d * (float)(sc & 0xFFu), d * (float)((sc >> 8) & 0xFFu), dmin * (float)(mn & 0xFFu), dmin * (float)((mn >> 8) & 0xFFu)};
}

struct SknQ4K {
    static constexpr int BYTES = Q4K_BYTES;
    static constexpr bool Q6 = false;
    struct Raw { uint4 hdr; uint32_t c[8]; };
    struct Scales { float s0, a0, s1, a1; };
    static __device__ __forceinline__ void load(Raw& r, const uint8_t* blk, int q) {
        r.hdr = *reinterpret_cast<const uint4*>(blk);
        const uint4 a = *reinterpret_cast<const uint4*>(blk + 16 + 32 * q), b = *reinterpret_cast<const uint4*>(blk + 32 + 32 * q);
        r.c[0] = a.x; r.c[1] = a.y; r.c[2] = a.z; r.c[3] = a.w; r.c[4] = b.x; r.c[5] = b.y; r.c[6] = b.z; r.c[7] = b.w;
    }
    static __device__ __forceinline__ Scales scales(const Raw& r, int q) {
        const SknK4 k = skn_k4(r.hdr, q);
        return Scales{k.s0 * SKN_2P24, -k.m0, k.s1 * SKN_2P20, -k.m1};
    }
    template <int U, class O> static __device__ __forceinline__ void decode(const Raw& r, const Scales& s, O& o) {
        const uint32_t c0 = r.c[2 * (U & 3)], c1 = r.c[2 * (U & 3) + 1];
        if constexpr (U < 4) { skn_nibbles4<0>(c0, s.s0, s.a0, o, 0); skn_nibbles4<0>(c1, s.s0, s.a0, o, 1); }
        else { skn_nibbles4<1>(c0, s.s1, s.a1, o, 0); skn_nibbles4<1>(c1, s.s1, s.a1, o, 1); }
    }
};
struct SknQ5K {
    static constexpr int BYTES = Q5K_BYTES;
    static constexpr bool Q6 = false;
    struct Raw { uint4 hdr; uint32_t c[8], h[8]; };
    struct Scales { float s0, a0, s1, a1; int bit; };
    static __device__ __forceinline__ void load(Raw& r, const uint8_t* blk, int q) {
        r.hdr = *reinterpret_cast<const uint4*>(blk);
        const uint4 h0 = *reinterpret_cast<const uint4*>(blk + 16), h1 = *reinterpret_cast<const uint4*>(blk + 32);
        const uint4 a = *reinterpret_cast<const uint4*>(blk + 48 + 32 * q), b = *reinterpret_cast<const uint4*>(blk + 64 + 32 * q);
        r.c[0] = a.x; r.c[1] = a.y; r.c[2] = a.z; r.c[3] = a.w; r.c[4] = b.x; r.c[5] = b.y; r.c[6] = b.z; r.c[7] = b.w;
        r.h[0] = h0.x; r.h[1] = h0.y; r.h[2] = h0.z; r.h[3] = h0.w; r.h[4] = h1.x; r.h[5] = h1.y; r.h[6] = h1.z; r.h[7] = h1.w;
    }
    static __device__ __forceinline__ Scales scales(const Raw& r, int q) {
        const SknK4 k = skn_k4(r.hdr, q);
        return Scales{k.s0, -k.m0, k.s1, -k.m1, 2 * q};
    }
    template <int U, class O> static __device__ __forceinline__ void decode(const Raw& r, const Scales& s, O& o) {
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const int at = 2 * (U & 3) + i;
            const uint32_t v = ((r.c[at] >> (U < 4 ? 0 : 4)) & 0x0F0F0F0Fu) | (((r.h[at] >> (s.bit + (U < 4 ? 0 : 1))) & 0x01010101u) << 4);
            skn_bytes4(v, U < 4 ? s.s0 : s.s1, U < 4 ? s.a0 : s.a1, o, i);
        }
    }
};
// 16 bytes from an address that is 0 or 2 bytes past a dword boundary (`odd`): dword-aligned loads and a byte shift. A
// 16-byte load at an odd half-word address takes the memory pipe about twice as long (Q8_0, 32 x 4096 x 4096: 14.5 us with
// such loads, 11.3 with these). With an even address the fifth dword is the fourth again: nothing past the run is read.
struct SknQ6K {
    static constexpr int BYTES = Q6K_BYTES;
    static constexpr bool Q6 = true;
    struct Raw { u32x4_vec a, b, h; u32x2_vec sc; uint32_t a4, b4, h4, sc2, d; int odd; };
    struct Scales { float s[4]; uint32_t a[4], b[4], h[4]; };
    static __device__ __forceinline__ void run(u32x4_vec& v, uint32_t& last, const uint8_t* base, int odd) {
        v = load_u32x4_a4(base);
        last = *reinterpret_cast<const uint32_t*>(base + 12 + 4 * odd);
    }
    static __device__ __forceinline__ void load(Raw& r, const uint8_t* blk, int q) {
        const int half = q >> 1, off = 16 * (q & 1);
        r.odd = (int)(reinterpret_cast<uintptr_t>(blk) >> 1) & 1;
        const uint8_t* base = blk - 2 * r.odd;
        run(r.a, r.a4, base + 64 * half + off, r.odd);
        run(r.b, r.b4, base + 64 * half + 32 + off, r.odd);
        run(r.h, r.h4, base + 128 + 32 * half + off, r.odd);
        const uint32_t* sc = reinterpret_cast<const uint32_t*>(base + 192 + 8 * half);
        r.sc = u32x2_vec{sc[0], sc[1]};
        r.sc2 = sc[1 + r.odd];
        r.d = load_u16(blk + 208);
    }
    static __device__ __forceinline__ void align(uint32_t (&o)[4], const u32x4_vec& v, uint32_t last, uint32_t sh) {
        o[0] = __builtin_amdgcn_alignbyte(v.y, v.x, sh);
        o[1] = __builtin_amdgcn_alignbyte(v.z, v.y, sh);
        o[2] = __builtin_amdgcn_alignbyte(v.w, v.z, sh);
        o[3] = __builtin_amdgcn_alignbyte(last, v.w, sh);
    }
    static __device__ __forceinline__ Scales scales(const Raw& r, int q) {
        const float d = half_bits_to_float_fast(r.d);
        const uint32_t sh = 2 * r.odd, s0 = __builtin_amdgcn_alignbyte(r.sc.y, r.sc.x, sh), s1 = __builtin_amdgcn_alignbyte(r.sc2, r.sc.y, sh);
        const int b = 8 * (q & 1);
        Scales s{{d * (float)(int8_t)(s0 >> b), d * (float)(int8_t)(s0 >> (16 + b)), d * (float)(int8_t)(s1 >> b), d * (float)(int8_t)(s1 >> (16 + b))}, {}, {}, {}};
        align(s.a, r.a, r.a4, sh); align(s.b, r.b, r.b4, sh); align(s.h, r.h, r.h4, sh);
        return s;
    }
    template <int U, class O> static __device__ __forceinline__ void decode(const Raw&, const Scales& s, O& o) {
        constexpr int Q = U >> 1, E = 2 * (U & 1);
        const float sc = s.s[Q], add = -32.f * sc;
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const uint32_t l = (Q & 1) ? s.b[E + i] : s.a[E + i];
            const uint32_t v = ((l >> (Q < 2 ? 0 : 4)) & 0x0F0F0F0Fu) | (((s.h[E + i] >> (2 * Q)) & 0x03030303u) << 4);
            skn_bytes4(v, sc, add, o, i);
        }
    }
};
// The formats of 32-element blocks: a lane's two blocks are 68, 36, 44 or 48 consecutive bytes from a dword boundary, and
// the second block's codes lie on dwords themselves; the first block's are shifted into place (Q5_1: no shift).
struct SknQ80 {
    static constexpr int BYTES = 8 * Q80_BYTES;
    static constexpr bool Q6 = false;
    struct Raw { uint32_t v[17]; };
    struct Scales { float d[2]; };
    static __device__ __forceinline__ void load(Raw& r, const uint8_t* blk, int q) {
        const uint8_t* b = blk + 68 * q;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const u32x4_vec x = load_u32x4_a4(b + 16 * i);
            r.v[4 * i] = x.x; r.v[4 * i + 1] = x.y; r.v[4 * i + 2] = x.z; r.v[4 * i + 3] = x.w;
        }
        r.v[16] = *reinterpret_cast<const uint32_t*>(b + 64);
    }
    static __device__ __forceinline__ Scales scales(const Raw& r, int) { return Scales{{half_bits_to_float_fast(r.v[0] & 0xFFFFu), half_bits_to_float_fast(r.v[8] >> 16)}}; }
    template <int U, class O> static __device__ __forceinline__ void decode(const Raw& r, const Scales& s, O& o) {
        const float d = s.d[U >> 2];
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const uint32_t v = U < 4 ? __builtin_amdgcn_alignbyte(r.v[2 * U + i + 1], r.v[2 * U + i], 2) : r.v[2 * U + i + 1];
            o.four(i, (float)(int8_t)v * d, (float)(int8_t)(v >> 8) * d, (float)(int8_t)(v >> 16) * d, (float)(int8_t)(v >> 24) * d);
        }
    }
};
// Q4_0 / Q5_0 / Q5_1 (FMT 0 / 1 / 2): low nibbles of the 16 code bytes are elements 0..15 of a block, high nibbles 16..31
template <int FMT> struct SknQ45 {
    static constexpr int BB = FMT == 0 ? Q40_BYTES : FMT == 1 ? Q50_BYTES : Q51_BYTES;
    static constexpr int BYTES = 8 * BB, DWORDS = BB / 2;
    static constexpr bool Q6 = false;
    struct Raw { uint32_t v[DWORDS]; };
    struct Scales { float d[2], add[2]; uint32_t h[2]; };
    static __device__ __forceinline__ void load(Raw& r, const uint8_t* blk, int q) {
        const uint8_t* b = blk + 2 * BB * q;
#pragma unroll
        for (int i = 0; i < DWORDS / 4; ++i) {
            const u32x4_vec x = load_u32x4_a4(b + 16 * i);
            r.v[4 * i] = x.x; r.v[4 * i + 1] = x.y; r.v[4 * i + 2] = x.z; r.v[4 * i + 3] = x.w;
        }
#pragma unroll
        for (int i = DWORDS / 4 * 4; i < DWORDS; ++i) r.v[i] = reinterpret_cast<const uint32_t*>(b)[i];
    }
    static __device__ __forceinline__ Scales scales(const Raw& r, int) {
        Scales s;
        const uint32_t d0 = r.v[0] & 0xFFFFu, d1 = FMT == 0 ? r.v[4] >> 16 : FMT == 1 ? r.v[5] >> 16 : r.v[6] & 0xFFFFu;
        s.d[0] = half_bits_to_float_fast(d0);
        s.d[1] = half_bits_to_float_fast(d1);
        s.add[0] = FMT == 0 ? -8.f * s.d[0] : FMT == 1 ? -16.f * s.d[0] : half_bits_to_float_fast(r.v[0] >> 16);
        s.add[1] = FMT == 0 ? -8.f * s.d[1] : FMT == 1 ? -16.f * s.d[1] : half_bits_to_float_fast(r.v[FMT == 2 ? 6 : 0] >> 16);
        s.h[0] = FMT == 1 ? __builtin_amdgcn_alignbyte(r.v[1], r.v[0], 2) : r.v[1];
        s.h[1] = FMT == 1 ? r.v[6] : r.v[FMT == 2 ? 7 : 1];
        return s;
    }
    template <int B> static __device__ __forceinline__ uint32_t code_dword(const Raw& r, int e) {      // dword e of block B's 16 code bytes
        if constexpr (FMT == 2) return r.v[6 * B + 2 + e];
        else if constexpr (B == 1) return r.v[(FMT == 0 ? 5 : 7) + e];
        else return __builtin_amdgcn_alignbyte(r.v[(FMT == 0 ? 1 : 2) + e], r.v[(FMT == 0 ? 0 : 1) + e], 2);
    }
    template <int U, class O> static __device__ __forceinline__ void decode(const Raw& r, const Scales& s, O& o) {
        constexpr int B = U >> 2, P = (U >> 1) & 1, E = 2 * (U & 1);       // block, nibble plane, first code dword
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const uint32_t c = code_dword<B>(r, E + i);
            if constexpr (FMT == 0) skn_nibbles4<P>(c, s.d[B] * (P ? SKN_2P20 : SKN_2P24), s.add[B], o, i);
            else {
                const uint32_t v = ((c >> (4 * P)) & 0x0F0F0F0Fu) | (((((s.h[B] >> (8 * (U & 3) + 4 * i)) & 0xFu) * 0x00204081u) & 0x01010101u) << 4);
                skn_bytes4(v, s.d[B], s.add[B], o, i);
            }
        }
    }
};

}  // namespace skh
