// Packed-weight GEMM for prompts and batches of few rows (9 to about 128), every format:
//   C[m, n] = sum_k A[m, k] * dequant(W[n, k]),  A fp32 [M, K] rounded to bf16 once, W packed in canonical row-major GGUF
//   order, products bf16 x bf16 on v_mfma_f32_16x16x32_bf16, fp32 accumulation, C fp32 [M, N].
// The decode is the block arithmetic of the reference (code * (d * sc) - dmin * m and its siblings) in fp32, rounded to
// bf16 (nearest even). Semantics: m rows = m scalar GEMVs,
//   skainet-backends/skainet-backend-cpu/src/commonMain/kotlin/sk/ainet/exec/kernel/PackedViewMatmulKernel.kt:69-108.
//
// What bounds it: every weight is decoded once per row block (2.3 to 3.7 vector instructions each), the weight is read
// once, and a workgroup reads its rows' activations for every 16 NT columns. The 256- and 128-row tiles of the other
// kernels spend their matrix work, their activation traffic and their LDS round trips on rows that do not exist here.
//   * A workgroup owns 16 MT rows x 16 NT columns; its NW waves split K by 256-element super-blocks (w, w + NW, ...).
//   * Lane (c, q) = (l % 16, l / 16) of a wave holds, of each of its NT weight rows c, the 64 weights of the super-block
//     that its own B operands need: it loads their bytes straight from memory (48 to 80 bytes in 16-byte loads; the four
//     lanes of a row read one consecutive run), decodes eight of them per matrix instruction, and no weight passes
//     through LDS. The compiler moves the request for the next super-block down to its use; held in front of the current
//     one it takes 200 registers instead of 120, two waves per SIMD instead of four: 24 x 14336 x 4096 15.4 -> 20.5 us.
//   * The contraction index is a free permutation as long as both operands agree: step u (0..7) of a super-block takes,
//     from lane q, elements 64 q + 8 u .. + 7 (a lane owns 64 consecutive elements), or for Q6_K, whose bytes interleave
//     quarters, 128 (q / 2) + 32 (u / 2) + 16 (q % 2) + 8 (u % 2) .. + 7. The pass in front writes the activations in that
//     order, 1 KB of consecutive memory per (16 rows, step), so an A operand is one 16-byte load per lane.
//   * The waves' partial tiles meet in LDS once; residual or SwiGLU are applied where the sums are stored.
// Measured (product and pass in front): Q4_K 24 x 14336 x 4096 22.4 -> 17 us (the weight in 8 us behind two
// launches of 2.75), 64 x 4096 x 4096 19.5 -> 10.8, 9 x 4096 x 14336 27.8 -> 13.6; Q8_0 64 x 4096 x 4096 21.4 -> 14.1.
#include "packed_lane64.h"

#include <cmath>
#include <type_traits>

namespace skh {

typedef __bf16 skn_bf16x8 __attribute__((ext_vector_type(8)));
typedef float skn_f32x4 __attribute__((ext_vector_type(4)));

void* kernel_workspace(size_t bytes);   // shim.hip

enum { SKN_EPI_NONE = 0, SKN_EPI_RESIDUAL = 1, SKN_EPI_SWIGLU = 2 };

__device__ __forceinline__ float skn_silu(float g) { return g * (1.0f / (1.0f + expf(-g))); }

// ---------------------------------------------------------------------------------------------- activations
// Inverse of skn_elem: 8-element piece j (0..31) of a super-block -> byte offset of its 16 bytes (row r of the tile) in the 8 KB of
// (row tile, super-block).
template <bool Q6>
__device__ __forceinline__ int skn_piece(int j, int r) {
    const int q = Q6 ? 2 * (j >> 4) + ((j >> 1) & 1) : j >> 3, u = Q6 ? 2 * ((j >> 2) & 3) + (j & 1) : j & 7;
    return u * 1024 + (r + 16 * q) * 16;
}
// One workgroup per (super-block, row tile of 16): 512 pieces, two per thread. PAIRS: rows of interleaved (gate, up)
// pairs, the activation is their SwiGLU.
template <bool Q6, bool PAIRS>
__global__ __launch_bounds__(256) void skinny_prepass_kernel(const float* __restrict__ x, uint8_t* __restrict__ out, int m, int k) {
    const int sb = blockIdx.x, mt = blockIdx.y, nsb = k >> 8;
    uint8_t* dst = out + ((int64_t)mt * nsb + sb) * 8192;
#pragma unroll
    for (int p = 0; p < 2; ++p) {
        const int r = (threadIdx.x >> 5) + 8 * p, j = threadIdx.x & 31, row = 16 * mt + r;
        uint4 v = make_uint4(0, 0, 0, 0);
        if (row < m) {
            const int64_t at = (int64_t)row * k + 256 * sb + 8 * j;
            if constexpr (PAIRS) {
                const float4* s = reinterpret_cast<const float4*>(x + 2 * at);
                const float4 a = s[0], b = s[1], c = s[2], d = s[3];
                v = make_uint4(skn_pack(skn_silu(a.x) * a.y, skn_silu(a.z) * a.w), skn_pack(skn_silu(b.x) * b.y, skn_silu(b.z) * b.w),
                               skn_pack(skn_silu(c.x) * c.y, skn_silu(c.z) * c.w), skn_pack(skn_silu(d.x) * d.y, skn_silu(d.z) * d.w));
            } else {
                const float4* s = reinterpret_cast<const float4*>(x + at);
                const float4 a = s[0], b = s[1];
                v = make_uint4(skn_pack(a.x, a.y), skn_pack(a.z, a.w), skn_pack(b.x, b.y), skn_pack(b.z, b.w));
            }
        }
        *reinterpret_cast<uint4*>(dst + skn_piece<Q6>(j, r)) = v;
    }
}
// The same with an RMSNorm folded in: one workgroup per row (rows past m: zeros), V pieces per thread held in registers.
template <bool Q6, int V>
__global__ __launch_bounds__(256) void skinny_prepass_rmsnorm_kernel(const float* __restrict__ x, const float* __restrict__ gain,
                                                                     uint8_t* __restrict__ out, int m, int k, float eps) {
    __shared__ float red[4];
    const int row = blockIdx.x, mt = row >> 4, r = row & 15, pieces = k >> 3;
    float4 a[V], b[V];
    float s = 0.f;
#pragma unroll
    for (int i = 0; i < V; ++i) {
        const int p = threadIdx.x + 256 * i;
        const bool in = p < pieces && row < m;
        const float4* src = reinterpret_cast<const float4*>(x + (int64_t)row * k) + 2 * p;
        a[i] = in ? src[0] : make_float4(0.f, 0.f, 0.f, 0.f);
        b[i] = in ? src[1] : make_float4(0.f, 0.f, 0.f, 0.f);
        s = fmaf(a[i].x, a[i].x, s); s = fmaf(a[i].y, a[i].y, s); s = fmaf(a[i].z, a[i].z, s); s = fmaf(a[i].w, a[i].w, s);
        s = fmaf(b[i].x, b[i].x, s); s = fmaf(b[i].y, b[i].y, s); s = fmaf(b[i].z, b[i].z, s); s = fmaf(b[i].w, b[i].w, s);
    }
    s = wave_sum(s);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
    __syncthreads();
    const float scale = 1.0f / sqrtf((red[0] + red[1] + red[2] + red[3]) * (1.0f / (float)k) + eps);
#pragma unroll
    for (int i = 0; i < V; ++i) {
        const int p = threadIdx.x + 256 * i;
        if (p >= pieces) continue;
        const float4* g4 = reinterpret_cast<const float4*>(gain) + 2 * p;
        const float4 g = g4[0], h = g4[1];
        const uint4 v = make_uint4(skn_pack(a[i].x * scale * g.x, a[i].y * scale * g.y), skn_pack(a[i].z * scale * g.z, a[i].w * scale * g.w),
                                   skn_pack(b[i].x * scale * h.x, b[i].y * scale * h.y), skn_pack(b[i].z * scale * h.z, b[i].w * scale * h.w));
        *reinterpret_cast<uint4*>(out + ((int64_t)mt * (k >> 8) + (p >> 5)) * 8192 + skn_piece<Q6>(p & 31, r)) = v;
    }
}

// ---------------------------------------------------------------------------------------------- the product
constexpr int SKN_WAVES = 8;      // one wave of a workgroup per super-block in turn (four waves measured the same or up to 10 % slower)
// The waves' partial tiles meet in LDS and are summed in wave order; residual or SwiGLU are applied where the sums are stored.
template <int MT, int NT>
__device__ __forceinline__ void skinny_finish(float* skn_part, const skn_f32x4 (&acc)[MT][NT], int lane, int wave, int m0, int n0, float* c,
                                              const float* residual, int m, int n, int epilogue) {
    constexpr int NW = SKN_WAVES;
    const int col = lane & 15, q = lane >> 4;
    // accumulator element e of lane (col, q): row 4 q + e, column col of its 16 x 16 tile
    float* mine = skn_part + (size_t)wave * (MT * NT * 256);
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
            for (int e = 0; e < 4; ++e) mine[(i * NT + t) * 256 + (4 * q + e) * 16 + col] = acc[i][t][e];
    __syncthreads();
    for (int p = threadIdx.x; p < MT * NT * 128; p += 64 * NW) {          // two adjacent columns each
        float2 s = make_float2(0.f, 0.f);
#pragma unroll
        for (int v = 0; v < NW; ++v) {
            const float2 t = *reinterpret_cast<const float2*>(skn_part + (size_t)v * (MT * NT * 256) + 2 * p);
            s.x += t.x; s.y += t.y;
        }
        const int tile = p >> 7, gr = m0 + 16 * (tile / NT) + ((p >> 3) & 15), gc = n0 + 16 * (tile % NT) + 2 * (p & 7);
        if (gr >= m || gc >= n) continue;
        if (epilogue == SKN_EPI_SWIGLU) {                                 // n is even: (gate, up) pairs
            c[(int64_t)gr * (n >> 1) + (gc >> 1)] = skn_silu(s.x) * s.y;
            continue;
        }
        const int64_t o = (int64_t)gr * n + gc;
        if (epilogue == SKN_EPI_RESIDUAL) { s.x += residual[o]; if (gc + 1 < n) s.y += residual[o + 1]; }
        c[o] = s.x;
        if (gc + 1 < n) c[o + 1] = s.y;
    }
}

template <class F, int MT, int NT>
__global__ __launch_bounds__(64 * SKN_WAVES) void packed_gemm_skinny_kernel(const uint8_t* __restrict__ a, const uint8_t* __restrict__ w, float* c,
                                                                     const float* residual, int m, int n, int k, int epilogue) {
    constexpr int NW = SKN_WAVES;
    extern __shared__ __attribute__((aligned(16))) float skn_part[];       // [NW][MT * NT][256]
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int col = lane & 15, q = lane >> 4;
    const int n0 = blockIdx.x * (16 * NT), mt0 = blockIdx.y * MT;
    const int nsb = k >> 8;
    const int mtiles = (m + 15) >> 4;
    const uint32_t row_bytes = (uint32_t)nsb * F::BYTES;
    uint32_t row[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) row[t] = (uint32_t)min(n0 + 16 * t + col, n - 1) * row_bytes;    // rows past N: a valid copy, never stored
    // A operands of (row tile, super-block): 8 KB; row tiles past the last are copies of it, never stored
    const uint8_t* at[MT];
#pragma unroll
    for (int i = 0; i < MT; ++i) at[i] = a + (int64_t)min(mt0 + i, mtiles - 1) * nsb * 8192 + 16 * lane;
    skn_f32x4 acc[MT][NT];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int t = 0; t < NT; ++t) acc[i][t] = skn_f32x4{0.f, 0.f, 0.f, 0.f};

    constexpr int AR = MT >= 4 ? 2 : 4;                                   // steps of A operands in flight or in use
    if (wave < nsb) {
        typename F::Raw raw[2][NT];
        auto load_w = [&](int set, int sb) __attribute__((always_inline)) {
            const uint8_t* base = w + (int64_t)sb * F::BYTES;
#pragma unroll
            for (int t = 0; t < NT; ++t) F::load(raw[set][t], base + row[t], q);
        };
        skn_bf16x8 af[AR][MT];
        auto load_a = [&](int slot, int sb, int u) __attribute__((always_inline)) {
#pragma unroll
            for (int i = 0; i < MT; ++i) af[slot][i] = *reinterpret_cast<const skn_bf16x8*>(at[i] + (int64_t)sb * 8192 + 1024 * u);
        };
        // one super-block: `set` holds its bytes, `next` (clamped to this wave's last) is requested meanwhile
        auto body = [&](auto set_c, int sb, int next) __attribute__((always_inline)) {
            constexpr int SET = decltype(set_c)::value;
            load_w(SET ^ 1, next);
            typename F::Scales sc[NT];
#pragma unroll
            for (int t = 0; t < NT; ++t) sc[t] = F::scales(raw[SET][t], q);
            auto step = [&](auto uc) __attribute__((always_inline)) {
                constexpr int U = decltype(uc)::value;
                constexpr int AHEAD = U + AR - 1;
                if constexpr (AHEAD < 8) load_a(AHEAD % AR, sb, AHEAD);
                else load_a(AHEAD % AR, next, AHEAD - 8);
#pragma unroll
                for (int t = 0; t < NT; ++t) {
                    SknBf16 o;
                    F::template decode<U>(raw[SET][t], sc[t], o);
                    const skn_bf16x8 b = __builtin_bit_cast(skn_bf16x8, uint4{o.o[0], o.o[1], o.o[2], o.o[3]});
#pragma unroll
                    for (int i = 0; i < MT; ++i) acc[i][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af[U % AR][i], b, acc[i][t], 0, 0, 0);
                }
            };
            step(std::integral_constant<int, 0>{}); step(std::integral_constant<int, 1>{});
            step(std::integral_constant<int, 2>{}); step(std::integral_constant<int, 3>{});
            step(std::integral_constant<int, 4>{}); step(std::integral_constant<int, 5>{});
            step(std::integral_constant<int, 6>{}); step(std::integral_constant<int, 7>{});
        };
        load_w(0, wave);
#pragma unroll
        for (int u = 0; u < AR - 1; ++u) load_a(u, wave, u);
        for (int sb = wave; sb < nsb; sb += 2 * NW) {
            const int second = sb + NW, third = sb + 2 * NW;
            body(std::integral_constant<int, 0>{}, sb, second < nsb ? second : sb);
            if (second >= nsb) break;
            body(std::integral_constant<int, 1>{}, second, third < nsb ? third : second);
        }
    }
    skinny_finish<MT, NT>(skn_part, acc, lane, wave, 16 * mt0, n0, c, residual, m, n, epilogue);
}

// ---------------------------------------------------------------------------------------------- the product, in one launch
// Small products spend more on the pass in front than it saves: a launch (2.3 us of the host, 1.3 behind another one on the device) and the trip of
// its result through memory. Here the activations come straight from their fp32 rows, twice the bytes per workgroup, which is what ends it:
// from about 10 us on the pass pays (gemm.hip has the rule). Back to back from the host (device alone in brackets): Q4_0 18 x 924 x 1024 6.7 ->
// 4.3 us (4.4 -> 3.0), Q5_K 43 x 515 x 768 6.6 -> 4.3, Q6_K 15 x 589 x 3072 7.1 -> 5.9, Q4_0 46 x 11272 x 1280 10.2 as before.
//
// Two forms. `direct`: the tiles, waves and sums of the kernel above; a wave's super-block of 16 MT rows comes in four stages of two
// steps, loaded in runs of 64 bytes, rounded to bf16 and put into LDS of the wave's own in fragment order, from where a step's A operand
// is one 16-byte read per lane. Nothing is shared between waves, so nothing waits before the partial tiles meet.
//   * LDS of a (row tile, stage): piece (r, q) of step u at UB u + QB q + 16 r bytes. A wave writes 4 rows x 4 q x 2 u x 2 halves of eight
//     bytes at once: QB of 320 bytes spreads them evenly over the banks. (Stages of four steps: 5 to 10 % slower, for their registers.)
constexpr int SKN_STAGE_STEPS = 2;
template <bool Q6, int MT>
struct SknStage {
    static constexpr int S = SKN_STAGE_STEPS, LOADS = 2 * S * MT, RPL = 8 / S;      // 16-byte loads per lane, rows of one load
    static constexpr int QB = 320, UB = 4 * QB, BYTES = MT * S * UB;
    static constexpr int STRIDE = Q6 ? 16 * S : 8 * S;                      // elements from one stage to the next
    // lane -> row of a load, first element of stage 0 inside the super-block, LDS offset of its eight bytes (the inverse of skn_elem)
    static __device__ __forceinline__ int row(int lane) { return lane / (8 * S); }
    static __device__ __forceinline__ int elem(int lane) {
        const int f = lane & (8 * S - 1);
        return Q6 ? 128 * (f / (4 * S)) + 4 * (f & (4 * S - 1)) : 64 * (f / (2 * S)) + 4 * (f & (2 * S - 1));
    }
    static __device__ __forceinline__ int lds(int lane) {
        const int f = lane & (8 * S - 1);
        const int q = Q6 ? 2 * (f / (4 * S)) + ((f >> 2) & 1) : f / (2 * S);
        const int u = Q6 ? 2 * ((f & (4 * S - 1)) >> 3) + ((f >> 1) & 1) : (f & (2 * S - 1)) >> 1;
        return u * UB + q * QB + 16 * row(lane) + 8 * (f & 1);
    }
};
template <class F, int MT, int NT>
__global__ __launch_bounds__(64 * SKN_WAVES) void packed_gemm_skinny_direct_kernel(const float* __restrict__ x, const uint8_t* __restrict__ w, float* c,
                                                                            const float* residual, int m, int n, int k, int epilogue) {
    constexpr int NW = SKN_WAVES, S = SKN_STAGE_STEPS, STAGES = 8 / S;
    using St = SknStage<F::Q6, MT>;
    extern __shared__ __attribute__((aligned(16))) float skn_part[];       // [NW][stage of activations], then [NW][MT * NT][256]
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int col = lane & 15, q = lane >> 4;
    const int n0 = blockIdx.x * (16 * NT), m0 = blockIdx.y * (16 * MT);
    const int nsb = k >> 8;
    const uint32_t row_bytes = (uint32_t)nsb * F::BYTES;
    uint32_t row[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) row[t] = (uint32_t)min(n0 + 16 * t + col, n - 1) * row_bytes;    // rows past N: a valid copy, never stored
    skn_f32x4 acc[MT][NT];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int t = 0; t < NT; ++t) acc[i][t] = skn_f32x4{0.f, 0.f, 0.f, 0.f};

    if (wave < nsb) {
        uint8_t* const mine = reinterpret_cast<uint8_t*>(skn_part) + (size_t)wave * St::BYTES;
        uint8_t* const put = mine + St::lds(lane);
        const uint8_t* const get = mine + q * St::QB + 16 * col;
        const int srow = m0 + St::row(lane), selem = St::elem(lane);
        float4 xs[St::LOADS];
        auto load_x = [&](int sb, int stage) __attribute__((always_inline)) {     // rows past m: copies of the last, never stored
#pragma unroll
            for (int i = 0; i < St::LOADS; ++i)
                xs[i] = *reinterpret_cast<const float4*>(x + (int64_t)min(srow + St::RPL * i, m - 1) * k + (256 * sb + St::STRIDE * stage + selem));
        };
        auto store_x = [&]() __attribute__((always_inline)) {
            __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");        // wave-private: LDS serves a wave's accesses in order
            __builtin_amdgcn_wave_barrier();
#pragma unroll
            for (int i = 0; i < St::LOADS; ++i) {                         // load i: rows RPL i .. of tile i / (2 S)
                uint2* dst = reinterpret_cast<uint2*>(put + (i / (2 * S)) * (S * St::UB) + 16 * St::RPL * (i % (2 * S)));
                *dst = make_uint2(skn_pack(xs[i].x, xs[i].y), skn_pack(xs[i].z, xs[i].w));
            }
            __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
            __builtin_amdgcn_wave_barrier();
        };
        typename F::Raw raw[2][NT];
        auto load_w = [&](int set, int sb) __attribute__((always_inline)) {
            const uint8_t* base = w + (int64_t)sb * F::BYTES;
#pragma unroll
            for (int t = 0; t < NT; ++t) F::load(raw[set][t], base + row[t], q);
        };
        // one super-block: `set` holds its bytes, LDS its first stage; `next` and `after` are this wave's super-blocks behind it (its last, where
        // there is none)
        auto body = [&](auto set_c, int sb, int next, int after) __attribute__((always_inline)) {
            constexpr int SET = decltype(set_c)::value;
            typename F::Scales sc[NT];
#pragma unroll
            for (int t = 0; t < NT; ++t) sc[t] = F::scales(raw[SET][t], q);
            auto step = [&](auto uc) __attribute__((always_inline)) {
                constexpr int U = decltype(uc)::value;
                if constexpr (U % S == 0) {
                    if constexpr (U / S + 1 < STAGES) load_x(sb, U / S + 1);
                    else load_x(next, 0);
                    __builtin_amdgcn_sched_barrier(0);
                }
                skn_bf16x8 af[MT];
#pragma unroll
                for (int i = 0; i < MT; ++i) af[i] = *reinterpret_cast<const skn_bf16x8*>(get + i * (S * St::UB) + (U % S) * St::UB);
#pragma unroll
                for (int t = 0; t < NT; ++t) {
                    SknBf16 o;
                    F::template decode<U>(raw[SET][t], sc[t], o);
                    const skn_bf16x8 b = __builtin_bit_cast(skn_bf16x8, uint4{o.o[0], o.o[1], o.o[2], o.o[3]});
#pragma unroll
                    for (int i = 0; i < MT; ++i) acc[i][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af[i], b, acc[i][t], 0, 0, 0);
                }
                if constexpr (U == 7) {
                    __builtin_amdgcn_sched_barrier(0);
                    load_w(SET, after);
                    __builtin_amdgcn_sched_barrier(0);
                }
                if constexpr (U % S == S - 1) store_x();
            };
            step(std::integral_constant<int, 0>{}); step(std::integral_constant<int, 1>{});
            step(std::integral_constant<int, 2>{}); step(std::integral_constant<int, 3>{});
            step(std::integral_constant<int, 4>{}); step(std::integral_constant<int, 5>{});
            step(std::integral_constant<int, 6>{}); step(std::integral_constant<int, 7>{});
        };
        const int last = wave + (nsb - 1 - wave) / NW * NW;               // this wave's last super-block
        load_x(wave, 0);
        __builtin_amdgcn_sched_barrier(0);
        load_w(0, wave);
        load_w(1, min(wave + NW, last));
        __builtin_amdgcn_sched_barrier(0);
        store_x();
        for (int sb = wave; sb < nsb; sb += 2 * NW) {
            const int second = min(sb + NW, last), third = min(sb + 2 * NW, last), fourth = min(sb + 3 * NW, last);
            body(std::integral_constant<int, 0>{}, sb, second, third);
            if (sb + NW >= nsb) break;
            body(std::integral_constant<int, 1>{}, second, third, fourth);
        }
    }
    __syncthreads();                                                      // the partial tiles go where the activations were
    skinny_finish<MT, NT>(skn_part, acc, lane, wave, m0, n0, c, residual, m, n, epilogue);
}

// `shared`: four waves on neighbouring columns take a share of K together, the two shares a super-block each in turn: the workgroup reads its
// fp32 rows once for 64 NT columns (16 NT above), rounds them and leaves them in LDS in fragment order, two rounds deep. For many columns
// of short rows: Q4_0 46 x 3830 x 1024 6.4 -> 5.2 us on the device, Q5_K 91 x 8978 x 512 10.7 -> 7.8.
// LDS of a (share, row tile, round): piece (r, q) of step u at 1088 u + 272 q + 16 r bytes, which spreads the 64 halves of a row that a wave
// writes at once evenly over the banks.
constexpr int SKN_QB = 272, SKN_UB = 4 * SKN_QB, SKN_TILE_BYTES = 8 * SKN_UB, SKN_WN = 4;
template <class F, int MT, int NT>
__global__ __launch_bounds__(64 * SKN_WAVES) void packed_gemm_skinny_shared_kernel(const float* __restrict__ x, const uint8_t* __restrict__ w, float* c,
                                                                            const float* residual, int m, int n, int k, int epilogue) {
    constexpr int NW = SKN_WAVES, WN = SKN_WN, WK = NW / WN, LOADS = 16 * MT * WK / NW;
    extern __shared__ __attribute__((aligned(16))) float skn_part[];       // [2][WK][MT] tiles of activations, then [WK][WN][MT * NT][256]
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int kg = wave / WN, wn = wave % WN;
    const int col = lane & 15, q = lane >> 4;
    const int n0 = (blockIdx.x * WN + wn) * (16 * NT), m0 = blockIdx.y * (16 * MT);
    const int nsb = k >> 8;
    const uint32_t row_bytes = (uint32_t)nsb * F::BYTES;
    uint32_t row[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) row[t] = (uint32_t)min(n0 + 16 * t + col, n - 1) * row_bytes;    // rows past N: a valid copy, never stored
    skn_f32x4 acc[MT][NT];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int t = 0; t < NT; ++t) acc[i][t] = skn_f32x4{0.f, 0.f, 0.f, 0.f};

    uint8_t* const smem = reinterpret_cast<uint8_t*>(skn_part);
    // wave w stages rows w LOADS .. of the [WK][16 MT] rows of a round: all of one share and row tile
    static_assert(16 % LOADS == 0 || LOADS % 16 == 0, "a wave's rows");
    const int srow = wave * LOADS, skg = srow / (16 * MT), sr = srow % (16 * MT);
    const int f = lane;
    const int fq = F::Q6 ? 2 * (f >> 5) + ((f >> 2) & 1) : f >> 4, fu = F::Q6 ? 2 * ((f >> 3) & 3) + ((f >> 1) & 1) : (f & 15) >> 1;
    uint8_t* const put = smem + (skg * MT + (sr >> 4)) * SKN_TILE_BYTES + (sr & 15) * 16 + fu * SKN_UB + fq * SKN_QB + 8 * (f & 1);
    const uint8_t* const get = smem + kg * MT * SKN_TILE_BYTES + q * SKN_QB + 16 * col;
    constexpr int ROUND_BYTES = WK * MT * SKN_TILE_BYTES;
    float4 xs[LOADS];
    auto load_x = [&](int round) __attribute__((always_inline)) {         // rows past m and super-blocks past the last: copies, not used
        const int sb = min(round * WK + skg, nsb - 1);
#pragma unroll
        for (int i = 0; i < LOADS; ++i) xs[i] = *reinterpret_cast<const float4*>(x + (int64_t)min(m0 + sr + i, m - 1) * k + (256 * sb + 4 * lane));
    };
    auto store_x = [&](int buf) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < LOADS; ++i)
            *reinterpret_cast<uint2*>(put + buf * ROUND_BYTES + (i >> 4) * SKN_TILE_BYTES + 16 * (i & 15)) = make_uint2(skn_pack(xs[i].x, xs[i].y), skn_pack(xs[i].z, xs[i].w));
    };
    typename F::Raw raw[2][NT];
    auto load_w = [&](int set, int round) __attribute__((always_inline)) {
        const uint8_t* base = w + (int64_t)min(round * WK + kg, nsb - 1) * F::BYTES;
#pragma unroll
        for (int t = 0; t < NT; ++t) F::load(raw[set][t], base + row[t], q);
    };
    const int rounds = (nsb + WK - 1) / WK;
    auto body = [&](auto set_c, int round) __attribute__((always_inline)) {
        constexpr int SET = decltype(set_c)::value;
        if (round * WK + kg < nsb) {
            typename F::Scales sc[NT];
#pragma unroll
            for (int t = 0; t < NT; ++t) sc[t] = F::scales(raw[SET][t], q);
            auto step = [&](auto uc) __attribute__((always_inline)) {
                constexpr int U = decltype(uc)::value;
                skn_bf16x8 af[MT];
#pragma unroll
                for (int i = 0; i < MT; ++i) af[i] = *reinterpret_cast<const skn_bf16x8*>(get + SET * ROUND_BYTES + i * SKN_TILE_BYTES + U * SKN_UB);
#pragma unroll
                for (int t = 0; t < NT; ++t) {
                    SknBf16 o;
                    F::template decode<U>(raw[SET][t], sc[t], o);
                    const skn_bf16x8 b = __builtin_bit_cast(skn_bf16x8, uint4{o.o[0], o.o[1], o.o[2], o.o[3]});
#pragma unroll
                    for (int i = 0; i < MT; ++i) acc[i][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af[i], b, acc[i][t], 0, 0, 0);
                }
            };
            step(std::integral_constant<int, 0>{}); step(std::integral_constant<int, 1>{});
            step(std::integral_constant<int, 2>{}); step(std::integral_constant<int, 3>{});
            step(std::integral_constant<int, 4>{}); step(std::integral_constant<int, 5>{});
            step(std::integral_constant<int, 6>{}); step(std::integral_constant<int, 7>{});
        }
        __builtin_amdgcn_sched_barrier(0);
        load_w(SET, round + 2);
        __builtin_amdgcn_sched_barrier(0);
        store_x(SET ^ 1);
        load_x(round + 2);
        __syncthreads();
    };
    load_x(0);
    __builtin_amdgcn_sched_barrier(0);
    load_w(0, 0);
    load_w(1, 1);
    __builtin_amdgcn_sched_barrier(0);
    store_x(0);
    load_x(1);
    __syncthreads();
    for (int round = 0; round < rounds; round += 2) {
        body(std::integral_constant<int, 0>{}, round);
        if (round + 1 >= rounds) break;
        body(std::integral_constant<int, 1>{}, round + 1);
    }
    // the shares' partial tiles meet where the activations were
    float* mine = skn_part + (size_t)wave * (MT * NT * 256);
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
            for (int e = 0; e < 4; ++e) mine[(i * NT + t) * 256 + (4 * q + e) * 16 + col] = acc[i][t][e];
    __syncthreads();
    for (int p = threadIdx.x; p < WN * MT * NT * 128; p += 64 * NW) {
        const int g = p / (MT * NT * 128), pt = p % (MT * NT * 128);
        float2 s = make_float2(0.f, 0.f);
#pragma unroll
        for (int v = 0; v < WK; ++v) {
            const float2 t = *reinterpret_cast<const float2*>(skn_part + (size_t)(v * WN + g) * (MT * NT * 256) + 2 * pt);
            s.x += t.x; s.y += t.y;
        }
        const int tile = pt >> 7, gr = m0 + 16 * (tile / NT) + ((pt >> 3) & 15);
        const int gc = (blockIdx.x * WN + g) * (16 * NT) + 16 * (tile % NT) + 2 * (pt & 7);
        if (gr >= m || gc >= n) continue;
        if (epilogue == SKN_EPI_SWIGLU) {                                 // n is even: (gate, up) pairs
            c[(int64_t)gr * (n >> 1) + (gc >> 1)] = skn_silu(s.x) * s.y;
            continue;
        }
        const int64_t o = (int64_t)gr * n + gc;
        if (epilogue == SKN_EPI_RESIDUAL) { s.x += residual[o]; if (gc + 1 < n) s.y += residual[o + 1]; }
        c[o] = s.x;
        if (gc + 1 < n) c[o + 1] = s.y;
    }
}

size_t gemm_skinny_activation_bytes(int m, int k) { return (size_t)((m + 15) / 16) * 16 * (size_t)k * 2; }
// k in whole super-blocks, byte offsets of a weight row in 32 bits
bool gemm_skinny_fits(int enc, int m, int n, int k) {
    return k % 256 == 0 && (uint64_t)n * (uint64_t)(k / block_elems(enc)) * block_bytes(enc) < ((uint64_t)1 << 32) && (m + 15) / 16 <= 65535;
}

template <class F, int MT, int NT, bool SHARED>
static int launch_skinny_direct_tile(const float* x, const uint8_t* w, float* c, const float* residual, int m, int n, int k, int epilogue, hipStream_t s) {
    constexpr size_t stage = SHARED ? 2 * (SKN_WAVES / SKN_WN) * MT * SKN_TILE_BYTES : SKN_WAVES * SknStage<F::Q6, MT>::BYTES;
    constexpr size_t tile = SKN_WAVES * MT * NT * 256 * sizeof(float), smem = stage > tile ? stage : tile;
    constexpr int columns = 16 * NT * (SHARED ? SKN_WN : 1);
    constexpr auto kernel = SHARED ? &packed_gemm_skinny_shared_kernel<F, MT, NT> : &packed_gemm_skinny_direct_kernel<F, MT, NT>;
    SKH_SET_MAX_DYNAMIC_LDS_ONCE(kernel, smem);
    note_kernel(SHARED ? "packed_gemm_skinny_shared_kernel" : "packed_gemm_skinny_direct_kernel");
    kernel<<<dim3((n + columns - 1) / columns, (m + 16 * MT - 1) / (16 * MT)), dim3(64 * SKN_WAVES), smem, s>>>(x, w, c, residual, m, n, k, epilogue);
    SKH_CHECK(hipGetLastError());
    return 0;
}
template <bool Q6>
static int skinny_prepass(const float* x, const float* gain, float eps, uint8_t* a, int m, int k, bool pairs, hipStream_t s) {
    const int mtiles = (m + 15) / 16;
    if (pairs) skinny_prepass_kernel<Q6, true><<<dim3(k / 256, mtiles), dim3(256), 0, s>>>(x, a, m, k);
    else if (!gain) skinny_prepass_kernel<Q6, false><<<dim3(k / 256, mtiles), dim3(256), 0, s>>>(x, a, m, k);
    else if (k <= 256 * 8 * 2) skinny_prepass_rmsnorm_kernel<Q6, 2><<<dim3(16 * mtiles), dim3(256), 0, s>>>(x, gain, a, m, k, eps);
    else skinny_prepass_rmsnorm_kernel<Q6, 8><<<dim3(16 * mtiles), dim3(256), 0, s>>>(x, gain, a, m, k, eps);
    SKH_CHECK(hipGetLastError());
    return 0;
}

template <class F, int MT, int NT>
static int launch_skinny_tile(const uint8_t* a, const uint8_t* w, float* c, const float* residual, int m, int n, int k, int epilogue, hipStream_t s) {
    constexpr size_t smem = (size_t)SKN_WAVES * MT * NT * 256 * sizeof(float);
    SKH_SET_MAX_DYNAMIC_LDS_ONCE((&packed_gemm_skinny_kernel<F, MT, NT>), smem);
    packed_gemm_skinny_kernel<F, MT, NT><<<dim3((n + 16 * NT - 1) / (16 * NT), ((m + 15) / 16 + MT - 1) / MT), dim3(64 * SKN_WAVES), smem, s>>>(
        a, w, c, residual, m, n, k, epilogue);
    SKH_CHECK(hipGetLastError());
    return 0;
}

// The tile of a shape and what it is estimated to take, in us: the two launches, what both move, and what the workgroups of a CU
// take: the first one and each further one for a share of K of one super-block per wave (2048 elements). Fitted to 142 000
// timings of random products (9 to 1024 rows, n 512 to 32000, K 512 to 14336, every format and tile), which it meets within 5
// to 6 % (rms). The last, partial round of a CU costs a share `whole` of a full one whatever there is in it, the last, partial
// share of K of the taller tiles a third.
struct SknTile { int mt, nt, wn; double us; };      // wn: waves that share activations in the one-launch forms (1: none)
SknTile gemm_skinny_tile(int enc, int m, int n, int k) {
    static const int shapes[6][2] = {{1, 1}, {2, 1}, {4, 1}, {1, 2}, {2, 2}, {4, 2}};     // tiles of 16 mt rows x 16 nt columns
    static const double q4k[6][2] = {{1.15, 1.24}, {2.37, 1.83}, {3.80, 3.86}, {2.17, 1.94}, {2.80, 2.37}, {3.58, 3.81}};
    static const double q5k[6][2] = {{1.63, 1.40}, {2.18, 1.98}, {3.97, 3.80}, {3.17, 2.71}, {3.68, 2.97}, {4.96, 5.02}};
    static const double q6k[6][2] = {{2.16, 2.08}, {2.76, 2.55}, {3.89, 4.14}, {4.31, 4.90}, {4.63, 5.67}, {6.04, 6.26}};
    static const double q80[6][2] = {{1.67, 2.01}, {2.63, 2.33}, {5.23, 3.44}, {3.07, 3.85}, {4.08, 4.03}, {4.98, 5.31}};
    static const double q40[6][2] = {{1.18, 1.29}, {2.02, 1.82}, {3.42, 2.46}, {2.03, 2.11}, {2.87, 2.44}, {3.81, 3.94}};
    static const double q50[6][2] = {{1.32, 1.36}, {2.06, 1.81}, {3.82, 2.60}, {2.65, 2.53}, {3.26, 2.81}, {4.07, 4.44}};
    static const double q51[6][2] = {{1.48, 1.37}, {2.01, 1.97}, {3.95, 2.57}, {2.76, 2.53}, {3.63, 2.94}, {4.69, 4.92}};
    static const double whole[6] = {0.86, 0.75, 0.78, 0.81, 0.82, 0.96}, whole_k[6] = {0.0, 0.06, 0.32, 0.04, 0.08, 0.32};
    const double (*cost)[2] = enc == ENC_Q4_K ? q4k : enc == ENC_Q5_K ? q5k : enc == ENC_Q6_K ? q6k : enc == ENC_Q4_0 ? q40 : enc == ENC_Q5_0 ? q50
                            : enc == ENC_Q5_1 ? q51 : q80;
    const int mtiles = (m + 15) / 16;
    const double shares = k / (256.0 * SKN_WAVES);
    SknTile best{1, 1, 0, 0.0};
    for (int i = 0; i < 6; ++i) {
        const int mt = shapes[i][0], nt = shapes[i][1];
        if (mt > 1 && mt >= 2 * mtiles) continue;                         // more rows than there are
        const double groups = (double)((mtiles + mt - 1) / mt) * ((n + 16 * nt - 1) / (16 * nt)) / num_cus();
        const double further = groups <= 1.0 ? 0.0 : whole[i] * ceil(groups) + (1 - whole[i]) * groups - 1;
        const double us = 3.9 + 2.06e-6 * m * k + 3.55e-6 * m * n +
                          (cost[i][0] + cost[i][1] * further) * ((1 - whole_k[i]) * shares + whole_k[i] * ceil(shares));
        if (best.us == 0.0 || us < best.us) best = SknTile{mt, nt, 0, us};
    }
    return best;
}
double gemm_skinny_estimate(int enc, int m, int n, int k) { return gemm_skinny_tile(enc, m, n, k).us; }

// The one-launch form of a shape and what it is estimated to take, in us, or mt = 0: outside its range. Terms as above: the launch, the result, the
// workgroups of a CU for their shares of K. Fitted to 2 560 random products (9 to 200 rows, m n k up to 1.2e9, every format), which it meets
// within 4 to 7 % (rms). Rows of more than 4864 are left out: the estimate is low there (from 6144 on by 20 to 30 %), and those that took a form gained
// nothing on the device (Q4_K 95 x 668 x 5888 8.5 us in two launches, 9.5 in one).
SknTile gemm_skinny_direct_tile(int enc, int m, int n, int k) {
    struct Form { int mt, nt, wn; double launch, result, whole, whole_k, cost[7][2]; };          // formats: Q4_K, Q5_K, Q6_K, Q8_0, Q4_0, Q5_0, Q5_1
    static const Form forms[4] = {
        {1, 1, 1, 2.16, 6.98e-06, 0.84, 0.00, {{1.69, 2.41}, {2.36, 2.64}, {3.47, 4.51}, {2.30, 3.08}, {1.85, 2.48}, {1.95, 2.52}, {2.08, 2.70}}},
        {1, 2, 1, 2.39, 4.43e-06, 0.86, 0.03, {{2.64, 4.09}, {3.92, 5.83}, {7.05, 9.79}, {4.02, 5.82}, {2.85, 2.90}, {3.21, 3.02}, {3.58, 3.52}}},
        {1, 1, 4, 2.46, 2.10e-06, 0.75, 0.47, {{1.10, 1.15}, {1.54, 1.59}, {2.65, 3.06}, {1.69, 1.71}, {1.12, 1.20}, {1.30, 1.24}, {1.35, 1.44}}},
        {2, 2, 4, 3.40, 1.21e-06, 0.75, 0.46, {{2.59, 4.99}, {3.41, 5.97}, {5.94, 8.48}, {3.63, 6.63}, {2.44, 4.65}, {2.79, 3.10}, {2.93, 3.57}}},
    };
    SknTile best{0, 0, 0, 0.0};
    if (k > 4864) return best;
    const int format = enc == ENC_Q4_K ? 0 : enc == ENC_Q5_K ? 1 : enc == ENC_Q6_K ? 2 : enc == ENC_Q8_0 ? 3 : enc == ENC_Q4_0 ? 4 : enc == ENC_Q5_0 ? 5 : 6;
    const int mtiles = (m + 15) / 16;
    for (const Form& f : forms) {
        if (f.mt > 1 && f.mt >= 2 * mtiles) continue;                     // more rows than there are
        const double shares = k / (256.0 * (SKN_WAVES / f.wn));
        const double groups = (double)((mtiles + f.mt - 1) / f.mt) * ((n + 16 * f.nt * f.wn - 1) / (16 * f.nt * f.wn)) / num_cus();
        const double further = groups <= 1.0 ? 0.0 : f.whole * ceil(groups) + (1 - f.whole) * groups - 1;
        const double us = f.launch + f.result * m * n + (f.cost[format][0] + f.cost[format][1] * further) * ((1 - f.whole_k) * shares + f.whole_k * ceil(shares));
        if (best.mt == 0 || us < best.us) best = SknTile{f.mt, f.nt, f.wn, us};
    }
    if (k % 2048 == 0) best.us *= 1.08;      // rows of 2^n KB meet in the same channels of the L2
    return best;
}
// From 8 us on the estimate is a tenth low for what single waves read for themselves, for Q6_K and for Q8_0: such products took 1.01 to 1.05 of what two launches
// take, on the device and from the host (Q6_K 55 x 9274 x 768 11.3 -> 12.0 us, Q8_0 46 x 8548 x 768 8.2 -> 9.9, 100 x 7267 x 1024 11.8 -> 13.2), the others 0.87.
double gemm_skinny_direct_estimate(int enc, int m, int n, int k) {
    const SknTile t = gemm_skinny_direct_tile(enc, m, n, k);
    return !t.mt || (t.us >= 8 && (t.wn == 1 || enc == ENC_Q6_K || enc == ENC_Q8_0)) ? 1e30 : t.us;
}

// 0 never, 1 where the estimates favour it, 2 (to 10) wherever it fits; 10 mt + nt: that tile, wherever it fits; 100 wn + 10 mt + nt: that one-launch
// form, wherever it fits. A value that names no built form changes nothing.
static std::atomic<int> g_gemm_skinny{1};
void set_gemm_skinny(int v) {
    static const int forms[] = {11, 12, 21, 22, 41, 42, 111, 112, 411, 422};
    bool known = v <= 10;
    for (int f : forms) known |= v == f;
    if (known) g_gemm_skinny = v < 0 ? 0 : v > 2 && v <= 10 ? 2 : v;
}
int gemm_skinny_mode() { return g_gemm_skinny.load(); }
static std::atomic<int> g_gemm_skinny_direct{1};   // the one-launch forms by rule: 0 never, 1 where the estimates favour them
void set_gemm_skinny_direct(int v) { g_gemm_skinny_direct = v != 0; }
bool gemm_skinny_direct_enabled() { return g_gemm_skinny_direct.load() != 0; }

template <class F>
static int launch_skinny_format(int enc, const float* x, const float* gain, float eps, bool pairs, uint8_t* a, const uint8_t* w, float* c,
                                const float* residual, int m, int n, int k, int epilogue, hipStream_t s) {
    if (skinny_prepass<F::Q6>(x, gain, eps, a, m, k, pairs, s) != 0) return -1;
    SknTile t = gemm_skinny_tile(enc, m, n, k);
    if (const int forced = g_gemm_skinny.load(); forced >= 11) { t.mt = forced / 10 % 10; t.nt = forced % 10; }
    note_kernel("packed_gemm_skinny_kernel");
    if (t.nt == 2) {
        if (t.mt == 4) return launch_skinny_tile<F, 4, 2>(a, w, c, residual, m, n, k, epilogue, s);
        if (t.mt == 2) return launch_skinny_tile<F, 2, 2>(a, w, c, residual, m, n, k, epilogue, s);
        return launch_skinny_tile<F, 1, 2>(a, w, c, residual, m, n, k, epilogue, s);
    }
    if (t.mt == 4) return launch_skinny_tile<F, 4, 1>(a, w, c, residual, m, n, k, epilogue, s);
    if (t.mt == 2) return launch_skinny_tile<F, 2, 1>(a, w, c, residual, m, n, k, epilogue, s);
    return launch_skinny_tile<F, 1, 1>(a, w, c, residual, m, n, k, epilogue, s);
}

template <class F>
static int launch_skinny_direct_format(SknTile t, const float* x, const uint8_t* w, float* c, const float* residual, int m, int n, int k, int epilogue, hipStream_t s) {
    if (t.wn > 1) {
        if (t.mt == 2) return launch_skinny_direct_tile<F, 2, 2, true>(x, w, c, residual, m, n, k, epilogue, s);
        return launch_skinny_direct_tile<F, 1, 1, true>(x, w, c, residual, m, n, k, epilogue, s);
    }
    if (t.nt == 2) return launch_skinny_direct_tile<F, 1, 2, false>(x, w, c, residual, m, n, k, epilogue, s);
    return launch_skinny_direct_tile<F, 1, 1, false>(x, w, c, residual, m, n, k, epilogue, s);
}
// c = epilogue(x . W^T) in one launch, inside gemm_skinny_fits. Workgroups read x while others store c: the two must not overlap.
int launch_gemm_skinny_direct(int enc, const uint8_t* w, const float* x, int m, int k, int n, float* c, const float* residual, int epilogue) {
    SknTile t = gemm_skinny_direct_tile(enc, m, n, k);
    if (const int forced = g_gemm_skinny.load(); forced >= 100) { t.wn = forced / 100; t.mt = forced / 10 % 10; t.nt = forced % 10; }
    hipStream_t s = current_stream();
    switch (enc) {
        case ENC_Q4_K: return launch_skinny_direct_format<SknQ4K>(t, x, w, c, residual, m, n, k, epilogue, s);
        case ENC_Q5_K: return launch_skinny_direct_format<SknQ5K>(t, x, w, c, residual, m, n, k, epilogue, s);
        case ENC_Q6_K: return launch_skinny_direct_format<SknQ6K>(t, x, w, c, residual, m, n, k, epilogue, s);
        case ENC_Q4_0: return launch_skinny_direct_format<SknQ45<0>>(t, x, w, c, residual, m, n, k, epilogue, s);
        case ENC_Q5_0: return launch_skinny_direct_format<SknQ45<1>>(t, x, w, c, residual, m, n, k, epilogue, s);
        case ENC_Q5_1: return launch_skinny_direct_format<SknQ45<2>>(t, x, w, c, residual, m, n, k, epilogue, s);
        default: return launch_skinny_direct_format<SknQ80>(t, x, w, c, residual, m, n, k, epilogue, s);
    }
}

// c = epilogue(prologue(x) . W^T), all of it: the pass in front and the product. `c` is [m, n] ([m, n / 2] with SwiGLU).
int launch_gemm_skinny(int enc, const uint8_t* w, const float* x, int m, int k, int n, float* c, const float* gain, float eps,
                       const float* residual, int epilogue, bool x_pairs) {
    uint8_t* a = static_cast<uint8_t*>(kernel_workspace(gemm_skinny_activation_bytes(m, k)));
    if (!a) return -1;
    hipStream_t s = current_stream();
    switch (enc) {
        case ENC_Q4_K: return launch_skinny_format<SknQ4K>(enc, x, gain, eps, x_pairs, a, w, c, residual, m, n, k, epilogue, s);
        case ENC_Q5_K: return launch_skinny_format<SknQ5K>(enc, x, gain, eps, x_pairs, a, w, c, residual, m, n, k, epilogue, s);
        case ENC_Q6_K: return launch_skinny_format<SknQ6K>(enc, x, gain, eps, x_pairs, a, w, c, residual, m, n, k, epilogue, s);
        case ENC_Q4_0: return launch_skinny_format<SknQ45<0>>(enc, x, gain, eps, x_pairs, a, w, c, residual, m, n, k, epilogue, s);
        case ENC_Q5_0: return launch_skinny_format<SknQ45<1>>(enc, x, gain, eps, x_pairs, a, w, c, residual, m, n, k, epilogue, s);
        case ENC_Q5_1: return launch_skinny_format<SknQ45<2>>(enc, x, gain, eps, x_pairs, a, w, c, residual, m, n, k, epilogue, s);
        default: return launch_skinny_format<SknQ80>(enc, x, gain, eps, x_pairs, a, w, c, residual, m, n, k, epilogue, s);
    }
}

}  // namespace skh
