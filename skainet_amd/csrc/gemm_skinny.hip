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
//     through LDS. The next super-block's bytes are requested before the current one is decoded.
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
        const int tile = p >> 7, gr = 16 * (mt0 + tile / NT) + ((p >> 3) & 15), gc = n0 + 16 * (tile % NT) + 2 * (p & 7);
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
struct SknTile { int mt, nt; double us; };
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
    SknTile best{1, 1, 0.0};
    for (int i = 0; i < 6; ++i) {
        const int mt = shapes[i][0], nt = shapes[i][1];
        if (mt > 1 && mt >= 2 * mtiles) continue;                         // more rows than there are
        const double groups = (double)((mtiles + mt - 1) / mt) * ((n + 16 * nt - 1) / (16 * nt)) / num_cus();
        const double further = groups <= 1.0 ? 0.0 : whole[i] * ceil(groups) + (1 - whole[i]) * groups - 1;
        const double us = 3.9 + 2.06e-6 * m * k + 3.55e-6 * m * n +
                          (cost[i][0] + cost[i][1] * further) * ((1 - whole_k[i]) * shares + whole_k[i] * ceil(shares));
        if (best.us == 0.0 || us < best.us) best = SknTile{mt, nt, us};
    }
    return best;
}
double gemm_skinny_estimate(int enc, int m, int n, int k) { return gemm_skinny_tile(enc, m, n, k).us; }

static std::atomic<int> g_gemm_skinny{1};   // 0 never, 1 where the estimate favours it, 2 wherever it fits; 10 mt + nt: that tile, wherever it fits
void set_gemm_skinny(int v) { g_gemm_skinny = v; }
int gemm_skinny_mode() { return g_gemm_skinny.load(); }

template <class F>
static int launch_skinny_format(int enc, const float* x, const float* gain, float eps, bool pairs, uint8_t* a, const uint8_t* w, float* c,
                                const float* residual, int m, int n, int k, int epilogue, hipStream_t s) {
    if (skinny_prepass<F::Q6>(x, gain, eps, a, m, k, pairs, s) != 0) return -1;
    SknTile t = gemm_skinny_tile(enc, m, n, k);
    if (const int forced = g_gemm_skinny.load(); forced >= 11) { t.mt = forced / 10; t.nt = forced % 10; }
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
