// Packed-weight products of 2 to 8 activation rows (a few sequences decoded together, a draft), fp32 throughout:
//   y[b, o] = sum_j x[b, j] * dequant(W[o, j])      fp32 activations, weights decoded to fp32, fp32 products and sums.
// Semantics: m rows = m scalar GEMVs of the reference's exact-fp32 kernels,
//   skainet-backends/skainet-backend-cpu/src/commonMain/kotlin/sk/ainet/exec/kernel/PackedViewMatmulKernel.kt:69-108.
//
// What bounds it: one read of the weight, and next to it the decode (1.75 to 2.75 vector instructions per weight). The row
// kernel of gemv.hip multiplies on the vector unit, one instruction per weight and activation row, keeps four rows of
// activations per lane beside few weights in flight, and reads the weight a second time from five rows on. Here:
//   * v_mfma_f32_4x4x1 (16 blocks of 4 x 4, exact fp32 products) multiplies: lane l = 4 blk + j holds weights of row j of a
//     quad of weight rows and the activations of batch row j, both of K slot blk; one instruction takes 64 weights times
//     four batch rows in 4.2 ns (a vector instruction: 0.96), and the two kinds do not overlap.

//   * A slot is the 64 weights that one lane decodes (packed_lane64.h). Its activations (64 floats per four batch rows) stay
//     in registers while the wave walks the workgroup's rows; 16 slots are a pass of 1024 elements of K and the waves of a
//     workgroup share the passes. R quads of weight rows are requested ahead.
//   * The 16 blocks' sums fold inside a DPP row; the four DPP rows and the waves meet in LDS once, summed in a fixed order.
#include "packed_lane64.h"

#include <type_traits>

namespace skh {

typedef float few_f32x4 __attribute__((ext_vector_type(4)));

constexpr int FEW_MAX_ROWS = 64;      // weight rows of a workgroup (bounds the LDS sums)
constexpr int FEW_MAX_WAVES = 8;      // two per SIMD: 256 registers each

constexpr int FEW_STAGE_FLOATS = 2 * 16 * 68;      // two batch rows x 16 slots of 64 floats, each padded by four against bank conflicts

// MB: batch rows in fours (1 or 2), R: quads in flight.
template <class F, int MB, int R>
__global__ __launch_bounds__(64 * FEW_MAX_WAVES) void packed_gemv_few_kernel(const uint8_t* __restrict__ w, const float* __restrict__ x,
                                                                             float* __restrict__ y, int m, int n, int k, int rows_per_wg) {
    extern __shared__ __attribute__((aligned(16))) float few_smem[];      // [wave][FEW_STAGE_FLOATS], then [wave][row][DPP row][4 MB]
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), nwaves = blockDim.x >> 6;
    const int blk = lane >> 2, j = lane & 3, q = blk & 3;                 // a pass starts on a super-block: slot % 4 is the lane's own
    const int nsb = k >> 8, passes = (nsb + 3) >> 2;
    const uint32_t row_bytes = (uint32_t)nsb * F::BYTES;
    const int r0 = blockIdx.x * rows_per_wg;
    const int nrows = min(n - r0, rows_per_wg), quads = (nrows + 3) >> 2;
    float4* const stage = reinterpret_cast<float4*>(few_smem + (size_t)wave * FEW_STAGE_FLOATS);
    float* const few_part = few_smem + (size_t)nwaves * FEW_STAGE_FLOATS;
    float* const mine = few_part + (size_t)wave * rows_per_wg * 16 * MB;

    // Rounds of one pass per wave; where the last round has fewer passes than waves, several waves share one and its rows
    // (five waves would leave three of four SIMDs idle half the time: 4 x 30000 x 5120, Q4_0: 38 -> 27 us).
    for (int base = 0, round = 0; base < passes; base += nwaves, ++round) {
        const int left = min(passes - base, nwaves), teams = nwaves / left;
        if (wave >= teams * left) break;
        const int pass = base + wave % left, team = wave / left;
        const int q0 = quads * team / teams, q1 = quads * (team + 1) / teams;      // this wave's quads
        if (q0 == q1) break;
        // The wave's activations: whole kilobytes of a batch row per load (a lane's own 64 floats would take a line per lane
        // and load, 128 KB of a CU's waves through a 32 KB L1: Q4_0 4 x 14336 x 4096 16.9 -> 14.2 us), the first four rows in
        // front of the weights, whose loads must not hold them up; then through LDS into the lanes' order, two rows at a time.
        float4 xr[4][4];
        auto load_x = [&](int four, int b0) __attribute__((always_inline)) {     // two rows
#pragma unroll
            for (int b = b0; b < b0 + 2; ++b)
#pragma unroll
                for (int i = 0; i < 4; ++i)                               // past K and past m: copies of the last
                    xr[b][i] = *reinterpret_cast<const float4*>(x + (int64_t)min(4 * four + b, m - 1) * k + min(1024 * pass + 4 * (64 * i + lane), k - 4));
        };
        load_x(0, 0);
        load_x(0, 2);
        __builtin_amdgcn_sched_barrier(0);
        // super-blocks past the last are copies of it whose bytes and activations become zeros
        const int sb = 4 * pass + (blk >> 2);
        const bool in = sb < nsb, ragged = 4 * pass + 4 > nsb;
        const uint32_t off = (uint32_t)(in ? sb : nsb - 1) * F::BYTES;
        typename F::Raw raw[R];
        auto load = [&](int slot, int quad) __attribute__((always_inline)) {
            F::load(raw[slot], w + ((uint32_t)min(r0 + 4 * quad + j, n - 1) * row_bytes + off), q);      // rows past n: copies, never stored
        };
        load(0, q0);
        __builtin_amdgcn_sched_barrier(0);
        float xa[MB][64];
#pragma unroll
        for (int four = 0; four < MB; ++four) {
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                if (four) load_x(four, 2 * h);                            // two rows at a time: all eight at once would spill
#pragma unroll
                for (int b = 0; b < 2; ++b)
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const int f = 64 * i + lane;                      // float4 of the pass; slot f / 16
                        float4 v = xr[2 * h + b][i];
                        if (1024 * pass + 4 * f >= k) v = make_float4(0.f, 0.f, 0.f, 0.f);
                        stage[b * 272 + (f >> 4) * 17 + (f & 15)] = v;
                    }
                __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");    // wave-private: LDS serves a wave's accesses in order
                __builtin_amdgcn_wave_barrier();
                if ((j >> 1) == h) {
#pragma unroll
                    for (int u = 0; u < 8; ++u) {
                        const int f = 64 * (blk >> 2) + (skn_elem<F::Q6>(q, u) >> 2);
                        const float4* src = stage + (j & 1) * 272 + (f >> 4) * 17 + (f & 15);
                        const float4 lo = src[0], hi = src[1];
                        float* d = &xa[four][8 * u];
                        d[0] = lo.x; d[1] = lo.y; d[2] = lo.z; d[3] = lo.w; d[4] = hi.x; d[5] = hi.y; d[6] = hi.z; d[7] = hi.w;
                    }
                }
                __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
                __builtin_amdgcn_wave_barrier();
            }
        }
        // (the further quads only now: their registers held the activations)
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 1; i < R; ++i) load(i, min(q0 + i, q1 - 1));
        __builtin_amdgcn_sched_barrier(0);
        auto compute = [&](int slot, int quad) __attribute__((always_inline)) {
            constexpr int NA = 4 / MB;                                    // independent sums per four batch rows
            few_f32x4 acc[MB][NA];
#pragma unroll
            for (int b = 0; b < MB; ++b)
#pragma unroll
                for (int a = 0; a < NA; ++a) acc[b][a] = few_f32x4{0.f, 0.f, 0.f, 0.f};
            if (ragged && !in) __builtin_memset(&raw[slot], 0, sizeof(raw[slot]));      // zero times an infinite scale would be a NaN
            const typename F::Scales sc = F::scales(raw[slot], q);
            // Matrix and vector instructions do not overlap here and changing from one to the other costs 1 to 2 ns
            // (4x4x1 alone 4.2 ns; one and two multiply-adds in turn 7.8, of which the latter 1.9): the decode of 16 or 32
            // weights and their products stay apart (Q4_0, 4 x 14336 x 4096: 14.2 -> 12.2 us).
            constexpr int G = MB == 1 ? 4 : 2;                            // steps of eight weights at a time
            auto step = [&](auto uc) __attribute__((always_inline)) {
                constexpr int U = decltype(uc)::value;
                SknF32 o[G];
                F::template decode<U>(raw[slot], sc, o[0]);
                F::template decode<U + 1>(raw[slot], sc, o[1]);
                if constexpr (G == 4) { F::template decode<U + 2>(raw[slot], sc, o[2]); F::template decode<U + 3>(raw[slot], sc, o[3]); }
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int e = 0; e < 8 * G; ++e)
#pragma unroll
                    for (int b = 0; b < MB; ++b)
                        acc[b][e % NA] = __builtin_amdgcn_mfma_f32_4x4x1f32(xa[b][8 * U + e], o[e >> 3].w[e & 7], acc[b][e % NA], 0, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
            };
            step(std::integral_constant<int, 0>{});
            if constexpr (G == 2) step(std::integral_constant<int, 2>{});
            step(std::integral_constant<int, 4>{});
            if constexpr (G == 2) step(std::integral_constant<int, 6>{});
            // element e of lane (blk, j): batch row e, weight row j, K slot blk; the four blocks of a DPP row fold here
#pragma unroll
            for (int b = 0; b < MB; ++b) {
                few_f32x4 s = acc[b][0] + acc[b][1];
                if constexpr (NA == 4) s += acc[b][2] + acc[b][3];
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    s[e] += dpp_row_move<0x128>(s[e]);                    // row_ror:8
                    s[e] += dpp_row_move<0x124>(s[e]);                    // row_ror:4
                }
                if ((lane & 12) == 0) {
                    few_f32x4* dst = reinterpret_cast<few_f32x4*>(mine + ((4 * quad + j) * 4 + (lane >> 4)) * 4 * MB + 4 * b);
                    *dst = round == 0 ? s : *dst + s;
                }
            }
        };
        // no branch around a load in the main loop: behind one the wave would wait for everything in flight
        int t = q0;
        for (; t + R <= q1; t += R)
#pragma unroll
            for (int i = 0; i < R; ++i) {
                compute(i, t + i);
                load(i, min(t + i + R, q1 - 1));
            }
#pragma unroll
        for (int i = 0; i < R - 1; ++i)
            if (t + i < q1) compute(i, t + i);
    }
    __syncthreads();
    for (int at = threadIdx.x; at < rows_per_wg * 4 * MB; at += blockDim.x) {
        const int row = at % rows_per_wg, b = at / rows_per_wg;           // consecutive threads: consecutive outputs of a batch row
        if (row >= nrows || b >= m) continue;
        float s = 0.f;
        for (int v = 0; v < nwaves; ++v) {
            const float* src = few_part + (((size_t)v * rows_per_wg + row) * 4) * 4 * MB + b;
            s += (src[0] + src[4 * MB]) + (src[8 * MB] + src[12 * MB]);
        }
        y[(int64_t)b * n + r0 + row] = s;
    }
}

template <class F, int MB, int R>
static int launch_few_rows(const uint8_t* w, const float* x, float* y, int m, int n, int k) {
    const int passes = (k / 256 + 3) / 4;
    // a wave per pass up to four and for eight; else rounds of four or eight and a shared rest, so that the SIMDs get the same
    const int nwaves = passes <= 4 ? passes : passes < 8 ? 4 : FEW_MAX_WAVES;
    // whole rounds of workgroups over the chip, eight waves on a CU at a time, rows in fours
    const int resident = num_cus() * (FEW_MAX_WAVES / nwaves);
    const int turns = (int)(((int64_t)n + (int64_t)resident * FEW_MAX_ROWS - 1) / ((int64_t)resident * FEW_MAX_ROWS));
    const int rows = (int)(((int64_t)n + (int64_t)resident * turns - 1) / ((int64_t)resident * turns) + 3) & ~3;      // at most FEW_MAX_ROWS
    const size_t smem = (size_t)nwaves * (FEW_STAGE_FLOATS + rows * 16 * MB) * sizeof(float);
    SKH_SET_MAX_DYNAMIC_LDS_ONCE((&packed_gemv_few_kernel<F, MB, R>), (size_t)FEW_MAX_WAVES * (FEW_STAGE_FLOATS + FEW_MAX_ROWS * 16 * MB) * sizeof(float));
    note_kernel("packed_gemv_few_kernel");
    packed_gemv_few_kernel<F, MB, R><<<dim3((n + rows - 1) / rows), dim3(64 * nwaves), smem, current_stream()>>>(w, x, y, m, n, k, rows);
    SKH_CHECK(hipGetLastError());
    return 1;
}
// Three quads ahead, or two beside the activations of eight rows. (Four to six for four rows: the same to 6 % slower.)
template <class F>
static int launch_few(const uint8_t* w, const float* x, float* y, int m, int n, int k) {
    return m > 4 ? launch_few_rows<F, 2, 2>(w, x, y, m, n, k) : launch_few_rows<F, 1, 3>(w, x, y, m, n, k);
}

static std::atomic<int> g_gemv_few{1};      // 0 never, 1 by rule, 2 wherever it fits
void set_gemv_few(int v) { g_gemv_few = v; }

// Where this kernel is faster than the row kernel, measured over n 1500 to 32000, K 512 to 14336 (row kernel -> this one, us).
// Three rows and more of a format of 32-element blocks: everywhere (Q8_0 4 x 4096 x 11008 26.1 -> 14.9, 8 x 32000 x 4096
// 111 -> 41; Q4_0 3 x 4000 x 512 5.8 -> 4.3). The row kernel holds its own where it multiplies little and loads well:
//   * two rows, half of this kernel's products for nothing: only with enough rows of weights per wave to cover the start, and
//     K beyond the row kernel's eight full waves (Q5_K 2 x 10000 x 12800 44.5 -> 33.4, but x 8192 16.0 -> 19.3), or for the
//     32-element blocks its two (Q8_0 2 x 14336 x 4096 17.3 -> 15.0, x 2048 7.7 -> 9.5);
//   * the K-quants, whose lanes decode more per byte: few weight rows with a K that takes this kernel a shared round (Q6_K
//     5 x 1500 x 7168 13.2 -> 15.0, x 8192 13.6 -> 11.4), and Q6_K up to four rows outside 4096 < K <= 6144 and K > 8192
//     (4 x 14336 x 4096 15.9 -> 16.8, 3 x 10000 x 11008 49.5 -> 30.4);
//   * Q4_K has batched kernels of its own (K 4096; any K): this one on rows shorter than a wave's share there (8 x 30000 x 512
//     35.5 -> 12.6, 3 x 4000 x 2048 6.3 -> 5.5; 4 x 10000 x 2560 8.4 -> 9.4) and on few long ones (4 x 2048 x 14336 15.3 -> 10.9;
//     4 x 10000 x 14336 27.3 -> 28.3).
static bool few_by_rule(int enc, int m, int n, int k) {
    const bool block32 = block_elems(enc) == 32, many = n >= 12 * num_cus();
    if (enc == ENC_Q4_K) {
        if (m == 2) return many && k <= 1280;
        return k <= 2048 || (n < 20 * num_cus() && k > 4096 && (k <= 5120 || k > 7168));
    }
    if (m == 2) return many && (k > 8192 || (block32 && k > 2048 && k <= 5120));
    if (block32) return true;
    if (m >= 5) return many || k <= 4096 || (k > 7168 && k <= 12288);
    if (enc == ENC_Q5_K) return many || k <= 4096;
    return k <= 768 || (many && (k > 8192 || (k > 4096 && k <= 6144)));
}

// Returns 1 when this kernel took the product, 0 when the row kernel is the faster one or the shape is outside its range, -1 on
// a launch error.
int launch_gemv_few(int enc, const uint8_t* w, const float* x, float* y, int m, int n, int k) {
    const int mode = g_gemv_few.load();
    if (!mode || m < 2 || m > 8 || n < 1 || k < 256 || k % 256 != 0) return 0;
    if ((reinterpret_cast<uintptr_t>(w) | reinterpret_cast<uintptr_t>(x)) & 15) return 0;
    if ((uint64_t)n * (uint64_t)(k / block_elems(enc)) * block_bytes(enc) >= ((uint64_t)1 << 32)) return 0;      // 32-bit byte offsets
    if (mode == 1 && !few_by_rule(enc, m, n, k)) return 0;
    switch (enc) {
        case ENC_Q4_K: return launch_few<SknQ4K>(w, x, y, m, n, k);
        case ENC_Q5_K: return launch_few<SknQ5K>(w, x, y, m, n, k);
        case ENC_Q6_K: return launch_few<SknQ6K>(w, x, y, m, n, k);
        case ENC_Q8_0: return launch_few<SknQ80>(w, x, y, m, n, k);
        case ENC_Q4_0: return launch_few<SknQ45<0>>(w, x, y, m, n, k);
        case ENC_Q5_0: return launch_few<SknQ45<1>>(w, x, y, m, n, k);
        case ENC_Q5_1: return launch_few<SknQ45<2>>(w, x, y, m, n, k);
        default: return 0;
    }
}

}  // namespace skh
