// Packed-weight products of 1 to 8 activation rows (a few sequences decoded together, a draft), fp32 throughout:
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
//   * One and two rows would leave the instruction half empty: the vector unit multiplies, same lanes and loads (Q8_0
//     2 x 10000 x 4096 13.9 us on the row kernel, 10.7 here; 2 x 4096 x 11008 16.5 on the matrix instruction, 13.0 at n 4000 here).
//   * The 16 blocks' sums fold inside a DPP row; the four DPP rows and the waves meet in LDS once, summed in a fixed order.
#include "packed_lane64.h"

#include <type_traits>

namespace skh {

typedef float few_f32x4 __attribute__((ext_vector_type(4)));

constexpr int FEW_MAX_ROWS = 64;      // weight rows of a workgroup (bounds the LDS sums)
constexpr int FEW_MAX_WAVES = 8;      // two per SIMD: 256 registers each

constexpr int FEW_STAGE_FLOATS = 2 * 16 * 68;      // two batch rows x 16 slots of 64 floats, each padded by four against bank conflicts

// ROWS: batch rows computed (4 or 8 on the matrix instruction; 1 or 2 on the vector unit, every lane with the rows' activations of
// its slot), R: quads in flight.
template <class F, int ROWS, int R, int WAVES = FEW_MAX_WAVES>
__global__ __launch_bounds__(64 * WAVES) void packed_gemv_few_kernel(const uint8_t* __restrict__ w, const float* __restrict__ x,
                                                                             float* __restrict__ y, int m, int n, int k, int rows_per_wg) {
    constexpr bool VECTOR = ROWS <= 2;
    constexpr int MB = VECTOR ? 1 : ROWS / 4, NX = VECTOR ? ROWS : MB;    // batch rows in fours; sets of 64 activations in a lane
    extern __shared__ __attribute__((aligned(16))) float few_smem[];      // [wave][FEW_STAGE_FLOATS], then [wave][row][DPP row][ROWS]
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), nwaves = blockDim.x >> 6;
    const int blk = lane >> 2, j = lane & 3, q = blk & 3;                 // a pass starts on a super-block: slot % 4 is the lane's own
    const int nsb = k >> 8, passes = (nsb + 3) >> 2;
    const uint32_t row_bytes = (uint32_t)nsb * F::BYTES;
    const int r0 = blockIdx.x * rows_per_wg;
    const int nrows = min(n - r0, rows_per_wg), quads = (nrows + 3) >> 2;
    float4* const stage = reinterpret_cast<float4*>(few_smem + (size_t)wave * FEW_STAGE_FLOATS);
    float* const few_part = few_smem + (size_t)nwaves * FEW_STAGE_FLOATS;
    float* const mine = few_part + (size_t)wave * rows_per_wg * 4 * ROWS;

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
        constexpr int PAIR = ROWS < 2 ? ROWS : 2;
        float4 xr[VECTOR ? PAIR : 4][4];
        auto load_x = [&](int four, int b0) __attribute__((always_inline)) {     // two rows
#pragma unroll
            for (int b = b0; b < b0 + PAIR; ++b)
#pragma unroll
                for (int i = 0; i < 4; ++i)                               // past K and past m: copies of the last
                    xr[b][i] = *reinterpret_cast<const float4*>(x + (int64_t)min(4 * four + b, m - 1) * k + min(1024 * pass + 4 * (64 * i + lane), k - 4));
        };
        load_x(0, 0);
        if constexpr (!VECTOR) load_x(0, 2);
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
        float xa[NX][64];
#pragma unroll
        for (int four = 0; four < MB; ++four) {
#pragma unroll
            for (int h = 0; h < (VECTOR ? 1 : 2); ++h) {
                if (four) load_x(four, 2 * h);                            // two rows at a time: all eight at once would spill
#pragma unroll
                for (int b = 0; b < PAIR; ++b)
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const int f = 64 * i + lane;                      // float4 of the pass; slot f / 16
                        float4 v = xr[2 * h + b][i];
                        if (1024 * pass + 4 * f >= k) v = make_float4(0.f, 0.f, 0.f, 0.f);
                        stage[b * 272 + (f >> 4) * 17 + (f & 15)] = v;
                    }
                __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");    // wave-private: LDS serves a wave's accesses in order
                __builtin_amdgcn_wave_barrier();
                auto take = [&](float (&d)[64], int row) __attribute__((always_inline)) {      // the lane's slot of a staged row
#pragma unroll
                    for (int u = 0; u < 8; ++u) {
                        const int f = 64 * (blk >> 2) + (skn_elem<F::Q6>(q, u) >> 2);
                        const float4* src = stage + row * 272 + (f >> 4) * 17 + (f & 15);
                        const float4 lo = src[0], hi = src[1];
                        d[8 * u] = lo.x; d[8 * u + 1] = lo.y; d[8 * u + 2] = lo.z; d[8 * u + 3] = lo.w;
                        d[8 * u + 4] = hi.x; d[8 * u + 5] = hi.y; d[8 * u + 6] = hi.z; d[8 * u + 7] = hi.w;
                    }
                };
                if constexpr (VECTOR) {
#pragma unroll
                    for (int b = 0; b < ROWS; ++b) take(xa[b], b);
                } else {
                    if ((j >> 1) == h) take(xa[four], j & 1);
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
            if (ragged && !in) __builtin_memset(&raw[slot], 0, sizeof(raw[slot]));      // zero times an infinite scale would be a NaN
            const typename F::Scales sc = F::scales(raw[slot], q);
            float* const dst = mine + ((4 * quad + j) * 4 + (lane >> 4)) * ROWS;          // the four blocks of a DPP row fold in registers
            if constexpr (VECTOR) {
                float acc[ROWS][4];
#pragma unroll
                for (int b = 0; b < ROWS; ++b) acc[b][0] = acc[b][1] = acc[b][2] = acc[b][3] = 0.f;
                auto step = [&](auto uc) __attribute__((always_inline)) {
                    constexpr int U = decltype(uc)::value;
                    SknF32 o;
                    F::template decode<U>(raw[slot], sc, o);
#pragma unroll
                    for (int e = 0; e < 8; ++e)
#pragma unroll
                        for (int b = 0; b < ROWS; ++b) acc[b][e & 3] = fmaf(xa[b][8 * U + e], o.w[e], acc[b][e & 3]);
                    __builtin_amdgcn_sched_barrier(0);
                };
                step(std::integral_constant<int, 0>{}); step(std::integral_constant<int, 1>{});
                step(std::integral_constant<int, 2>{}); step(std::integral_constant<int, 3>{});
                step(std::integral_constant<int, 4>{}); step(std::integral_constant<int, 5>{});
                step(std::integral_constant<int, 6>{}); step(std::integral_constant<int, 7>{});
#pragma unroll
                for (int b = 0; b < ROWS; ++b) {
                    float s = (acc[b][0] + acc[b][1]) + (acc[b][2] + acc[b][3]);
                    s += dpp_row_move<0x128>(s);                          // row_ror:8
                    s += dpp_row_move<0x124>(s);                          // row_ror:4
                    if ((lane & 12) == 0) dst[b] = round == 0 ? s : dst[b] + s;
                }
            } else {
                constexpr int NA = 4 / MB;                                // independent sums per four batch rows
                few_f32x4 acc[MB][NA];
#pragma unroll
                for (int b = 0; b < MB; ++b)
#pragma unroll
                    for (int a = 0; a < NA; ++a) acc[b][a] = few_f32x4{0.f, 0.f, 0.f, 0.f};
                // Matrix and vector instructions do not overlap here and changing from one to the other costs 1 to 2 ns
                // (4x4x1 alone 4.2 ns; one and two multiply-adds in turn 7.8, of which the latter 1.9): the decode of 16 or 32
                // weights and their products stay apart (Q4_0, 4 x 14336 x 4096: 14.2 -> 12.2 us).
                constexpr int G = MB == 1 ? 4 : 2;                        // steps of eight weights at a time
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
                // element e of lane (blk, j): batch row e, weight row j, K slot blk
#pragma unroll
                for (int b = 0; b < MB; ++b) {
                    few_f32x4 s = acc[b][0] + acc[b][1];
                    if constexpr (NA == 4) s += acc[b][2] + acc[b][3];
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        s[e] += dpp_row_move<0x128>(s[e]);                // row_ror:8
                        s[e] += dpp_row_move<0x124>(s[e]);                // row_ror:4
                    }
                    if ((lane & 12) == 0) {
                        few_f32x4* const d4 = reinterpret_cast<few_f32x4*>(dst) + b;
                        *d4 = round == 0 ? s : *d4 + s;
                    }
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
    for (int at = threadIdx.x; at < rows_per_wg * ROWS; at += blockDim.x) {
        const int row = at % rows_per_wg, b = at / rows_per_wg;           // consecutive threads: consecutive outputs of a batch row
        if (row >= nrows || b >= m) continue;
        float s = 0.f;
        for (int v = 0; v < nwaves; ++v) {
            const float* src = few_part + (((size_t)v * rows_per_wg + row) * 4) * ROWS + b;
            s += (src[0] + src[ROWS]) + (src[2 * ROWS] + src[3 * ROWS]);
        }
        y[(int64_t)b * n + r0 + row] = s;
    }
}

template <class F, int ROWS, int R, int WAVES = FEW_MAX_WAVES>
static int launch_few_rows(const uint8_t* w, const float* x, float* y, int m, int n, int k) {
    const int passes = (k / 256 + 3) / 4;
    const int cus = num_cus();
    // 9 to 12 passes: as many waves, in the registers of three per SIMD (two quads ahead instead of three or four), so that no wave has to
    // load activations a second time (Q8_0 4 x 4096 x 11008 15.1 -> 13.0 us, Q4_K 4 x 8000 x 12288 20.3 -> 18.7). Eight batch rows and Q6_K
    // do not fit there; nine passes leave three SIMDs of four two waves, which costs more than it saves from 24 rows per CU on.
    if constexpr ((ROWS == 4 || ROWS == 1) && WAVES == FEW_MAX_WAVES && !F::Q6) {
        if (passes > 8 && passes <= 12 && (passes > 9 || n <= 24 * cus)) return launch_few_rows<F, ROWS, 2, 12>(w, x, y, m, n, k);
    }
    // A wave per pass up to four and for eight. Five to seven: one workgroup per CU with a wave per pass while the one round of activations
    // outweighs the SIMDs with one wave of two (five, six and seven passes up to 16, 32 and 64 rows per CU: Q6_K 2 x 3000 x 6144 0.77 of its time,
    // 8 x 2000 x 7168 0.76); else two of four, the second round shared. From there on rounds of eight and a shared rest.
    const bool one_round = passes == 5 ? n <= 16 * cus : passes == 6 ? n <= 32 * cus : n <= 64 * cus;
    const int nwaves = WAVES == 12 || passes <= 4 || (passes < 8 && one_round) ? passes : passes < 8 ? 4 : FEW_MAX_WAVES;
    // whole rounds of workgroups over the chip, eight waves on a CU at a time, rows in fours
    const int resident = cus * (WAVES / nwaves);
    const int turns = (int)(((int64_t)n + (int64_t)resident * FEW_MAX_ROWS - 1) / ((int64_t)resident * FEW_MAX_ROWS));
    const int rows = (int)(((int64_t)n + (int64_t)resident * turns - 1) / ((int64_t)resident * turns) + 3) & ~3;      // at most FEW_MAX_ROWS
    const size_t smem = (size_t)nwaves * (FEW_STAGE_FLOATS + rows * 4 * ROWS) * sizeof(float);
    SKH_SET_MAX_DYNAMIC_LDS_ONCE((&packed_gemv_few_kernel<F, ROWS, R, WAVES>), (size_t)WAVES * (FEW_STAGE_FLOATS + FEW_MAX_ROWS * 4 * ROWS) * sizeof(float));
    note_kernel("packed_gemv_few_kernel");
    packed_gemv_few_kernel<F, ROWS, R, WAVES><<<dim3((n + rows - 1) / rows), dim3(64 * nwaves), smem, current_stream()>>>(w, x, y, m, n, k, rows);
    SKH_CHECK(hipGetLastError());
    return 1;
}
// Quads ahead: what the registers hold beside the activations. (Four to six for four rows: the same to 6 % slower.)
template <class F>
static int launch_few(const uint8_t* w, const float* x, float* y, int m, int n, int k) {
    if (m == 1) return launch_few_rows<F, 1, 4>(w, x, y, m, n, k);
    if (m == 2) return launch_few_rows<F, 2, 2>(w, x, y, m, n, k);
    return m > 4 ? launch_few_rows<F, 8, 2>(w, x, y, m, n, k) : launch_few_rows<F, 4, 3>(w, x, y, m, n, k);
}

static std::atomic<int> g_gemv_few{1};      // 0 never, 1 by rule, 2 wherever it fits
void set_gemv_few(int v) { g_gemv_few = v; }

// Where this kernel is faster than the ones behind it (row kernel; for one row of 32-element blocks the streaming kernel and Q8_0's
// integer kernel; Q4_K's own kernels), from 91 000 random products of n 512 to 32000, K 512 to 15360, in us, theirs -> this one's. It is
// where they multiply much or load badly: many activation rows, rows of few kilobytes, K that leaves their waves unequal shares. They
// hold their own with few products on full waves, and where K takes this kernel a second round that few waves share (5120 to 7168).
//   32-element blocks, 3 to 8 rows: everywhere (Q8_0 4 x 4096 x 11008 26.1 -> 14.6, 8 x 32000 x 4096 111 -> 41)
//     2 rows: outside 6144 < K <= 7168 (Q4_0 4000 x 4096 7.2 -> 5.3, 4000 x 8192 9.6 -> 8.0, Q8_0 10000 x 4096 13.9 -> 10.7, x 7168 16.2 ->
//     17.2)
//     1 row, formats of 4 and 5 bits: K up to 4096 (Q5_0 6800 x 768 6.9 -> 4.5, 1780 x 3072 5.6 -> 4.6, 30000 x 4096 27.7 -> 20.7), and beyond
//     the streaming kernel's K (Q5_0 620 x 15100 9.6 -> 6.5; Q4_0 4000 x 11008 11.7 -> 9.9; Q5_1 31331 x 14080 73 -> 85). Rows of 4096
//     and 8192 fill the waves of the kernels behind: those stay there up to 48 rows per CU (Q4_0 4096 x 4096 5.9, here 5.1)
//     1 row of Q8_0: many short rows and between the integer kernel's K (30000 x 768 10.5 -> 7.3, 12170 x 2560 12.7 -> 10.5)
//   Q6_K, Q5_K: their decode costs more, so 5 to 8 rows (Q6_K 8 x 4096 x 11008 53 -> 24, Q5_K 8 x 3000 x 13312 30.6 -> 20.6; Q6_K 5 x 1500 x 7168
//     13.2 -> 15.0), 3 and 4 of Q5_K, and below that rows that leave the row kernel's lanes idle (Q6_K 1 x 30000 x 768 18.0 -> 10.0, Q5_K 2 x
//     30800 x 1024 13.0 -> 8.9, 2 x 10000 x 11008 36.6 -> 25.6; 4 x 14336 x 4096 15.9 -> 16.8)
//   Q4_K: rows shorter than a wave's share there (1 x 31600 x 512 12.2 -> 7.0, 8 x 30000 x 512 35.5 -> 12.6), long ones (4 x 2048 x 14336 15.3 ->
//     10.9, 5 x 13000 x 9216 61.6 -> 36.1; 4 x 10000 x 14336 27.3 -> 28.3), and more rows than their workgroups take in whole rounds (8 x 15000 x
//     3328 28 -> 21). K = 4096 has kernels for its four full slices (8 x 15000 x 4096 13.5 -> 21.8).
// Where it is slower it stays, for its error against float64 is a third of the row kernel's (1.1e-7 against 3e-7 to 5e-7) and
// a fortieth of the bf16 quads' (4e-6): Q5_K 1 row, Q6_K 2 to 4 rows, 32-element blocks 1 and 2 rows, K above 8192 (Q5_K 3500 x 10240 10.4 ->
// 15.8, Q6_K 2 x 3300 x 12800 12.3 -> 17.9, Q5_1 7300 x 14848 18.3 -> 24.2), Q4_K 3 and 4 rows below 1024 x 2048 (4.5 -> 4.7 to 5.4).
// Besides: rows go in fours per workgroup, so a little more than 16 per CU costs a quarter (Q6_K 4 x 4147 x 6144 13.6 -> 16.2, x 4000
// 12.1 -> 12.2), and products of 4 us are as long as their launch on either side (within 0.3 us).
static bool few_by_rule(int enc, int m, int n, int k) {
    const int cus = num_cus();
    const bool many = n >= 12 * cus, lots = n >= 48 * cus, uneven = n > 16 * cus && n < 24 * cus;
    if (enc == ENC_Q4_K) {
        const bool third = n > 48 * cus && n <= 64 * cus;                 // a third round of the kernels behind, the first one here
        if (m == 1) {
            if (k <= 1024) return n >= (k <= 768 ? 24 : 32) * cus;
            return k % 1024 != 0 && (k <= 2048 ? n >= 24 * cus : k > 4096 && k <= 5120 && n > 64 * cus);      // K % 1024 = 0: the integer kernel
        }
        if (k <= 2048) return m > 2 || many;
        if (k <= 4096) return k < 4096 && (m > 4 ? third || (k <= 3072 && lots) : m > 2 && n <= 8 * cus);
        if (k <= 5120) return true;
        if (k <= 6144) return m == 2 || n <= 16 * cus || n > 48 * cus;
        if (k <= 7168) return m > 2 && (n <= (m <= 4 ? 8 : 4) * cus || third);
        if (n < 24 * cus || (m > 2 && third && k <= 11264)) return true;
        const int most = m == 2 ? 64 : k <= 9216 && m <= 4 ? 64 : 32;
        return k > 8192 && k <= 10240 && n <= most * cus;
    }
    if (block_elems(enc) == 32) {
        if (m >= 3) return true;
        if (m == 2) {
            if (k <= 1024) return many;
            if (enc == ENC_Q8_0 && k <= 2048) return !lots;
            if (k > 7168 && k <= 8192) return n <= (enc == ENC_Q8_0 ? 12 : 64) * cus;
            return k <= 4096 || (n >= 4 * cus && k <= 6144) || (k > 8192 && (k <= 12288 || !lots));
        }
        if (enc == ENC_Q8_0) return k % 1024 != 0 && (k <= 768 ? n >= 32 * cus : k <= 1536 ? n > 64 * cus : k > 2048 && k <= 4096 && many);
        if (k <= 2048) return n >= (enc == ENC_Q5_0 && k > 1024 ? 16 : 24) * cus;
        if (k <= 4096) return n >= (k == 4096 ? 48 : 5) * cus;
        if (k > 7168 && k < 8192) return enc == ENC_Q4_0 ? n <= 64 * cus : !many;
        if (k > 8192 && enc != ENC_Q5_1 && (many ? k <= 10240 : k > 10240 || n <= 4 * cus || n > 6 * cus)) return true;
        return many && !lots && (k <= 6144 || k > 8192);
    }
    if (m >= 5) {
        if (enc == ENC_Q5_K && (m >= 6 || k <= 12288 || n >= 6 * cus)) return true;
        if (enc == ENC_Q6_K && m >= 7 && !(k > 6144 && k <= 7168)) return true;
        return many || k <= 4096 || (k > 7168 && k <= 11264);
    }
    if (m >= 3 && enc == ENC_Q5_K) return k <= 4096 || (k > 7168 && k <= 8192) || (many && !(uneven && k <= 8192));
    const bool q5k_3072 = enc == ENC_Q5_K && k > 2048 && k <= 3072;       // the row kernel's second wave half empty
    if (!many) return m >= 2 && (k <= 1024 || q5k_3072) && n >= 4 * cus;
    if (m == 1 && enc == ENC_Q6_K) return k <= 768 || (k <= 1792 && n >= 32 * cus);
    if (m == 1) return k <= 1024 ? n >= 32 * cus : k > 8192 && k <= 12288 && (!lots || k <= 10240);
    if (m == 2 && q5k_3072 && n <= 24 * cus) return true;
    return k <= 1024 || (k > 8192 && (k <= 12288 || !lots)) || (k > 4096 && k <= (m == 2 ? 5120 : 6144) && !uneven);
}

// Returns 1 when this kernel took the product, 0 when the row kernel is the faster one or the shape is outside its range, -1 on
// a launch error.
int launch_gemv_few(int enc, const uint8_t* w, const float* x, float* y, int m, int n, int k) {
    const int mode = g_gemv_few.load();
    if (!mode || m < 1 || m > 8 || n < 1 || k < 256 || k % 256 != 0) return 0;
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
