// Dense fp32 matmul entries of the kernel SPI. No decoder configuration routes through them (every linear layer
// there is packed). Three kernels:
//   sgemm_mfma_skinny_kernel  fp32 operands on v_mfma_f32_16x16x4_f32, K split over the waves of a workgroup and nothing
//                      staged through LDS: products whose 64 x 128 tiles would leave CUs idle (few rows, or few columns
//                      with a long K), any stride, alignment and remainder;
//   sgemm_mfma_kernel  fp32 operands on the fp32 matrix instruction (v_mfma_f32_32x32x2_f32: exact fp32 products, fp32
//                      accumulation), 128 x 128 x 16 tiles, for products of at least 64 rows whose operands are 16-byte
//                      aligned with strides and K (and N, when B is read along its rows) multiples of four;
//   sgemm_kernel       everything else (any stride and alignment, bf16 / fp16 B): an LDS-tiled SGEMM, 64 x 64 output
//                      tile per workgroup, 16-deep K slices, 4 x 4 outputs per thread, fp32 FMA accumulation in
//                      ascending k.
//
//   fp32_matmul     C(m,n) = A(m,k) B(k,n), row strides in floats, full overwrite (k == 0 zeroes C)
//                   /root/reference/skainet-backends/skainet-backend-native-cpu/native/include/skainet_kernels.h:262-276
//   fp32_matmul_wt  out[i,o] = sum_p in[i,p] * w[o,p]
//                   /root/reference/skainet-backends/skainet-backend-native-cpu/native/include/skainet_kernels.h:495-515
//   bf16 / fp16 matmul  C(m,n) = A(m,k) B(k,n) with B two bytes per element, byte row stride (bf16: the high half of
//                   an fp32; fp16: IEEE binary16), same tile kernel with the decode in the tile load
//                   /root/reference/skainet-backends/skainet-backend-native-cpu/native/include/skainet_kernels.h:278-312
#include "common.h"

namespace skh {

constexpr int DT = 64, DK = 16;

// BK 0: B(p, j) = b[p * b_stride + j];  BK 1: B(p, j) = b[j * b_stride + p] (x . W^T);
// BK 2 / 3: B(p, j) = bf16 / fp16 at byte p * b_stride + 2 j of b (b_stride in bytes, any alignment: read bytewise).
template <int BK>
__global__ __launch_bounds__(256) void sgemm_kernel(const float* __restrict__ a, int64_t a_stride, const float* __restrict__ b,
                                                    int64_t b_stride, float* __restrict__ c, int64_t c_stride, int m, int n, int k) {
    constexpr bool BT = BK == 1;
    __shared__ float as[DK][DT + 1];
    __shared__ float bs[DK][DT + 1];
    const int tx = threadIdx.x & 15, ty = threadIdx.x >> 4;
    const int i0 = blockIdx.y * DT, j0 = blockIdx.x * DT;
    float acc[4][4] = {};
    for (int p0 = 0; p0 < k; p0 += DK) {
        for (int t = threadIdx.x; t < DT * DK; t += 256) {
            // A tile: row i (64) x depth p (16), read along p
            const int ai = t / DK, ap = t % DK;
            as[ap][ai] = (i0 + ai < m && p0 + ap < k) ? a[(int64_t)(i0 + ai) * a_stride + p0 + ap] : 0.f;
            if (BT) {
                const int bj = t / DK, bp = t % DK;
                bs[bp][bj] = (j0 + bj < n && p0 + bp < k) ? b[(int64_t)(j0 + bj) * b_stride + p0 + bp] : 0.f;
            } else if (BK == 0) {
                const int bp = t / DT, bj = t % DT;
                bs[bp][bj] = (j0 + bj < n && p0 + bp < k) ? b[(int64_t)(p0 + bp) * b_stride + j0 + bj] : 0.f;
            } else {
                const int bp = t / DT, bj = t % DT;
                float v = 0.f;
                if (j0 + bj < n && p0 + bp < k) {
                    const uint8_t* e = reinterpret_cast<const uint8_t*>(b) + (int64_t)(p0 + bp) * b_stride + 2 * (j0 + bj);
                    const uint32_t h = (uint32_t)e[0] | ((uint32_t)e[1] << 8);
                    v = BK == 2 ? __uint_as_float(h << 16) : half_bits_to_float(h);
                }
                bs[bp][bj] = v;
            }
        }
        __syncthreads();
#pragma unroll
        for (int p = 0; p < DK; ++p) {
            float av[4], bv[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) { av[r] = as[p][ty * 4 + r]; bv[r] = bs[p][tx * 4 + r]; }
#pragma unroll
            for (int r = 0; r < 4; ++r)
#pragma unroll
                for (int s = 0; s < 4; ++s) acc[r][s] = fmaf(av[r], bv[s], acc[r][s]);
        }
        __syncthreads();
    }
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            const int i = i0 + ty * 4 + r, j = j0 + tx * 4 + s;
            if (i < m && j < n) c[(int64_t)i * c_stride + j] = acc[r][s];
        }
}

// fp32 on the matrix cores. Workgroup tile 64 WM x 128 (WM = 2: 128 x 128; WM = 1: 64 x 128, for products whose taller
// tiles would leave CUs idle), K slices of 16; four waves in 2 x 2, each 32 WM x 64 outputs as WM x 2 tiles of 32 x 32. A slice goes global -> registers (requested a slice ahead) -> LDS
// (two stages, one barrier per slice) with K as the slow index of both tiles: the matrix instruction's operands are
// one float per lane -- row (or column) lane % 32 at depth lane / 32 of a two-deep step -- so a wave reads 32
// consecutive floats of two tile rows. BT: B(p, j) = b[j * b_stride + p] (x . W^T), else b[p * b_stride + j].
constexpr int MT = 128, MK = 16, MP = MT + 4;      // tile edge, slice depth, LDS row pitch in floats (16-byte rows)
typedef float dense_f32x16 __attribute__((ext_vector_type(16)));

template <bool BT, int WM>
__global__ __launch_bounds__(256) void sgemm_mfma_kernel(const float* __restrict__ a, int64_t a_stride, const float* __restrict__ b,
                                                         int64_t b_stride, float* __restrict__ c, int64_t c_stride, int m, int n, int k) {
    __shared__ __attribute__((aligned(16))) float as[2][MK][MP];
    __shared__ __attribute__((aligned(16))) float bs[2][MK][MP];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wm = wave >> 1, wn = wave & 1;
    const int i0 = blockIdx.y * (64 * WM), j0 = blockIdx.x * MT;
    // loads of a slice: "row-like" operands (A, and B when transposed) 128 rows x 4 float4 along K, two per thread;
    // B read along its rows: 16 depths x 32 float4, two per thread
    const int lr = tid >> 2, lq = tid & 3;            // row (+ 64 j), float4 along K
    const int bp = tid >> 5, bq = tid & 31;           // depth (+ 8 j), float4 along N
    float4 ra[WM], rb[2];
    auto load_slice = [&](int p0) {
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int row = i0 + lr + 64 * j, p = p0 + 4 * lq;
            if (j < WM) ra[j] = (row < m && p < k) ? *reinterpret_cast<const float4*>(a + (int64_t)row * a_stride + p) : make_float4(0.f, 0.f, 0.f, 0.f);
            if (BT) {
                const int col = j0 + lr + 64 * j;
                rb[j] = (col < n && p < k) ? *reinterpret_cast<const float4*>(b + (int64_t)col * b_stride + p) : make_float4(0.f, 0.f, 0.f, 0.f);
            } else {
                const int pp = p0 + bp + 8 * j, col = j0 + 4 * bq;
                rb[j] = (pp < k && col < n) ? *reinterpret_cast<const float4*>(b + (int64_t)pp * b_stride + col) : make_float4(0.f, 0.f, 0.f, 0.f);
            }
        }
    };
    auto store_slice = [&](int buf) {
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int r = lr + 64 * j;
            if (j < WM) { as[buf][4 * lq][r] = ra[j].x; as[buf][4 * lq + 1][r] = ra[j].y; as[buf][4 * lq + 2][r] = ra[j].z; as[buf][4 * lq + 3][r] = ra[j].w; }
            if (BT) {
                bs[buf][4 * lq][r] = rb[j].x; bs[buf][4 * lq + 1][r] = rb[j].y; bs[buf][4 * lq + 2][r] = rb[j].z; bs[buf][4 * lq + 3][r] = rb[j].w;
            } else {
                *reinterpret_cast<float4*>(&bs[buf][bp + 8 * j][4 * bq]) = rb[j];
            }
        }
    };
    dense_f32x16 acc[WM][2];
#pragma unroll
    for (int i = 0; i < WM; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;
    const int nsl = (k + MK - 1) / MK;
    if (nsl > 0) { load_slice(0); store_slice(0); }
    __syncthreads();
    const int col = lane & 31, dh = lane >> 5;
    for (int sl = 0; sl < nsl; ++sl) {
        const int buf = sl & 1;
        if (sl + 1 < nsl) load_slice((sl + 1) * MK);
#pragma unroll
        for (int s2 = 0; s2 < MK / 2; ++s2) {
            float av[WM], bv[2];
#pragma unroll
            for (int i = 0; i < WM; ++i) av[i] = as[buf][2 * s2 + dh][wm * (32 * WM) + 32 * i + col];
#pragma unroll
            for (int i = 0; i < 2; ++i) bv[i] = bs[buf][2 * s2 + dh][wn * 64 + 32 * i + col];
#pragma unroll
            for (int i = 0; i < WM; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(av[i], bv[j], acc[i][j], 0, 0, 0);
        }
        if (sl + 1 < nsl) store_slice(buf ^ 1);
        __syncthreads();
    }
    // accumulator element e of lane l: row 8 (e / 4) + 4 (l / 32) + e % 4, column l % 32 of its 32 x 32 tile
#pragma unroll
    for (int i = 0; i < WM; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                const int row = i0 + wm * (32 * WM) + 32 * i + 8 * (e >> 2) + 4 * dh + (e & 3), cc = j0 + wn * 64 + 32 * j + col;
                if (row < m && cc < n) c[(int64_t)row * c_stride + cc] = acc[i][j][e];
            }
}

// Few rows (or few output columns with a long K): what bounds these products is the one read of the weight, and with
// 64-wide tiles it was latency -- 32 x 4096 x 4096 is 64 tiles, each a chain of 256 K slices behind barriers (720 us).
// Here a workgroup owns 16 NT output columns x 16 MTILES rows and its NW waves split K, 32 elements at a time in turn,
// so that the workgroup reads NW x 128 consecutive bytes of each of its weight rows per round; 4096 columns are 256
// workgroups. Operands go from global memory straight into the matrix instruction's registers: lane (r, q) = (l % 16,
// l / 16) loads floats 4 q .. 4 q + 3 and 16 + 4 q .. of a step of row r of either operand (64 consecutive bytes of 16
// rows per load; dword alignment is enough), and instruction j multiplies everybody's j-th float -- the contraction
// index is a free permutation as long as both operands use the same one. One step is requested ahead of the one that
// multiplies. Partial tiles meet in LDS once. A: [m, k] rows; BT: B(p, j) = b[j * b_stride + p], else b[p * b_stride + j].
// Measured: 32 rows x 4096 x 4096: 720 -> 24 us (2.8 TB/s of operands); one row 17 us (3.9 TB/s);
// 256 rows 101 us (85 TFLOP/s).
struct __attribute__((packed, aligned(4))) f32x4_a4 { float v[4]; };

template <bool BT, int MTILES, int NT, int NW>
__global__ __launch_bounds__(64 * NW) void sgemm_mfma_skinny_kernel(const float* __restrict__ a, int64_t a_stride, const float* __restrict__ b,
                                                                    int64_t b_stride, float* __restrict__ c, int64_t c_stride, int m, int n, int k) {
    typedef float f32x4 __attribute__((ext_vector_type(4)));
    __shared__ float part[NW][MTILES * NT][256];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int r = lane & 15, q = lane >> 4;
    const int j0 = blockIdx.x * (16 * NT), i0 = blockIdx.y * (16 * MTILES);
    // rows and columns past the end are copies of the last one that nobody stores
    const float* pa[MTILES];
    const float* pb[NT];
#pragma unroll
    for (int t = 0; t < MTILES; ++t) {
        const int row = i0 + 16 * t + r;
        pa[t] = a + (int64_t)(row < m ? row : m - 1) * a_stride + 4 * q;
    }
#pragma unroll
    for (int t = 0; t < NT; ++t) {
        const int col = j0 + 16 * t + r < n ? j0 + 16 * t + r : n - 1;
        pb[t] = BT ? b + (int64_t)col * b_stride + 4 * q : b + (int64_t)(4 * q) * b_stride + col;
    }
    struct Step { float a[MTILES][8], b[NT][8]; };
    auto load = [&](Step& s, int64_t p) {
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            if constexpr (BT) {
                const f32x4_a4 x = *reinterpret_cast<const f32x4_a4*>(pb[t] + p), y = *reinterpret_cast<const f32x4_a4*>(pb[t] + p + 16);
#pragma unroll
                for (int e = 0; e < 4; ++e) { s.b[t][e] = x.v[e]; s.b[t][4 + e] = y.v[e]; }
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e) { s.b[t][e] = pb[t][(p + e) * b_stride]; s.b[t][4 + e] = pb[t][(p + 16 + e) * b_stride]; }
            }
        }
#pragma unroll
        for (int t = 0; t < MTILES; ++t) {
            const f32x4_a4 x = *reinterpret_cast<const f32x4_a4*>(pa[t] + p), y = *reinterpret_cast<const f32x4_a4*>(pa[t] + p + 16);
#pragma unroll
            for (int e = 0; e < 4; ++e) { s.a[t][e] = x.v[e]; s.a[t][4 + e] = y.v[e]; }
        }
    };
    f32x4 acc[MTILES][NT];
#pragma unroll
    for (int t = 0; t < MTILES; ++t)
#pragma unroll
        for (int u = 0; u < NT; ++u) acc[t][u] = f32x4{0.f, 0.f, 0.f, 0.f};
    auto multiply = [&](const Step& s) {
#pragma unroll
        for (int e = 0; e < 8; ++e)
#pragma unroll
            for (int t = 0; t < MTILES; ++t)
#pragma unroll
                for (int u = 0; u < NT; ++u) acc[t][u] = __builtin_amdgcn_mfma_f32_16x16x4f32(s.a[t][e], s.b[u][e], acc[t][u], 0, 0, 0);
    };
    const int full = k >> 5;                       // whole steps; wave w takes w, w + NW, ...
    if (wave < full) {
        Step s0, s1;
        load(s0, (int64_t)wave * 32);
        int st = wave;
        for (; st + NW < full; st += 2 * NW) {
            load(s1, (int64_t)(st + NW) * 32);
            multiply(s0);
            // the request past the last step repeats it: in bounds and never multiplied
            load(s0, (int64_t)(st + 2 * NW < full ? st + 2 * NW : st + NW) * 32);
            multiply(s1);
        }
        if (st < full) multiply(s0);
    }
    if ((k & 31) && wave == full % NW) {           // the last, partial step: elements past K are zeros on both sides
        Step s;
        const int64_t p = (int64_t)full * 32;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const int64_t at = p + (e < 4 ? e : 12 + e);
            const bool in = at + 4 * q < k;
#pragma unroll
            for (int t = 0; t < NT; ++t) s.b[t][e] = in ? (BT ? pb[t][at] : pb[t][at * b_stride]) : 0.f;
#pragma unroll
            for (int t = 0; t < MTILES; ++t) s.a[t][e] = in ? pa[t][at] : 0.f;
        }
        multiply(s);
    }
    // accumulator element e of lane (r, q): row 4 q + e, column r of the tile
#pragma unroll
    for (int t = 0; t < MTILES; ++t)
#pragma unroll
        for (int u = 0; u < NT; ++u)
#pragma unroll
            for (int e = 0; e < 4; ++e) part[wave][t * NT + u][(4 * q + e) * 16 + r] = acc[t][u][e];
    __syncthreads();
    for (int at = threadIdx.x; at < MTILES * NT * 256; at += 64 * NW) {
        float sum = 0.f;
#pragma unroll
        for (int w = 0; w < NW; ++w) sum += (&part[w][0][0])[at];
        const int tile = at >> 8;
        const int row = i0 + 16 * (tile / NT) + ((at >> 4) & 15), cc = j0 + 16 * (tile % NT) + (at & 15);
        if (row < m && cc < n) c[(int64_t)row * c_stride + cc] = sum;
    }
}

// The same product (BT) with the operands brought in through LDS, in loads of W = 4 floats a lane where both operands' rows are 16-byte
// aligned, of one where they are not. What bounds the kernel above
// is the address unit: the 16 lanes that one pass of a load serves sit in 16 rows, 16 bytes of a cache line each, and a CU takes in 16 to
// 18 bytes a cycle (the number of steps in flight, 2 to 4, made no difference). Here a load covers 8 rows (W 1: 2) of 128 consecutive
// bytes and writes LDS directly; the lanes then read their operands from there. Piece c of row r lies at position c ^ (r % 8) of the
// row's eight, which the loading lanes arrange by picking their address, so that the reads of 16 rows spread over the banks. STAGES steps of 32
// elements per wave are in LDS, the same waves take the same steps in the same order as above: the sums have the same bits.
// Measured (us, above / here): 32 x 4096 x 4096 25.9 / 16.6 (a read of its weight 15), 32 x 1000 x 4096 18.0 / 8.3, 32 x 4096 x 1024
// 9.2 / 5.9, 32 x 1001 x 4097 18.1 / 10.6, 256 x 4096 x 4096 101 / 77, 32 x 10 x 8192 26.2 / 10.8.
template <int W>
__device__ __forceinline__ void dense_load_to_lds(uint32_t lds_addr, uint32_t off, const float* base) {
    if constexpr (W == 4) asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds_addr), "v"(off), "s"(base) : "memory");
    else asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, %2" ::"s"(lds_addr), "v"(off), "s"(base) : "memory");
}
template <int MTILES, int NT, int NW, int STAGES, int W>
__global__ __launch_bounds__(64 * NW) void sgemm_mfma_skinny_lds_kernel(const float* __restrict__ a, int64_t a_stride, const float* __restrict__ b,
                                                                        int64_t b_stride, float* __restrict__ c, int64_t c_stride, int m, int n, int k) {
    typedef float f32x4 __attribute__((ext_vector_type(4)));
    constexpr int TILES = MTILES + NT, STAGE_BYTES = TILES * 2048, PER_TILE = 8 / W, LOADS = PER_TILE * TILES;
    static_assert((STAGES - 1) * LOADS <= 63, "loads in flight must fit the wave's counter");
    extern __shared__ __attribute__((aligned(16))) uint8_t dense_smem[];      // [wave][stage][tile][16 rows][8 pieces of 16 bytes]; at the end the partial tiles
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int r = lane & 15, q = lane >> 4;
    const int j0 = blockIdx.x * (16 * NT), i0 = blockIdx.y * (16 * MTILES);
    uint8_t* const mine = dense_smem + wave * (STAGES * STAGE_BYTES);
    const uint32_t mine_addr = (uint32_t)(size_t)(__attribute__((address_space(3))) uint8_t*)mine;
    // byte offset of what this lane loads of tile t, rows 2 W u .. 2 W u + 2 W - 1 (rows past the end are copies of the last one)
    uint32_t off[TILES][PER_TILE];
#pragma unroll
    for (int t = 0; t < TILES; ++t)
#pragma unroll
        for (int u = 0; u < PER_TILE; ++u) {
            const int flt = 64 * W * u + W * lane, row = flt >> 5, piece = ((flt >> 2) & 7) ^ (row & 7);
            const int at = t < MTILES ? min(i0 + 16 * t + row, m - 1) : min(j0 + 16 * (t - MTILES) + row, n - 1);
            off[t][u] = (uint32_t)(at * (t < MTILES ? a_stride : b_stride) * 4) + 16u * piece + 4u * (flt & 3);
        }
    auto issue = [&](int stage, int step) {
        const int64_t p = (int64_t)(wave + NW * step) * 32;
#pragma unroll
        for (int t = 0; t < TILES; ++t)
#pragma unroll
            for (int u = 0; u < PER_TILE; ++u)
                dense_load_to_lds<W>(mine_addr + stage * STAGE_BYTES + t * 2048 + u * (256 * W), off[t][u], (t < MTILES ? a : b) + p);
    };
    f32x4 acc[MTILES][NT];
#pragma unroll
    for (int t = 0; t < MTILES; ++t)
#pragma unroll
        for (int u = 0; u < NT; ++u) acc[t][u] = f32x4{0.f, 0.f, 0.f, 0.f};
    float sa[MTILES][8], sb[NT][8];
    auto multiply = [&]() {
#pragma unroll
        for (int e = 0; e < 8; ++e)
#pragma unroll
            for (int t = 0; t < MTILES; ++t)
#pragma unroll
                for (int u = 0; u < NT; ++u) acc[t][u] = __builtin_amdgcn_mfma_f32_16x16x4f32(sa[t][e], sb[u][e], acc[t][u], 0, 0, 0);
    };
    const int full = k >> 5;                       // whole steps; wave w takes w, w + NW, ...
    const int steps = full > wave ? (full - wave + NW - 1) / NW : 0;
#pragma unroll
    for (int s = 0; s < STAGES; ++s)
        if (s < steps) issue(s, s);
    const uint32_t at0 = (uint32_t)(r * 128 + ((q ^ (r & 7)) << 4)), at1 = (uint32_t)(r * 128 + (((q + 4) ^ (r & 7)) << 4));
    int stage = 0;
    for (int st = 0; st < steps; ++st) {
        if (st + STAGES <= steps) asm volatile("s_waitcnt vmcnt(%0)" ::"n"((STAGES - 1) * LOADS) : "memory");
        else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        const uint8_t* const from = mine + stage * STAGE_BYTES;
#pragma unroll
        for (int t = 0; t < TILES; ++t) {
            const float4 x = *reinterpret_cast<const float4*>(from + t * 2048 + at0), y = *reinterpret_cast<const float4*>(from + t * 2048 + at1);
            float (&s)[8] = t < MTILES ? sa[t < MTILES ? t : 0] : sb[t < MTILES ? 0 : t - MTILES];
            s[0] = x.x; s[1] = x.y; s[2] = x.z; s[3] = x.w; s[4] = y.x; s[5] = y.y; s[6] = y.z; s[7] = y.w;
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");      // the stage has been read: it may be filled again
        if (st + STAGES < steps) issue(stage, st + STAGES);
        multiply();
        stage = stage + 1 == STAGES ? 0 : stage + 1;
    }
    if ((k & 31) && wave == full % NW) {           // the last, partial step: elements past K are zeros on both sides
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const int64_t at = (int64_t)full * 32 + 4 * q + (e < 4 ? e : 12 + e);
#pragma unroll
            for (int t = 0; t < NT; ++t) sb[t][e] = at < k ? b[(int64_t)min(j0 + 16 * t + r, n - 1) * b_stride + at] : 0.f;
#pragma unroll
            for (int t = 0; t < MTILES; ++t) sa[t][e] = at < k ? a[(int64_t)min(i0 + 16 * t + r, m - 1) * a_stride + at] : 0.f;
        }
        multiply();
    }
    __syncthreads();                               // every wave is through with its stages
    float* const part = reinterpret_cast<float*>(dense_smem);      // [wave][tile][256]
    // accumulator element e of lane (r, q): row 4 q + e, column r of the tile
#pragma unroll
    for (int t = 0; t < MTILES; ++t)
#pragma unroll
        for (int u = 0; u < NT; ++u)
#pragma unroll
            for (int e = 0; e < 4; ++e) part[(wave * (MTILES * NT) + t * NT + u) * 256 + (4 * q + e) * 16 + r] = acc[t][u][e];
    __syncthreads();
    for (int at = threadIdx.x; at < MTILES * NT * 256; at += 64 * NW) {
        float sum = 0.f;
#pragma unroll
        for (int w = 0; w < NW; ++w) sum += part[w * (MTILES * NT * 256) + at];
        const int tile = at >> 8;
        const int row = i0 + 16 * (tile / NT) + ((at >> 4) & 15), cc = j0 + 16 * (tile % NT) + (at & 15);
        if (row < m && cc < n) c[(int64_t)row * c_stride + cc] = sum;
    }
}
template <int MTILES, int NT, int NW, int W>
static int launch_skinny_lds_w(const float* a, int64_t a_stride, const float* b, int64_t b_stride, float* c, int64_t c_stride, int m, int n, int k, dim3 grid) {
    // as many stages as 160 KB of LDS and the wave's load counter hold, two to four
    constexpr int STAGE = (MTILES + NT) * 2048 * NW, LOADS = (MTILES + NT) * 8 / W;
    constexpr int STAGES = 4 * STAGE <= 160 * 1024 && 3 * LOADS <= 63 ? 4 : 3 * STAGE <= 160 * 1024 && 2 * LOADS <= 63 ? 3 : 2;
    constexpr size_t smem = (size_t)STAGES * STAGE > (size_t)NW * MTILES * NT * 1024 ? (size_t)STAGES * STAGE : (size_t)NW * MTILES * NT * 1024;
    static_assert(smem <= 160 * 1024, "stages and partial tiles fit the CU's LDS");
    SKH_SET_MAX_DYNAMIC_LDS_ONCE((&sgemm_mfma_skinny_lds_kernel<MTILES, NT, NW, STAGES, W>), smem);
    sgemm_mfma_skinny_lds_kernel<MTILES, NT, NW, STAGES, W><<<grid, dim3(64 * NW), smem, current_stream()>>>(a, a_stride, b, b_stride, c, c_stride, m, n, k);
    return 0;
}
template <int MTILES, int NT, int NW>
static int launch_skinny_lds(const float* a, int64_t a_stride, const float* b, int64_t b_stride, float* c, int64_t c_stride, int m, int n, int k, dim3 grid) {
    const bool rows16 = ((reinterpret_cast<uintptr_t>(a) | reinterpret_cast<uintptr_t>(b)) & 15) == 0 && (a_stride & 3) == 0 && (b_stride & 3) == 0;
    return rows16 ? launch_skinny_lds_w<MTILES, NT, NW, 4>(a, a_stride, b, b_stride, c, c_stride, m, n, k, grid)
                  : launch_skinny_lds_w<MTILES, NT, NW, 1>(a, a_stride, b, b_stride, c, c_stride, m, n, k, grid);
}

template <bool BT, int MTILES, int NT>
static int launch_skinny(const float* a, int64_t a_stride, const float* b, int64_t b_stride, float* c, int64_t c_stride,
                          int m, int n, int k) {
    const dim3 grid((n + 16 * NT - 1) / (16 * NT), (m + 16 * MTILES - 1) / (16 * MTILES));
    // waves per workgroup: enough for eight waves per CU over the whole grid, as long as every wave has a step of K
    const int64_t groups = (int64_t)grid.x * grid.y;
    int nw = 4;
    while (nw < 16 / NT && groups * nw < 8 * (int64_t)num_cus() && 32 * nw < k) nw *= 2;
    // Through LDS from a few steps per wave on: with fewer, what the loads cost to set up is not earned back (us, straight / through LDS,
    // 16-byte rows: 36 x 4109 x 676, 2.6 steps, 12.0 / 13.0; 32 x 4096 x 1024, 4 steps, 9.2 / 5.9; rows at 4 bytes and the eight-tile
    // form, whose loads are four times as many or whose matrix instructions hide more, a few steps later: 239 x 4789 x 692,
    // 5.4 steps, 35.8 / 37.7; 131 x 476 x 774, 3 steps, 6.1 / 7.0). Sixteen waves, grids of less than half the CUs, always: from 1.8
    // steps on 1.07 to 2.0 times faster. Offsets are 32 bits wide.
    if constexpr (BT) {
        const bool rows16 = ((reinterpret_cast<uintptr_t>(a) | reinterpret_cast<uintptr_t>(b)) & 15) == 0 && (a_stride & 3) == 0 && (b_stride & 3) == 0;
        const int least = nw == 16 ? 1 : rows16 && MTILES * NT < 8 ? 4 : 8;
        if (k >= 32 * nw * least && (uint64_t)m * (uint64_t)a_stride < ((uint64_t)1 << 30) && (uint64_t)n * (uint64_t)b_stride < ((uint64_t)1 << 30)) {
            // (two stages of more tiles and waves than these do not fit the LDS)
            if constexpr (MTILES * NT == 1) if (nw == 16) return launch_skinny_lds<1, 1, 16>(a, a_stride, b, b_stride, c, c_stride, m, n, k, grid);
            if constexpr (NT == 1) if (nw == 8) return launch_skinny_lds<MTILES, 1, 8>(a, a_stride, b, b_stride, c, c_stride, m, n, k, grid);
            if (nw == 4 || NT == 2) return launch_skinny_lds<MTILES, NT, 4>(a, a_stride, b, b_stride, c, c_stride, m, n, k, grid);
        }
    }
    if (NT == 1 && nw == 16) sgemm_mfma_skinny_kernel<BT, MTILES, 1, 16><<<grid, dim3(1024), 0, current_stream()>>>(a, a_stride, b, b_stride, c, c_stride, m, n, k);
    else if (nw == 8) sgemm_mfma_skinny_kernel<BT, MTILES, NT, 8><<<grid, dim3(512), 0, current_stream()>>>(a, a_stride, b, b_stride, c, c_stride, m, n, k);
    else sgemm_mfma_skinny_kernel<BT, MTILES, NT, 4><<<grid, dim3(256), 0, current_stream()>>>(a, a_stride, b, b_stride, c, c_stride, m, n, k);
    return 0;
}
// The largest tile whose grid still gives every CU a workgroup (a larger tile reads its operands less often, an idle CU
// costs more than that), and no more rows than the product has.
template <bool BT>
static int launch_skinny_rows(const float* a, int64_t a_stride, const float* b, int64_t b_stride, float* c, int64_t c_stride,
                               int m, int n, int k) {
    auto groups = [&](int mt, int nt) { return (int64_t)((n + 16 * nt - 1) / (16 * nt)) * ((m + 16 * mt - 1) / (16 * mt)); };
    const int cus = num_cus();
    if (m > 32 && groups(4, 2) >= cus) return launch_skinny<BT, 4, 2>(a, a_stride, b, b_stride, c, c_stride, m, n, k);
    if (m > 32 && groups(4, 1) >= cus) return launch_skinny<BT, 4, 1>(a, a_stride, b, b_stride, c, c_stride, m, n, k);
    if (m > 16 && groups(2, 1) >= cus) return launch_skinny<BT, 2, 1>(a, a_stride, b, b_stride, c, c_stride, m, n, k);
    return launch_skinny<BT, 1, 1>(a, a_stride, b, b_stride, c, c_stride, m, n, k);
}

static std::atomic<int> g_dense_mfma{1};
void set_dense_mfma(int v) { g_dense_mfma = v != 0; }

int launch_fp32_matmul(const float* a, int64_t a_stride, const float* b, int64_t b_stride, float* c, int64_t c_stride,
                       int m, int n, int k, bool b_transposed) {
    if (m <= 0 || n <= 0) return 0;
    if (k < 0) k = 0;
    const bool aligned = ((reinterpret_cast<uintptr_t>(a) | reinterpret_cast<uintptr_t>(b)) & 15) == 0 && (a_stride & 3) == 0 &&
                         (b_stride & 3) == 0 && (k & 3) == 0 && (b_transposed || (n & 3) == 0);
    // 64 x 128 tiles that do not fill the CUs leave the product to the kernel that splits K over waves; where they fill
    // them the tile kernel reads each operand less often
    const int64_t tiles64 = (int64_t)((n + MT - 1) / MT) * ((m + 63) / 64);
    // (B read along its rows at an odd alignment and 64 rows or more: the LDS tile kernel, whose loads do not mind). A K of one
    // step of a wave has nothing to split: from a quarter of the CUs (half of them for a whole step) the tile kernel is faster
    // at the same error (232 x 7124 x 20 9.7 -> 6.2 us, 8.3e-8 of float64 either way; 301 x 4660 x 24 7.9 -> 6.0). At larger K
    // it is, too, above three quarters (712 x 2600 x 84 17.4 and 9.7 us, 468 x 3684 x 416 31.8 and 26.4; none from K 1024 on), but one
    // chain of K is up to twice as far from float64 as K in shares (1.7e-7 and 1.1e-7 at 84, 4.1e-7 and 2.1e-7 at 512): that stays.
    const bool shallow = aligned && m >= 64 && n >= 32 && k >= 4 && k <= 32 && tiles64 * (k < 32 ? 4 : 2) >= num_cus();
    if (g_dense_mfma && k >= 1 && tiles64 < num_cus() && !shallow && (b_transposed || aligned || m < 64)) {
        note_kernel("sgemm_mfma_skinny_kernel");
        const int rc = b_transposed ? launch_skinny_rows<true>(a, a_stride, b, b_stride, c, c_stride, m, n, k)
                                    : launch_skinny_rows<false>(a, a_stride, b, b_stride, c, c_stride, m, n, k);
        if (rc != 0) return rc;
        SKH_CHECK(hipGetLastError());
        return 0;
    }
    if (g_dense_mfma && aligned && m >= 64 && n >= 32 && k >= 4) {
        // 128-row tiles where they give every CU at least one; else 64-row tiles
        const int tiles128 = ((n + MT - 1) / MT) * ((m + 127) / 128);
        const int wmr = tiles128 >= num_cus() ? 2 : 1;
        const dim3 grid((n + MT - 1) / MT, (m + 64 * wmr - 1) / (64 * wmr));
        note_kernel("sgemm_mfma_kernel");
        if (b_transposed) {
            if (wmr == 2) sgemm_mfma_kernel<true, 2><<<grid, dim3(256), 0, current_stream()>>>(a, a_stride, b, b_stride, c, c_stride, m, n, k);
            else sgemm_mfma_kernel<true, 1><<<grid, dim3(256), 0, current_stream()>>>(a, a_stride, b, b_stride, c, c_stride, m, n, k);
        } else {
            if (wmr == 2) sgemm_mfma_kernel<false, 2><<<grid, dim3(256), 0, current_stream()>>>(a, a_stride, b, b_stride, c, c_stride, m, n, k);
            else sgemm_mfma_kernel<false, 1><<<grid, dim3(256), 0, current_stream()>>>(a, a_stride, b, b_stride, c, c_stride, m, n, k);
        }
        SKH_CHECK(hipGetLastError());
        return 0;
    }
    note_kernel("sgemm_kernel");
    const dim3 grid((n + DT - 1) / DT, (m + DT - 1) / DT);
    if (b_transposed) sgemm_kernel<1><<<grid, dim3(256), 0, current_stream()>>>(a, a_stride, b, b_stride, c, c_stride, m, n, k);
    else sgemm_kernel<0><<<grid, dim3(256), 0, current_stream()>>>(a, a_stride, b, b_stride, c, c_stride, m, n, k);
    SKH_CHECK(hipGetLastError());
    return 0;
}

// C(m, n) = A(m, k) B(k, n), B bf16 (fp16 != 0: IEEE binary16) bytes with a byte row stride.
int launch_narrow_matmul(const float* a, int64_t a_stride, const uint8_t* b, int64_t b_byte_stride, float* c, int64_t c_stride,
                         int m, int n, int k, int fp16) {
    if (m <= 0 || n <= 0) return 0;
    if (k < 0) k = 0;
    const dim3 grid((n + DT - 1) / DT, (m + DT - 1) / DT);
    const float* bf = reinterpret_cast<const float*>(b);
    if (fp16) sgemm_kernel<3><<<grid, dim3(256), 0, current_stream()>>>(a, a_stride, bf, b_byte_stride, c, c_stride, m, n, k);
    else sgemm_kernel<2><<<grid, dim3(256), 0, current_stream()>>>(a, a_stride, bf, b_byte_stride, c, c_stride, m, n, k);
    SKH_CHECK(hipGetLastError());
    return 0;
}

}  // namespace skh
