// Prefill-shape attention on the matrix cores: out = softmax(q k^T * scale + causal rule) v, fp32 in and out,
// bf16 operands on v_mfma_f32_32x32x16_bf16, fp32 accumulation and fp32 online softmax.
//
// Contract: the reference's skainet_f32_sdpa
//   /root/reference/skainet-backends/skainet-backend-native-cpu/native/src/f32_fused.c:290-396
// restricted to what a prompt pass uses: seq_q <= seq_kv, head_dim 64 or 128; causal or full, with or without a
// sliding window (window, rightContext) and per-sequence key lengths, by the rules of
//   /root/reference/skainet-lang/skainet-lang-core/src/commonMain/kotlin/sk/ainet/lang/tensor/ops/AttentionMask.kt:24-104
// and with or without an additive mask broadcast over [B|1, H|Hkv|1, Sq|1, Skv|1] (f32_fused.c:312-331).
// Every other call stays on the general fp32 kernel (sdpa.hip). Without a mask, a query whose rules leave it at least
// one key gives the same result whether excluded keys score -1e30 (the reference) or take no part (here), and a query
// they leave none weighs every key of the sequence equally, as the reference's row of equal scores does. With a mask
// the reference's arithmetic is kept as it stands: every key of the sequence takes part, an excluded one at -1e30
// plus its mask value (the mask is added to every score), so no key block is skipped.
//
// Two launches (three where keys are split over workgroups, see the kernel):
//   1. kv_to_fragments_kernel: K and V -> bf16 in the order the matrix instructions read them, one run of 2 x 64 x D values
//      per 64-key block (keys padded with zeros). An operand of v_mfma_f32_32x32x16_bf16 is then 1 KB of consecutive bytes
//      per wave: a block is copied into LDS as it lies (loads that write LDS directly, no registers, no rows to pad) and
//      read with one conflict-free 16-byte access per lane and instruction. (The PV product contracts over keys, and an
//      MFMA operand wants 8 consecutive contraction values per lane: V is read along keys, hence the pass in front.)
//   2. sdpa_prefill_kernel: one workgroup per CU, two teams of 4 waves; a wave = one of up to 4 query heads that share a KV
//      head x 32 query positions (fewer heads per KV head: more query blocks). Both teams hold the SAME queries; team t
//      takes key blocks 2 s + t of the group's range in step s and the two states meet in LDS at the end, so the chain of
//      blocks a wave walks is half the keys and every SIMD has two waves at work until the last step. (With the teams on a late
//      and an early query group, the workgroup with the latest group ran 32 blocks with one wave per SIMD.) A workgroup takes its
//      query groups one after the other, a late one and an early one under the causal rule: the same work everywhere, and the
//      next group's queries and first blocks arrive while the one before is put together and stored.
//      Measured, 32 heads over 8, D 128, causal, both launches, before and after: 2048 x 2048 67.1 and 50.2 us, 300 x 300 19.1 and
//      14.9, 1000 x 1000 40.9 and 27.4, 3000 x 3000 152 and 98, a window of 512 keys on 2048 43.0 and 39.1; 64 heads over 8, D 64,
//      3000 on 5000 286 and 226.
//      Per wave and block of 64 keys:
//        S^T[key][query] = K_tile . Q^T           16 MFMAs (Q lives in registers, pre-multiplied by scale * log2 e)
//        online softmax per query: a query is one accumulator COLUMN, so its 32 scores per 32-key tile sit in
//          one lane pair (l, l ^ 32): the row statistics need a single cross-lane step
//        O^T[d][query] += V^T_tile . P            16 MFMAs; P is the S^T accumulator converted in place: the MFMA
//          contraction index is a free permutation, so the keys a lane holds (4h + {0..3}, 8 + 4h + {0..3} of each
//          16) are simply declared to be its 8 k-slots and V^T is laid out in the same order.
//      Blocks wholly above the diagonal are skipped, only blocks that cross it (or the end of the keys) mask.
//      What bounds it: a step of 128 keys takes a CU 1.5 to 1.9 us. Its matrix instructions alone take 0.95 (64 per SIMD of 32
//      cycles), the LDS reads they need the same (256 KB at 128 B/clk) next to the 64 KB written, the softmax 0.4 to 0.5 per wave pair
//      of vector time of which little hides behind matrix instructions: measured by taking one kind out at a time, 0.28 us without
//      the softmax, 0.32 without the loads, 0.18 without the LDS reads. Besides the steps: kv_to_fragments_kernel 6 to 7 us, the first
//      round trip 4, two to five for a group's end (the second pass over that code takes a third of the first: instruction cache).
#include "common.h"

#include <type_traits>

namespace skh {

typedef __bf16 pf_bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 pf_bf16x4 __attribute__((ext_vector_type(4)));
typedef float pf_f32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t pf_u32x4 __attribute__((ext_vector_type(4)));   // a native 16-byte vector: staging registers stay registers

constexpr int PF_KB = 64;          // keys per block
constexpr int PF_QW = 32;          // query positions per wave
constexpr int PF_THREADS = 512;    // two teams of four waves
template <int D> constexpr int pf_block_bytes() { return 2 * PF_KB * D * (int)sizeof(__bf16); }   // K, then V, of one block

// K, V [b][kvh][kv_capacity][D] fp32 -> [b * kvh][block of 64 keys][K | V] bf16, each of the two in operand order:
//   K: [32-key tile][step of 16 d][lane = (key of the tile, half h)][d 8 h .. 8 h + 7 of the step]
//   V: [32-key tile][16 keys][32-row tile of d][lane = (d of the tile, half h)][keys 4 h .. 4 h + 3, 8 + 4 h .. 8 + 4 h + 3 of the 16]
// One workgroup per (32-key tile, kv head, batch), built in LDS and written out as consecutive kilobytes; keys >= seq_kv are
// zeros. Bound by latency: a round trip for the loads, one for the stores (2048 keys x 8 heads are 512 workgroups of 48 KB).
template <int D>
__global__ __launch_bounds__(256) void kv_to_fragments_kernel(const float* __restrict__ k, const float* __restrict__ v,
                                                              __bf16* __restrict__ frag, int kv_heads, int seq_kv, int kv_capacity, int spad) {
    __shared__ __attribute__((aligned(16))) __bf16 kimg[32 * D];
    __shared__ __attribute__((aligned(16))) __bf16 vimg[32 * D];
    const int tile = blockIdx.x, k0 = 32 * tile, tid = threadIdx.x;
    const int64_t head = (int64_t)blockIdx.z * kv_heads + blockIdx.y;
    const float* ksrc = k + head * kv_capacity * D;
    const float* vsrc = v + head * kv_capacity * D;
    constexpr int KT = 32 * D / 8 / 256;                     // K: thread-step = 8 consecutive d of a key
    constexpr int VN = 8 * (D / 4);                          // V: threads with a task of 4 consecutive keys x 4 consecutive d
    float4 kx[KT][2], vx[4];
#pragma unroll
    for (int i = 0; i < KT; ++i) {
        const int t = tid + 256 * i, key = t / (D / 8), c = t % (D / 8);
        const float* p = ksrc + (int64_t)min(k0 + key, seq_kv - 1) * D + 8 * c;
        kx[i][0] = *reinterpret_cast<const float4*>(p);
        kx[i][1] = *reinterpret_cast<const float4*>(p + 4);
    }
    const int d4 = tid % (D / 4), kq = tid / (D / 4);
    if (VN == 256 || tid < VN)
#pragma unroll
        for (int j = 0; j < 4; ++j) vx[j] = *reinterpret_cast<const float4*>(vsrc + (int64_t)min(k0 + 4 * kq + j, seq_kv - 1) * D + 4 * d4);
#pragma unroll
    for (int i = 0; i < KT; ++i) {
        const int t = tid + 256 * i, key = t / (D / 8), c = t % (D / 8);
        const float keep = k0 + key < seq_kv ? 1.0f : 0.0f;
        const float4 a = kx[i][0], b = kx[i][1];
        *reinterpret_cast<pf_bf16x8*>(kimg + (c >> 1) * 512 + ((c & 1) * 32 + key) * 8) =
            pf_bf16x8{(__bf16)(a.x * keep), (__bf16)(a.y * keep), (__bf16)(a.z * keep), (__bf16)(a.w * keep),
                      (__bf16)(b.x * keep), (__bf16)(b.y * keep), (__bf16)(b.z * keep), (__bf16)(b.w * keep)};
    }
    if (VN == 256 || tid < VN) {
        // keys 4 kq .. + 3 of the tile: 16-key group kq / 4, of which quad kq % 4 = 2 (slot half) + h
        const int g = kq >> 2, r = kq & 3, h = r & 1, half = r >> 1;
        float e[4][4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const float keep = k0 + 4 * kq + j < seq_kv ? 1.0f : 0.0f;
            e[j][0] = vx[j].x * keep; e[j][1] = vx[j].y * keep; e[j][2] = vx[j].z * keep; e[j][3] = vx[j].w * keep;
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int d = 4 * d4 + i;
            *reinterpret_cast<pf_bf16x4*>(vimg + (g * (D / 32) + (d >> 5)) * 512 + (h * 32 + (d & 31)) * 8 + 4 * half) =
                pf_bf16x4{(__bf16)e[0][i], (__bf16)e[1][i], (__bf16)e[2][i], (__bf16)e[3][i]};
        }
    }
    __syncthreads();
    // tile `tile` is half (tile % 2) of its block's K part and of its V part
    __bf16* dst = frag + (head * spad + (k0 & ~(PF_KB - 1))) * 2 * D + (tile & 1) * 32 * D;
#pragma unroll
    for (int i = 0; i < 32 * D / 8 / 256; ++i) {
        const int c = 8 * (tid + 256 * i);
        *reinterpret_cast<pf_u32x4*>(dst + c) = *reinterpret_cast<const pf_u32x4*>(kimg + c);
        *reinterpret_cast<pf_u32x4*>(dst + PF_KB * D + c) = *reinterpret_cast<const pf_u32x4*>(vimg + c);
    }
}

struct PrefillParams {
    const float* q;
    const __bf16* frag;        // kv_to_fragments_kernel's output
    float* out;
    int heads, kv_heads, seq_q, seq_kv, spad;
    float scale_log2e;
    int causal, window, right_context;
    const int32_t* lengths;    // per-sequence key counts on the device, or null
    int heads_per_wg;          // 1, 2 or 4 query heads of one KV head per workgroup
    int head_groups;           // workgroups' worth of query heads per KV head
    int ngroups;               // query groups of 128 / heads_per_wg positions
    const float* mask;         // additive mask or null; dims 1 or the full extent (heads: 1, kv_heads or heads)
    int mask_b, mask_h, mask_q, mask_k;
    int places;                // workgroups that share the query groups of a KV head's heads
    int splits;                // workgroups that share a query group's keys (one group per workgroup only)
    float* part;               // [row][splits][D] unnormalised outputs, row = (b, head, query); splits > 1 only
    float* ml;                 // [row][splits][2] running maximum (in units of ln 2) and sum
    int out_rows;              // 0: out is [batch, heads, seq_q, D]; 1: [batch, seq_q, heads, D], token rows of a projection's input
};

// 16 bytes per lane from base + off into LDS at lds_addr + 16 * lane (M0 carries the LDS address). Nothing but
// pf_wait_loads waits for it.
__device__ __forceinline__ void pf_load_to_lds(uint32_t lds_addr, uint32_t off, const uint8_t* base) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds_addr), "v"(off), "s"(base) : "memory");
}
// max(v of this lane, v of the lane 32 away)
__device__ __forceinline__ float pf_max_halves(float v) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
// A barrier for what the waves exchange through LDS. (__syncthreads also waits for every global load and store in flight: the next
// group's queries, the outputs of the one before.)
__device__ __forceinline__ void pf_lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }
// MASKED: the builtin and not inline asm, so that the compiler knows that its own loads, the mask's values, have arrived too.
template <bool MASKED>
__device__ __forceinline__ void pf_wait_loads() {
    if constexpr (MASKED) __builtin_amdgcn_s_waitcnt(0x0F70);           // vmcnt(0)
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
}

// SPLIT: several workgroups share a group's keys, where one group per workgroup leaves CUs idle, and
// sdpa_prefill_merge_kernel puts their outputs together: what bounds such a call is the chain of blocks a workgroup walks.
// MASKED: the softmax is what bounds it (13 vector instructions per score where each score is compared with its range and computed
// twice), so the range is looked at per block, a weight is computed once and the mask's values are there before they are needed
// (us, 32 heads over 8, causal, before and after: 2048 x 2048, D 128, one mask for all heads 159 and 117, a mask row of keys 129 and 98;
// 1024 x 1024, D 64 42.5 and 33.4; the kernel with 4-wave workgroups 160, 128, 54).
template <int D, bool SPLIT, bool MASKED>
__global__ __launch_bounds__(PF_THREADS, 2) void sdpa_prefill_kernel(PrefillParams p) {
    constexpr int NT = D / 16;         // MFMA steps along head_dim for S
    constexpr int ND = D / 32;         // 32-row tiles of O^T
    constexpr int BLK = pf_block_bytes<D>();
    constexpr int SHARE = BLK / 4;     // bytes of a block that each of a team's four waves loads
    // two buffers of two blocks (one per team); the teams' states meet in whichever is not being read, and in pf_ml
    extern __shared__ __attribute__((aligned(16))) uint8_t pf_smem[];
    float2* const pf_ml = reinterpret_cast<float2*>(pf_smem + 4 * BLK);     // [team][wave][lane]
    // [wave][lane]: team 0's first reference for both. Not in pf_ml: over one step there is no barrier between team 1 reading it and
    // team 0 writing its state
    float* const pf_ref = reinterpret_cast<float*>(pf_ml + 2 * 4 * 64);

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave_all = __builtin_amdgcn_readfirstlane(tid >> 6), team = wave_all >> 2, wave = wave_all & 3;
    const int col = lane & 31, h = lane >> 5;
    const int hpw = p.heads_per_wg;               // 1, 2 or 4
    const int q_per_group = 4 * PF_QW >> (hpw >> 1);
    // heads run fastest over the grid: workgroups that read the same keys land on the same die where there are 8 KV heads
    const int place = blockIdx.y;
    const int head = blockIdx.x * hpw + (wave & (hpw - 1));
    const int kvh = p.head_groups == 1 ? blockIdx.x : blockIdx.x / p.head_groups;
    const int qblock = wave >> (hpw >> 1);        // this wave's 32 queries of a group
    const int b = SPLIT ? blockIdx.z / p.splits : blockIdx.z;
    // the workgroup's groups, those with the most keys first: of every 2 p.places groups the one at its place and the one at its
    // place from the end
    auto group_of = [&](int turn) {
        const int rank = turn * p.places + ((turn & 1) ? p.places - 1 - place : place);
        return rank >= p.ngroups ? -1 : p.causal ? p.ngroups - 1 - rank : rank;
    };
    const int shift = p.seq_kv - p.seq_q;                                   // absolute position of query 0
    const int len = p.lengths ? p.lengths[b] : p.seq_kv;
    // attended keys [first, end) of a query position: both bounds grow with the position
    auto first_of = [&](int qi) { return p.window > 0 ? max(0, qi + shift - p.window + 1) : 0; };
    auto end_of = [&](int qi) {
        int e = p.seq_kv;
        if (p.window > 0) e = min(e, qi + shift + p.right_context + 1);
        if (p.causal) e = min(e, qi + shift + 1);
        return max(min(e, len), 0);
    };
    constexpr bool masked = MASKED;
    const int64_t kvhead = (int64_t)b * p.kv_heads + kvh;
    const uint8_t* const frag = reinterpret_cast<const uint8_t*>(p.frag) + kvhead * p.spad * (4 * D) + wave * SHARE;
    const uint32_t lds0 = (uint32_t)(size_t)(__attribute__((address_space(3))) uint8_t*)pf_smem + team * BLK + wave * SHARE;
    const uint32_t lane_off = 16u * lane;
    // this wave's share of block blk into its team's place in buffer buf
    auto load_block = [&](int blk, int buf) {
        const uint8_t* src = frag + (int64_t)__builtin_amdgcn_readfirstlane(blk) * BLK;
        const uint32_t dst = lds0 + __builtin_amdgcn_readfirstlane(buf) * (2 * BLK);
#pragma unroll
        for (int u = 0; u < SHARE / 1024; ++u) pf_load_to_lds(dst + u * 1024, lane_off, src + u * 1024);
    };

    const int split = SPLIT ? blockIdx.z % p.splits : 0;
    // does a group hold a query that the rules leave no key? Such a query weighs every key of the sequence equally (with a mask
    // the -1e30 scores do that by themselves), so its group walks all of them. The same answer in every wave.
    auto walks_all = [&](int group) {
        if (masked) return true;
        const int qa = min(group * q_per_group + min(lane, q_per_group - 1), p.seq_q - 1);
        const int qb = min(group * q_per_group + min(lane + 64, q_per_group - 1), p.seq_q - 1);
        return __ballot(first_of(qa) >= end_of(qa) || first_of(qb) >= end_of(qb)) != 0;
    };
    // the key blocks [blk0, blk1) a group walks (under SPLIT this workgroup's share of them, which may be none)
    auto blocks_of = [&](int group, int& blk0, int& blk1) {
        const bool all_keys = walks_all(group);
        blk0 = all_keys ? 0 : first_of(group * q_per_group) / PF_KB;
        blk1 = ((all_keys ? p.seq_kv : end_of(min(p.seq_q, (group + 1) * q_per_group) - 1)) + PF_KB - 1) / PF_KB;
        if (SPLIT) {
            const int share = (blk1 - blk0 + p.splits - 1) / p.splits;
            blk0 += split * share;
            blk1 = min(blk1, blk0 + share);
        }
        blk1 = max(blk1, blk0);
    };
    // Half of a wave's 32 x D queries (the other half is its partner's in the other team): 16 rows x 64 bytes per load
    float4 qraw[NT];
    auto load_q = [&](int group) {
        int at = lane;
        asm volatile("" : "+v"(at));              // see the end of a group
        const int row = min(group * q_per_group + qblock * PF_QW + 16 * team + (at & 15), p.seq_q - 1);
        const float* qp = p.q + (((int64_t)b * p.heads + head) * p.seq_q + row) * D + 4 * (at >> 4);
#pragma unroll
        for (int t = 0; t < NT; ++t) qraw[t] = *reinterpret_cast<const float4*>(qp + 16 * t);
    };
    int blk0, blk1, par = 0;                                                // step st of a group reads buffer (par + st) % 2
    int group = group_of(0);
    blocks_of(group, blk0, blk1);
    if (blk0 + team < blk1) load_block(blk0 + team, par);
    load_q(group);

    for (int turn = 1; group >= 0; ++turn) {
        const int q0 = group * q_per_group + qblock * PF_QW;          // first query position of this wave
        const int my_q = q0 + col, my_qc = min(my_q, p.seq_q - 1);
        const int real_first = first_of(my_qc), real_last = end_of(my_qc) - 1;  // the rules' own range (may be empty)
        const bool my_uniform = !masked && first_of(my_qc) >= end_of(my_qc);
        const int my_first_key = my_uniform ? 0 : real_first;
        const int my_last_key = my_uniform ? p.seq_kv - 1 : real_last;
        const bool wave_uniform = __ballot(my_uniform) != 0;
        const int steps = (blk1 - blk0 + 1) >> 1;
        // this wave's 32 positions: the keys any of them attends, and the keys all of them attend
        const int q_wave_last = min(q0 + PF_QW - 1, p.seq_q - 1), q_wave_first = min(q0, p.seq_q - 1);
        const int wave_first_key = (wave_uniform || masked) ? 0 : first_of(q_wave_first);
        const int wave_last_key = (wave_uniform || masked) ? p.seq_kv - 1 : end_of(q_wave_last) - 1;
        const int wave_common_first = first_of(q_wave_last), wave_common_last = end_of(q_wave_first) - 1;

        // Q fragment: lane (query col, half h) holds q[16 t + 8 h .. + 7] for every t, times scale * log2(e). The two halves meet in the
        // buffer that the first step does not read (loading the fragment as it is held would touch 32 rows with every load,
        // in both teams: 512 pieces of 32 bytes per wave where this takes 128 of 64).
        pf_bf16x8 qf[NT];
        {
            __bf16* const qs = reinterpret_cast<__bf16*>(pf_smem + (par ^ 1) * (2 * BLK)) + wave * (32 * D);
            pf_lds_barrier();                      // the group before has left that buffer
            const float f = p.scale_log2e;
#pragma unroll
            for (int t = 0; t < NT; ++t)
                *reinterpret_cast<pf_bf16x4*>(qs + t * 512 + ((lane >> 5) * 32 + 16 * team + (lane & 15)) * 8 + 4 * ((lane >> 4) & 1)) =
                    pf_bf16x4{(__bf16)(qraw[t].x * f), (__bf16)(qraw[t].y * f), (__bf16)(qraw[t].z * f), (__bf16)(qraw[t].w * f)};
            pf_lds_barrier();
#pragma unroll
            for (int t = 0; t < NT; ++t) qf[t] = *reinterpret_cast<const pf_bf16x8*>(qs + t * 512 + lane * 8);
        }
        // this lane's row of the mask (one query position; the key index is added per score), in units of ln 2 later
        const float* mrow = nullptr;
        if (masked) {
            const int bi = p.mask_b == 1 ? 0 : b;
            const int hi = p.mask_h == 1 ? 0 : (p.mask_h == p.heads ? head : kvh);
            mrow = p.mask + (((int64_t)bi * p.mask_h + hi) * p.mask_q + (p.mask_q == 1 ? 0 : my_qc)) * p.mask_k;
        }
        // The mask values of a block's keys for this lane's query, four adjacent keys per 16-byte load. They are requested while the block
        // before is multiplied, behind the last use of that block's: asked for where they are added, each half of a block waited for
        // a round trip to memory (half a step's time).
        float4 mval[2][4];
        auto load_mask = [&](int blk) {
#pragma unroll
            for (int c = 0; c < 8; ++c) {
                const int key4 = PF_KB * blk + 8 * c + 4 * h;
                float4 mv;
                if (p.mask_k == 1) { const float m1 = mrow[0]; mv = make_float4(m1, m1, m1, m1); }
                else mv = *reinterpret_cast<const float4*>(mrow + min(key4, p.seq_kv - 4));     // seq_kv is a multiple of 4 here
                mval[c >> 2][c & 3] = mv;
            }
        };
        if (masked && blk0 + team < blk1) load_mask(blk0 + team);
        // O^T; accumulator i is d tile (i + team ND / 2) % ND, so the first half of them is what this team finishes
        pf_f32x16 oacc[ND];
#pragma unroll
        for (int i = 0; i < ND; ++i)
#pragma unroll
            for (int e = 0; e < 16; ++e) oacc[i][e] = 0.f;
        float m_run = -INFINITY, l_run = 0.f;     // per query (column); l_run is this lane's half of the keys
        // Scores come out of the matrix instructions with the reference of their exponentials taken off: it is what the accumulators
        // start from. Large references (where a score near zero would lose digits to it) and masked calls take it off in settle().
        pf_f32x16 minus_ref;
        bool explicit_ref = false;                // wave-uniform
        auto set_reference = [&]() {
            const float m = m_run == -INFINITY ? 0.f : m_run;
            explicit_ref = masked || __ballot(!(fabsf(m) <= 1024.0f)) != 0;
#pragma unroll
            for (int e = 0; e < 16; ++e) minus_ref[e] = explicit_ref ? 0.f : -m;
        };
        set_reference();

        // The reference starts as the maximum over the group's first block, for both teams (weights rounded against two references would
        // differ by bf16's rounding from those of one): step -1 is team 0's scores of that block and no more.
        if (team == 0) pf_ref[wave * 64 + lane] = -INFINITY;
        for (int st = steps ? -1 : 0; st < steps; ++st) {
            const int blk = st < 0 ? blk0 : blk0 + 2 * st + team, k0 = blk * PF_KB;
            if (st != 0) pf_wait_loads<MASKED>();         // this wave's share of the step's block (of step 0 with step -1) ...
            pf_lds_barrier();                     // ... and everybody's; the other buffer has been read by all
            const int ahead = st < 0 ? 1 : st + 1;
            if (st != 0 && blk0 + 2 * ahead + team < blk1) load_block(blk0 + 2 * ahead + team, (par + ahead) & 1);
            if (st == 0) { m_run = pf_ref[wave * 64 + lane]; set_reference(); }
            if ((st < 0 && team) || blk >= blk1 || k0 > wave_last_key || k0 + PF_KB <= wave_first_key) continue;      // wave-uniform: no keys in the block
            // The block in two halves of 32 keys, a and b: S of a; S of b with the softmax of a between its matrix instructions;
            // O += V^T . P of a with the softmax of b in between; O += V^T . P of b. The order is pinned (sched_barrier) and
            // AHEAD operand reads are in flight throughout: left alone, the compiler waits out the latency of every read and puts the
            // vector work behind the matrix work.
            const uint8_t* const tile = pf_smem + (2 * ((par + max(st, 0)) & 1) + team) * BLK + lane_off;
            constexpr int AHEAD = 3, OPS = 2 * NT + 4 * ND;       // K's operands, then V's, as they lie
            pf_bf16x8 fr[AHEAD];
            // (V's d tiles in this team's order: team 1 starts with the second half of them)
            const uint8_t* const first_v = tile + team * (ND / 2) * 1024;
            const uint8_t* const second_v = tile - team * (ND / 2) * 1024;
            auto read = [&](int n) {
                const uint8_t* from = n < 2 * NT ? tile : n % ND < ND / 2 ? first_v : second_v;
                if (n < OPS) fr[n % AHEAD] = *reinterpret_cast<const pf_bf16x8*>(from + n * 1024);
            };
            pf_f32x16 s[2];                       // s[j]: keys k0 + 32 j .. + 31 (rows) x this wave's 32 queries (columns)
#pragma unroll
            for (int n = 0; n < AHEAD; ++n) read(n);
#pragma unroll
            for (int e = 0; e < 16; ++e) s[0][e] = s[1][e] = minus_ref[e];
            auto qk = [&](int n) {
                __builtin_amdgcn_sched_barrier(0);
                s[n / NT] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fr[n % AHEAD], qf[n % NT], s[n / NT], 0, 0, 0);
                read(n + AHEAD);
                __builtin_amdgcn_sched_barrier(0);
            };
            auto hide = [&](int j) {              // the mask and the range rules on the scores of half j
                if (masked) {
                    // the reference's arithmetic: an excluded key scores -1e30, the mask is added to every score; keys past
                    // the sequence (padding of the last block) take no part
                    constexpr float LOG2E = 1.4426950408889634f;
                    if (k0 < wave_common_first || k0 + PF_KB - 1 > wave_common_last) {       // wave-uniform, as is the next: some query excludes some key
                        if (k0 > end_of(q_wave_last) - 1 || k0 + PF_KB <= first_of(q_wave_first)) {      // every query excludes every key
#pragma unroll
                            for (int e = 0; e < 16; ++e) s[j][e] = -1.0e30f * LOG2E;
                        } else {
                            const int lo = real_first - k0 - 4 * h, hi = real_last - k0 - 4 * h;
#pragma unroll
                            for (int e = 0; e < 16; ++e) {
                                const int key = 32 * j + 8 * (e >> 2) + (e & 3);              // relative to k0 + 4 h
                                if (key > hi || key < lo) s[j][e] = -1.0e30f * LOG2E;
                            }
                        }
                    }
#pragma unroll
                    for (int e = 0; e < 16; ++e) {
                        const float4 mv = mval[j][e >> 2];
                        s[j][e] = fmaf((e & 3) == 0 ? mv.x : (e & 3) == 1 ? mv.y : (e & 3) == 2 ? mv.z : mv.w, LOG2E, s[j][e]);
                    }
                    if (k0 + PF_KB > p.seq_kv) {
                        const int end = p.seq_kv - k0 - 4 * h;
#pragma unroll
                        for (int e = 0; e < 16; ++e)
                            if (32 * j + 8 * (e >> 2) + (e & 3) >= end) s[j][e] = -INFINITY;
                    }
                } else
                // keys outside this query's range score -inf (they take no part); a query without a range scores every key 0
                if (wave_uniform || k0 < wave_common_first || k0 + PF_KB - 1 > wave_common_last) {   // wave-uniform: the block crosses a boundary
                    const int lo = my_first_key - k0 - 4 * h, hi = my_last_key - k0 - 4 * h;
#pragma unroll
                    for (int e = 0; e < 16; ++e) {
                        const int key = 32 * j + 8 * (e >> 2) + (e & 3);                  // relative to k0 + 4 h
                        if (my_uniform) s[j][e] = minus_ref[0];
                        if (key > hi || key < lo) s[j][e] = -INFINITY;
                    }
                }
            };
            // Four weights: scores 4 c .. 4 c + 3 of half j
            float psum[2];
            auto exps = [&](int j, int c, pf_bf16x8 (&to)[2]) {
                const float p0 = __builtin_amdgcn_exp2f(s[j][4 * c]), p1 = __builtin_amdgcn_exp2f(s[j][4 * c + 1]);
                const float p2 = __builtin_amdgcn_exp2f(s[j][4 * c + 2]), p3 = __builtin_amdgcn_exp2f(s[j][4 * c + 3]);
                psum[0] += p0 + p1; psum[1] += p2 + p3;
                const int at = 4 * (c & 1);
                to[c >> 1][at] = (__bf16)p0; to[c >> 1][at + 1] = (__bf16)p1; to[c >> 1][at + 2] = (__bf16)p2; to[c >> 1][at + 3] = (__bf16)p3;
            };
            // The reference point of a query's exponentials is lazy: it stays as long as the weights of a half sum to at most 2^8 per
            // lane (far inside bf16 and fp32 range; the final division by the sum takes the common factor out), so neither the
            // maximum of a block nor the rescaling of the output accumulators is computed but where some query of the wave needs a
            // new reference -- for most waves the first half of the first block only. A sum that is no number comes here too. Masked
            // calls, whose scores come with no reference off, compute their weights here and nowhere else.
            auto settle = [&](int j, pf_bf16x8 (&to)[2]) {
                if (!explicit_ref && __ballot(!(psum[0] + psum[1] <= 256.0f) || m_run == -INFINITY) == 0) return;      // wave-uniform
                const float off = -minus_ref[0];                              // what the scores are already less
                float mx = s[j][0];
#pragma unroll
                for (int e = 1; e < 16; ++e) mx = fmaxf(mx, s[j][e]);
                mx = pf_max_halves(mx) + off;
                const bool move = mx > m_run + (explicit_ref ? 8.0f : 0.0f);  // no reference yet (-inf): with any finite score
                const float m_new = move ? mx : m_run, use = m_new == -INFINITY ? 0.f : m_new;      // keys wholly past a query's range leave it at -inf
                const float alpha = move ? __builtin_amdgcn_exp2f(m_run - use) : 1.0f;              // m_run = -inf -> 0
                if (!masked || __ballot(move) != 0) {                         // wave-uniform
                    m_run = m_new;
                    l_run *= alpha;
#pragma unroll
                    for (int i = 0; i < ND; ++i)
#pragma unroll
                        for (int e = 0; e < 16; ++e) oacc[i][e] *= alpha;
                    set_reference();
                }
#pragma unroll
                for (int e = 0; e < 16; ++e) { s[j][e] -= use - off; if (!masked && j == 0) s[1][e] += off + minus_ref[0]; }
                psum[0] = psum[1] = 0.f;
#pragma unroll
                for (int c = 0; c < 4; ++c) exps(j, c, to);
            };
            pf_bf16x8 pf[2], pg[2];               // weights of the two halves: keys 16 g .. of a half, this lane's 8 slots
            // O^T += V^T . P : A = V^T rows d, this lane's k-slots are keys 16 g + 4 h + {0..3} and 16 g + 8 + 4 h + {0..3}
            auto pv = [&](int n, pf_bf16x8 (&from)[2]) {
                __builtin_amdgcn_sched_barrier(0);
                oacc[n % ND] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fr[(2 * NT + n) % AHEAD], from[(n / ND) & 1], oacc[n % ND], 0, 0, 0);
                read(2 * NT + n + AHEAD);
                __builtin_amdgcn_sched_barrier(0);
            };
#pragma unroll
            for (int n = 0; n < NT + NT / 4; ++n) qk(n);
            hide(0);
            psum[0] = psum[1] = 0.f;
#pragma unroll
            for (int n = NT + NT / 4; n < 2 * NT; ++n) {
                qk(n);
                if (n >= 2 * NT - 4 && NT >= 8 && !masked) exps(0, n - (2 * NT - 4), pf);
            }
            if (NT < 8 && !masked)
#pragma unroll
                for (int c = 0; c < 4; ++c) exps(0, c, pf);
            hide(1);
            if (st < 0) {
                float mx = s[0][0];
#pragma unroll
                for (int e = 1; e < 32; ++e) mx = fmaxf(mx, s[e >> 4][e & 15]);
                pf_ref[wave * 64 + lane] = pf_max_halves(mx);
                continue;
            }
            if (masked && blk + 2 < blk1) load_mask(blk + 2);
            settle(0, pf);
            l_run += psum[0] + psum[1];
            psum[0] = psum[1] = 0.f;
#pragma unroll
            for (int n = 0; n < 2 * ND; ++n) {
                pv(n, pf);
                if (n >= 2 * ND - 4 && !masked) exps(1, n - (2 * ND - 4), pg);
            }
            settle(1, pg);
            l_run += psum[0] + psum[1];
#pragma unroll
            for (int n = 2 * ND; n < 4 * ND; ++n) pv(n, pg);
        }

        // The two teams' states of a query put together. Team t finishes d tiles t * ND / 2 .. and hands the others over, through the
        // buffer that nobody reads any more (the last step read the other one). A team without keys has a maximum of -inf and
        // takes no part. The next group's queries and first blocks are on their way meanwhile.
        // (its addresses are formed here, not ahead of the loop: held through it they would not fit the registers, and the reload waits
        // for everything in flight)
        int at = lane;
        asm volatile("" : "+v"(at));
        const int next_group = group_of(turn);                             // uniform; negative: none
        if (next_group >= 0) load_q(next_group);
        const float l_tot = l_run + __shfl_xor(l_run, 32, 64);
        constexpr int HALF = ND / 2, CH = 8 * HALF;                         // 16-byte chunks of an output row's half
        float4* const xch = reinterpret_cast<float4*>(pf_smem + ((par + steps) & 1) * (2 * BLK));          // [team][wave][4 HALF][lane]
        float4* const mine_at = xch + (team * 4 + wave) * (4 * HALF * 64);
        const float4* const theirs_at = xch + ((team ^ 1) * 4 + wave) * (4 * HALF * 64);
        pf_ml[(team * 4 + wave) * 64 + at] = make_float2(m_run, l_tot);
#pragma unroll
        for (int i = 0; i < HALF; ++i)
#pragma unroll
            for (int e4 = 0; e4 < 4; ++e4) {
                const pf_f32x16& o = oacc[HALF + i];
                mine_at[(4 * i + e4) * 64 + at] = make_float4(o[4 * e4], o[4 * e4 + 1], o[4 * e4 + 2], o[4 * e4 + 3]);
            }
        pf_lds_barrier();
        par = (par + steps + 1) & 1;
        if (next_group >= 0) {
            blocks_of(next_group, blk0, blk1);
            if (blk0 + team < blk1) load_block(blk0 + team, par);
        }
        const float2 other = pf_ml[((team ^ 1) * 4 + wave) * 64 + at];
        const float m_all = fmaxf(m_run, other.x), m_ref = m_all == -INFINITY ? 0.f : m_all;
        float mine = __builtin_amdgcn_exp2f(m_run - m_ref), theirs = __builtin_amdgcn_exp2f(other.x - m_ref);
        const float l_all = fmaf(mine, l_tot, theirs * other.y);
        const int64_t row0 = ((int64_t)b * p.heads + head) * p.seq_q;
        if (SPLIT) {
            if (team == 0 && at < 32 && q0 + (at & 31) < p.seq_q)
                *reinterpret_cast<float2*>(p.ml + 2 * ((row0 + q0 + (at & 31)) * p.splits + split)) = make_float2(m_all, l_all);
        } else {
            const float inv = l_all > 0.f ? 1.0f / l_all : 0.f;
            mine *= inv; theirs *= inv;
        }
#pragma unroll
        for (int i = 0; i < HALF; ++i)
#pragma unroll
            for (int e4 = 0; e4 < 4; ++e4) {
                pf_f32x16& o = oacc[i];
                const float4 t = theirs_at[(4 * i + e4) * 64 + at];
                o[4 * e4] = fmaf(mine, o[4 * e4], theirs * t.x); o[4 * e4 + 1] = fmaf(mine, o[4 * e4 + 1], theirs * t.y);
                o[4 * e4 + 2] = fmaf(mine, o[4 * e4 + 2], theirs * t.z); o[4 * e4 + 3] = fmaf(mine, o[4 * e4 + 3], theirs * t.w);
            }
        pf_lds_barrier();                         // what this wave handed over has been read: its place turns the outputs into rows
#pragma unroll
        for (int c = 0; c < 4 * HALF; ++c) {
            const pf_f32x16& o = oacc[c / 4];
            mine_at[(at & 31) * CH + ((2 * c + (at >> 5)) ^ (at & (CH - 1)))] = make_float4(o[4 * (c % 4)], o[4 * (c % 4) + 1], o[4 * (c % 4) + 2], o[4 * (c % 4) + 3]);
        }
        float* const out0 = SPLIT ? p.part + (row0 * p.splits + split) * D : p.out + (p.out_rows ? (int64_t)b * p.seq_q * p.heads + head : row0) * D;
        const int64_t pitch = (SPLIT ? p.splits : p.out_rows ? p.heads : 1) * D;
        const int r0 = at / CH, c0 = at & (CH - 1);
        float* op = out0 + (q0 + r0) * pitch + 32 * team * HALF + 4 * c0;
#pragma unroll
        for (int i = 0; i < 32 * CH / 64; ++i, op += (64 / CH) * pitch) {
            const int r = (64 / CH) * i + r0;
            const float4 v = mine_at[r * CH + (c0 ^ (r & (CH - 1)))];
            if (q0 + r < p.seq_q) *reinterpret_cast<float4*>(op) = v;
        }
        group = next_group;
    }
}

// The splits of a row put together: thread = (row, four elements). A split without keys has a maximum of -inf and takes no part.
template <int D>
__global__ __launch_bounds__(256) void sdpa_prefill_merge_kernel(PrefillParams p, int64_t rows) {
    const int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x, row = t / (D / 4);
    const int d = 4 * (int)(t % (D / 4));
    if (row >= rows) return;
    const float2* ml = reinterpret_cast<const float2*>(p.ml) + row * p.splits;
    float m = -INFINITY;
    for (int i = 0; i < p.splits; ++i) m = fmaxf(m, ml[i].x);
    const float ref = m == -INFINITY ? 0.f : m;
    float4 o = make_float4(0.f, 0.f, 0.f, 0.f);
    float l = 0.f;
    for (int i = 0; i < p.splits; ++i) {
        const float2 s = ml[i];
        const float c = __builtin_amdgcn_exp2f(s.x - ref);                  // -inf: 0
        const float4 v = *reinterpret_cast<const float4*>(p.part + (row * p.splits + i) * D + d);
        o.x = fmaf(c, v.x, o.x); o.y = fmaf(c, v.y, o.y); o.z = fmaf(c, v.z, o.z); o.w = fmaf(c, v.w, o.w);
        l = fmaf(c, s.y, l);
    }
    const float inv = l > 0.f ? 1.0f / l : 0.f;
    int64_t to = row;
    if (p.out_rows) {
        const int64_t qi = row % p.seq_q, bh = row / p.seq_q;
        to = (bh / p.heads * p.seq_q + qi) * p.heads + bh % p.heads;
    }
    *reinterpret_cast<float4*>(p.out + to * D + d) = make_float4(o.x * inv, o.y * inv, o.z * inv, o.w * inv);
}

void* kernel_workspace(size_t bytes);   // shim.hip: per-thread scratch, grown on demand

static std::atomic<int> g_prefill_mfma{1};
void set_sdpa_prefill_mfma(int v) { g_prefill_mfma = v; }
static std::atomic<int> g_prefill_splits{0};  // 0: chosen from the shape
void set_sdpa_prefill_splits(int v) { if (v >= 0 && v <= 32) g_prefill_splits = v; }
static std::atomic<int> g_prefill_teams{0};   // 0: chosen from the grid, 1: one query group per workgroup, 2: two, one after the other
void set_sdpa_prefill_teams(int v) { if (v >= 0 && v <= 2) g_prefill_teams = v; }

// How many workgroups share a query group's keys, where one group per workgroup leaves CUs idle: a chunk of a long prompt, few
// heads. Estimates in us, read off 40 shapes of 1 to 64 heads, 16 to 2500 queries, 20 to 2500 keys at 1 to 32 splits (within 8 % of
// most of them): launches, prologue and output 9.5; a step of 128 keys 1.65 (D 128) or 1.0 (D 64); splitting costs the merging launch,
// 3.3, and the partial outputs, written and read at 3 bytes per ps. Measured with one and with the chosen number: 8 heads over 4, 143
// queries on 1214 keys 26.2 -> 20.4; 4 heads over 2, 73 on 1865, D 64, 23.0 -> 15.5; 8 heads over 4, 1519 on 1519 stays (30.6, 31.1 with two).
// With a mask every key is walked, whatever the window, and a step takes 2.8 or 2.2 (15 600 masked prompts of these sizes, each with one to
// 32 splits: the choice is within 1 % of the best on average). One head, D 128, 1638 on 2256 under a mask and a window of 446: 62.6 with one, 26.1
// with the chosen number; 8 heads over 1, D 64, 357 on 752, 26.2 -> 18.
static int prefill_splits(int64_t wgs, int64_t rows, int head_dim, int seq_kv, int q_per_group, int window, int right_context, int batch, bool masked) {
    const int64_t keys = window > 0 && !masked ? min((int64_t)seq_kv, (int64_t)window + right_context + q_per_group) : seq_kv;
    const int blocks = (int)((keys + PF_KB - 1) / PF_KB);
    const int room = (int)min((int64_t)32, (int64_t)min(blocks, 65535 / batch));
    if (g_prefill_splits.load() > 0) return max(1, min((int)min((int64_t)room, 2 * (int64_t)num_cus() / wgs), g_prefill_splits.load()));
    const double step_us = head_dim == 64 ? (masked ? 2.2 : 1.0) : masked ? 2.8 : 1.65;
    int splits = 1;
    double best = 0.97 * (9.5 + step_us * ((blocks + 1) / 2));
    for (int n = 2; n <= room && n * wgs <= num_cus(); ++n) {
        const double t = 9.5 + step_us * (((blocks + n - 1) / n + 1) / 2) + 3.3 + 8.0 * rows * n * (head_dim + 2) / 3e6;
        if (t < best) { best = t; splits = n; }
    }
    return splits;
}

// Query groups, the workgroups that take them and the splits of their keys.
struct PrefillPlan { int hpw, q_per_group, ngroups, places, splits; int64_t head_wgs; };
static PrefillPlan prefill_plan(int batch, int heads, int kv_heads, int seq_q, int seq_kv, int head_dim, int window, int right_context, bool masked) {
    const int per_kv = heads / kv_heads;
    PrefillPlan p{};
    p.hpw = per_kv % 4 == 0 ? 4 : (per_kv % 2 == 0 ? 2 : 1);
    p.q_per_group = (4 / p.hpw) * PF_QW;
    p.ngroups = (seq_q + p.q_per_group - 1) / p.q_per_group;
    p.head_wgs = (int64_t)kv_heads * (per_kv / p.hpw) * batch;
    // One workgroup per CU that takes its share of the query groups one after the other, where such workgroups fill the chip: the next
    // group's first loads then run under the end of the one before
    const int share = (int)(num_cus() / p.head_wgs);
    const int teams = g_prefill_teams.load();
    p.places = min(65535, teams == 1 ? p.ngroups : teams == 2 ? (p.ngroups + 1) / 2
                 : share >= 1 && share < p.ngroups && share * p.head_wgs * 10 >= 9 * (int64_t)num_cus() ? share : p.ngroups);
    p.splits = p.places < p.ngroups ? 1 : prefill_splits(p.ngroups * p.head_wgs, (int64_t)batch * heads * seq_q, head_dim, seq_kv, p.q_per_group, window, right_context, batch, masked);
    return p;
}

// What a prompt without a mask takes on this kernel, in us back to back from the host: rounds of workgroups, a workgroup's steps of 128 keys, all
// steps over the CUs, the merge and the partial outputs, the pass that lays K and V out, the outputs. Fitted to 42 000 random prompts (16 to 3000
// queries, up to 32 768 earlier keys, a third under windows, 1 to 64 heads, D 64 and 128): 8 % rms.
double sdpa_prefill_estimate(int batch, int heads, int kv_heads, int seq_q, int seq_kv, int head_dim, int causal, int window, int right_context) {
    const PrefillPlan p = prefill_plan(batch, heads, kv_heads, seq_q, seq_kv, head_dim, window, right_context, false);
    const double rows = (double)batch * heads * seq_q, wgs = (double)p.ngroups * p.head_wgs, cus = num_cus();
    double keys = causal ? seq_kv - 0.5 * (seq_q - 1) : seq_kv, most = seq_kv;           // of a query group, on average and at most
    if (window > 0) {
        keys = fmin(keys, (double)window + right_context + 0.5 * p.q_per_group);
        most = fmin(most, (double)window + right_context + p.q_per_group);
    }
    const double steps = ceil(ceil(most / PF_KB) / p.splits / 2), total = wgs * keys / 128 / cus, rounds = ceil(wgs * p.splits / cus);
    const double kb = 1e-3 * batch * kv_heads * seq_kv, out_mb = 8e-6 * rows * head_dim, part_mb = p.splits > 1 ? 8e-6 / 3 * rows * p.splits * (head_dim + 2) : 0.0;
    if (head_dim == 64) return 8.66 * rounds + 0.841 * steps + 3.50 * total + (p.splits > 1 ? 5.41 : 0.0) + 0.221 * part_mb + 0.105 * kb + 0.063 * out_mb;
    return 3.98 + 5.65 * rounds + 1.42 * steps + 3.58 * total + (p.splits > 1 ? 5.02 : 0.0) + 0.589 * part_mb + 0.219 * kb + 0.192 * out_mb;
}

template <int D, bool SPLIT, bool MASKED>
static int launch_prefill_kernel(dim3 grid, size_t smem, hipStream_t s, const PrefillParams& p) {
    SKH_SET_MAX_DYNAMIC_LDS_ONCE((&sdpa_prefill_kernel<D, SPLIT, MASKED>), smem);
    sdpa_prefill_kernel<D, SPLIT, MASKED><<<grid, dim3(PF_THREADS), smem, s>>>(p);
    return 0;
}

template <int D>
static int launch_prefill_d(const float* q, const float* k, const float* v, float* out, int batch, int heads, int kv_heads,
                            int seq_q, int seq_kv, int kv_capacity, float scale, int causal, int window, int right_context,
                            const int32_t* lengths, const float* mask, int mask_b, int mask_h, int mask_q, int mask_k, int out_rows) {
    const int spad = (seq_kv + PF_KB - 1) / PF_KB * PF_KB;
    const size_t elems = (size_t)batch * kv_heads * spad * D;
    hipStream_t s = current_stream();
    const int per_kv = heads / kv_heads;
    const PrefillPlan plan = prefill_plan(batch, heads, kv_heads, seq_q, seq_kv, D, window, right_context, mask != nullptr);
    const int hpw = plan.hpw, splits = plan.splits;
    const size_t rows = (size_t)batch * heads * seq_q;
    uint8_t* ws = static_cast<uint8_t*>(kernel_workspace(2 * elems * sizeof(__bf16) + (splits > 1 ? rows * splits * (D + 2) * sizeof(float) : 0)));
    if (!ws) return -1;
    __bf16* frag = reinterpret_cast<__bf16*>(ws);
    float* part = reinterpret_cast<float*>(frag + 2 * elems);
    kv_to_fragments_kernel<D><<<dim3(spad / 32, kv_heads, batch), dim3(256), 0, s>>>(k, v, frag, kv_heads, seq_kv, kv_capacity, spad);
    SKH_CHECK(hipGetLastError());
    PrefillParams p{q, frag, out, heads, kv_heads, seq_q, seq_kv, spad, scale * 1.4426950408889634f, causal, window, right_context, lengths, hpw, per_kv / hpw, plan.ngroups,
                    mask, mask_b, mask_h, mask_q, mask_k, plan.places, splits, part, part + rows * splits * D, out_rows};
    const dim3 grid(kv_heads * (per_kv / hpw), plan.places, batch * splits);
    constexpr size_t smem = 4 * pf_block_bytes<D>() + 2 * 4 * 64 * sizeof(float2) + 4 * 64 * sizeof(float);
    note_kernel("sdpa_prefill_kernel");
    const int rc = splits > 1 ? (mask ? launch_prefill_kernel<D, true, true>(grid, smem, s, p) : launch_prefill_kernel<D, true, false>(grid, smem, s, p))
                              : (mask ? launch_prefill_kernel<D, false, true>(grid, smem, s, p) : launch_prefill_kernel<D, false, false>(grid, smem, s, p));
    if (rc != 0) return rc;
    SKH_CHECK(hipGetLastError());
    if (splits > 1) {
        sdpa_prefill_merge_kernel<D><<<dim3((unsigned)((rows * (D / 4) + 255) / 256)), dim3(256), 0, s>>>(p, (int64_t)rows);
        SKH_CHECK(hipGetLastError());
    }
    return 1;
}

// No form of this kernel is forced and it is not switched off: the launcher may weigh it against others.
bool sdpa_prefill_by_rule() { return g_prefill_mfma.load() && g_prefill_teams.load() == 0 && g_prefill_splits.load() == 0; }

// Returns 1 when the MFMA path took the call, 0 when the shape is outside its range, -1 on error.
int launch_sdpa_prefill(const float* q, const float* k, const float* v, float* out, int batch, int heads, int kv_heads,
                        int seq_q, int seq_kv, int kv_capacity, int head_dim, float scale, int causal, int window,
                        int right_context, const int32_t* lengths, const float* mask, int mask_b, int mask_h, int mask_q,
                        int mask_k, int out_rows) {
    if (!g_prefill_mfma) return 0;
    // a mask row is read four keys at a time: rows of a multiple of four keys from a 16-byte aligned base (or one value per row)
    if (mask && mask_k != 1 && ((mask_k & 3) || (reinterpret_cast<uintptr_t>(mask) & 15))) return 0;
    if (head_dim != 64 && head_dim != 128) return 0;
    if (seq_q < 16 || seq_q > seq_kv) return 0;          // a handful of rows is the row kernel's business
    if (batch > 65535 || (int64_t)kv_heads * heads > 65535) return 0;
    if ((reinterpret_cast<uintptr_t>(q) | reinterpret_cast<uintptr_t>(k) | reinterpret_cast<uintptr_t>(v) |
         reinterpret_cast<uintptr_t>(out)) & 15) return 0;
    if (head_dim == 64) return launch_prefill_d<64>(q, k, v, out, batch, heads, kv_heads, seq_q, seq_kv, kv_capacity, scale, causal, window, right_context, lengths, mask, mask_b, mask_h, mask_q, mask_k, out_rows);
    return launch_prefill_d<128>(q, k, v, out, batch, heads, kv_heads, seq_q, seq_kv, kv_capacity, scale, causal, window, right_context, lengths, mask, mask_b, mask_h, mask_q, mask_k, out_rows);
}

}  // namespace skh
