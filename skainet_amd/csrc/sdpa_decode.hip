// Decode-shape attention (one query position per sequence, the few of a draft, or a short prompt) over a KV cache: bandwidth-bound split-K.
//
// Same contract as the general kernel in sdpa.hip (reference: skainet_f32_sdpa,
//   /root/reference/skainet-backends/skainet-backend-native-cpu/native/src/f32_fused.c:290-396, rules of
//   /root/reference/skainet-lang/skainet-lang-core/src/commonMain/kotlin/sk/ainet/lang/tensor/ops/AttentionMask.kt:24-104)
// for seq_q == 1 and no additive mask: the attended keys are one range [first, end) per sequence (window, causal
// and key-length rules all cut a range), an empty range means uniform weights over every key.
//
// The K/V rows of a cache are read exactly once, straight from HBM into registers, no LDS staging:
//   * grid (key splits, kv heads x head sub-groups, batch); a workgroup owns one split of the key range of one
//     KV head and GS of the query heads that share it, so a K/V row is loaded once for GS heads;
//   * 16 lanes hold one key row (D / 16 consecutive floats each), a wave covers 4 adjacent keys per load
//     instruction (one contiguous span of 4 rows), the 4 waves interleave groups of 4 keys;
//   * every 16-lane group keeps its own online-softmax state (running max, sum, output slice) for its keys, so
//     the key loop has no cross-lane traffic beyond the 4-step dot-product reduction (DPP rotates inside a row of 16
//     lanes); the 16 states of a workgroup are merged once, through LDS;
//   * splits > 1: each workgroup writes an unnormalised partial (output, max, sum) and a second, small kernel
//     merges them. Merging in the last-arriving workgroup instead was built twice and is slower on this multi-die
//     part: with an agent-scope release / acquire per workgroup (whole L2s written back and invalidated), and with
//     no fence at all -- partials as agent-scope atomic stores / loads that bypass the L2s, one relaxed ticket per
//     workgroup: results identical, but the ticket and the reads behind it are two more trips to memory, about what
//     the second launch costs at 10 splits and far more at 64 (4096 keys: 21.8 us against 12.3).
#include "gemv_q4k.h"

#include <cmath>

namespace skh {

constexpr float SDPA_DECODE_MASKED = -1.0e30f;
constexpr int SDPA_DECODE_MAX_SPLITS = 64;

struct SdpaDecodeParams {
    const float *q, *k, *v;
    float* out;
    int batch, heads, kv_heads, seq_kv, kv_capacity;
    float scale;
    int window, right_context;
    const int32_t* lengths;
    int splits;
    float* part;          // [query rows][splits][D] unnormalised outputs; null: one split, the normalised result goes to out
    float* ml;            // [query rows][splits][2] running maximum (in units of ln 2) and sum of each split
    int subs, tuples;     // workgroups that share a split's keys, and how many such (split, kv head, sequence) there are; tuples 0: a grid of three dimensions
    int seq_q, causal;    // queries per sequence (the last ones of its positions) and whether a later key is hidden from them
    int out_rows;         // the output as [batch, seq_q, heads, D] instead of [batch, heads, seq_q, D]
};

// Scores are kept in units of ln 2 (the query is scaled by scale * log2(e) once), so every exponential of the softmax is
// one v_exp_f32 of a difference: no range reduction, no multiply. For the differences that carry weight (|x| < 30) the
// rounding of the scaled score moves the result by under 3e-6 relative.
constexpr float SDPA_LOG2E = 1.44269504088896340736f;
__device__ __forceinline__ float exp2_raw(float x) { return __builtin_amdgcn_exp2f(x); }
// 2^(m_old - m_new), 0 for an empty state; the exponential is evaluated unconditionally (a select, not a branch)
__device__ __forceinline__ float exp_diff(float m_old, float m_new) {
    const float e = exp2_raw(m_old - m_new);
    return m_old == -INFINITY ? 0.f : e;
}

// ROWS: one query per sequence, a draft of a few (MQ) or a prompt. The rows that share a KV head are then its query heads times
// the queries, GS of them to a workgroup: each has a key range of its own (causal and window move with the query) and the
// workgroup walks the union. A key outside a row's range takes no part in that row: it scores -inf and its V is replaced by
// zeros, since a weight of zero times an infinite or undefined element (a later token's, or the padding of a cache) is not
// zero. Passes whose keys lie in every row's range, nearly all of them, skip both.
// A draft's rows come head by head. A prompt's come query by query, so that a workgroup holds neighbouring queries, at most GS of them: head by head
// some hold the last queries of one head and the first of the next, which share no key under a window (385 queries on 1828 keys under a
// window of 153, 8 heads over 1: 537 keys walked by six of 770 workgroups, about 156 by the others).
// DIES: a grid of one dimension, below. Both are template arguments, since a run-time choice costs every call 0.03 to 0.1 us (DIES) or a draft 0.1 to
// 0.4 (the order of its rows) in front of its first load.
enum DecodeRows { ROWS_ONE, ROWS_DRAFT, ROWS_PROMPT };
template <int GS, int DPL, DecodeRows ROWS, bool DIES>
__global__ __launch_bounds__(256) void sdpa_decode_kernel(SdpaDecodeParams p) {
    constexpr int D = 16 * DPL;
    constexpr bool MQ = ROWS != ROWS_ONE, BY_QUERY = ROWS == ROWS_PROMPT;
    constexpr int U = 2;                       // groups of 4 keys a wave has in flight
    __shared__ __attribute__((aligned(16))) float wacc[16][GS][D];
    __shared__ __attribute__((aligned(16))) float cw[GS][16];
    __shared__ float wm[GS][16], wl[GS][16], wmm[GS], wls[GS];

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);   // uniform, and said so: the key loop's exits stay scalar branches
    const int sub = lane & 15, kg = lane >> 4;
    const int per_kv = p.heads / p.kv_heads;
    const int rows_kv = MQ ? per_kv * p.seq_q : per_kv;        // query rows that share a KV head
    int split = blockIdx.x, b = blockIdx.z, kvh = blockIdx.y, sub_group = 0;
    if constexpr (DIES) {
        // workgroups go to the dies in turn: every eighth one takes the next group of rows of the same keys, so that one L2 has them
        const int turn = blockIdx.x >> 3, tuple = turn / p.subs * 8 + (blockIdx.x & 7);
        if (tuple >= p.tuples) return;
        sub_group = turn % p.subs;
        split = tuple % p.splits;
        kvh = tuple / p.splits % p.kv_heads;
        b = tuple / p.splits / p.kv_heads;
    } else {
        const int subs = MQ ? (rows_kv + GS - 1) / GS : per_kv / GS;
        kvh = blockIdx.y / subs;
        sub_group = blockIdx.y % subs;
    }
    const int r0 = sub_group * GS;
    auto head_of = [&](int r) { return !MQ ? r : BY_QUERY ? r % per_kv : r / p.seq_q; };
    auto query_of = [&](int r) { return !MQ ? 0 : BY_QUERY ? r / per_kv : r % p.seq_q; };
    // row g of the workgroup: its place among the [batch, heads, seq_q] query rows (rows past the last are copies of it)
    int64_t row_of[GS];
    int first_of[GS], end_of[GS];
    bool uniform_of[GS];
    int first = 0x7FFFFFFF, end = 0;           // the union of the rows' ranges, and the keys that all rows share
    int common_first = 0, common_end = 0x7FFFFFFF;
#pragma unroll
    for (int g = 0; g < GS; ++g) {
        const int r = MQ ? min(r0 + g, rows_kv - 1) : r0 + g;
        const int qi = query_of(r), h = head_of(r);
        row_of[g] = MQ ? ((int64_t)b * p.heads + kvh * per_kv + h) * p.seq_q + qi : (int64_t)b * p.heads + kvh * per_kv + h;
        // attended key range of this row's query (one query: absolute position seq_kv - 1, so causal cuts nothing)
        const int pos = MQ ? p.seq_kv - p.seq_q + qi : p.seq_kv - 1;
        int f = 0, e = p.seq_kv;
        if (p.window > 0) {
            f = max(f, pos - p.window + 1);
            e = min(e, pos + p.right_context + 1);
        }
        if (MQ && p.causal) e = min(e, pos + 1);
        if (p.lengths) e = min(e, p.lengths[b]);
        e = max(e, 0);
        uniform_of[g] = f >= e;                // nothing attended: every key scores the same finite value
        if (uniform_of[g]) { f = 0; e = p.seq_kv; }
        first_of[g] = f; end_of[g] = e;
        first = min(first, f); end = max(end, e);
        common_first = max(common_first, f); common_end = min(common_end, e);
    }
    const bool uniform = uniform_of[0];        // one query: the same for all rows of the workgroup
    const int chunk = ((end - first + p.splits - 1) / p.splits + 15) & ~15;
    const int lo = first + split * chunk;
    const int hi = min(end, lo + chunk);

    const float qscale = p.scale * SDPA_LOG2E;
    float qr[GS][DPL];
#pragma unroll
    for (int g = 0; g < GS; ++g) {
        const float* qp = p.q + row_of[g] * D + sub * 4;
#pragma unroll
        for (int d = 0; d < DPL; d += 4) {
            const float4 t = *reinterpret_cast<const float4*>(qp + 16 * d);   // float4 number d / 4 of the lane: elements 64 (d / 4) + 4 sub ..
            qr[g][d] = t.x * qscale; qr[g][d + 1] = t.y * qscale; qr[g][d + 2] = t.z * qscale; qr[g][d + 3] = t.w * qscale;
        }
    }
    float m[GS], l[GS], acc[GS][DPL];
#pragma unroll
    for (int g = 0; g < GS; ++g) {
        m[g] = -INFINITY; l[g] = 0.f;
#pragma unroll
        for (int d = 0; d < DPL; ++d) acc[g][d] = 0.f;
    }

    // A lane's DPL elements of a row are float4s 64 elements apart (float4 number j: elements 64 j + 4 sub ..), so that the
    // 16 lanes of a row read 256 consecutive bytes per load instruction and a row's cache lines are each touched once
    // (with DPL consecutive elements per lane every instruction touched every line of the row).
    const float* kb = p.k + ((int64_t)b * p.kv_heads + kvh) * p.kv_capacity * D + sub * 4;
    const float* vb = p.v + ((int64_t)b * p.kv_heads + kvh) * p.kv_capacity * D + sub * 4;
    // The K / V rows of a pass (U groups of 4 keys per wave) are requested one pass ahead of their use, into the other of
    // two register sets: a split of 64 keys is two passes per wave, and both are in flight from the start.
    constexpr int STEP = 16 * U;
    auto request = [&](float (&kr)[U][DPL], float (&vr)[U][DPL], int k0) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int64_t off = (int64_t)min(k0 + 16 * u + kg, hi - 1) * D;   // a lane past the range re-reads the last row
#pragma unroll
            for (int d = 0; d < DPL; d += 4) {
                const float4 a = *reinterpret_cast<const float4*>(kb + off + 16 * d);
                const float4 c = *reinterpret_cast<const float4*>(vb + off + 16 * d);
                kr[u][d] = a.x; kr[u][d + 1] = a.y; kr[u][d + 2] = a.z; kr[u][d + 3] = a.w;
                vr[u][d] = c.x; vr[u][d + 1] = c.y; vr[u][d + 2] = c.z; vr[u][d + 3] = c.w;
            }
        }
    };
    // cut: some row's range leaves out a key of this pass (MQ only, wave-uniform)
    auto consume = [&](const float (&kr)[U][DPL], const float (&vr)[U][DPL], int k0, auto cut_c) __attribute__((always_inline)) {
        constexpr bool CUT = MQ && decltype(cut_c)::value;
        bool valid[U][MQ ? GS : 1];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int key = k0 + 16 * u + kg;
#pragma unroll
            for (int g = 0; g < (MQ ? GS : 1); ++g)
                valid[u][g] = !MQ ? key < hi : CUT ? key < min(hi, end_of[g]) && key >= first_of[g] : true;
        }
        // Branch-free from here to the end of the body: the U x GS score chains (dot product, row reduction, exponentials)
        // are independent and the compiler interleaves them; behind a per-key branch each ran on its own, one
        // dependent instruction at a time -- with one wave per SIMD that chain, not the memory, set the pace.
        float sc[U][GS];
#pragma unroll
        for (int u = 0; u < U; ++u) {
#pragma unroll
            for (int g = 0; g < GS; ++g) {
                float s = 0.f;
#pragma unroll
                for (int d = 0; d < DPL; ++d) s = fmaf(qr[g][d], kr[u][d], s);
                s = row16_sum(s);
                if (MQ ? uniform_of[g] : uniform) s = SDPA_DECODE_MASKED;
                sc[u][g] = valid[u][MQ ? g : 0] ? s : -INFINITY;
            }
        }
#pragma unroll
        for (int g = 0; g < GS; ++g) {
            // both key groups enter the running state in one update: one rescale of the accumulator per pass
            float m_new = m[g];
#pragma unroll
            for (int u = 0; u < U; ++u) m_new = fmaxf(m_new, sc[u][g]);
            const float alpha = exp_diff(m[g], m_new);
            float pr[U], psum = 0.f;
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const float e = exp2_raw(sc[u][g] - m_new);        // NaN for (-inf) - (-inf): discarded by the select
                pr[u] = valid[u][MQ ? g : 0] ? e : 0.f;
                psum += pr[u];
            }
            l[g] = fmaf(l[g], alpha, psum);
#pragma unroll
            for (int d = 0; d < DPL; ++d) {
                float a = acc[g][d] * alpha;
#pragma unroll
                for (int u = 0; u < U; ++u) a = fmaf(pr[u], CUT && !valid[u][g] ? 0.f : vr[u][d], a);
                acc[g][d] = a;
            }
            m[g] = m_new;
        }
    };
    // Passes are taken in pairs so that the loop has one exit and one back edge (with an exit between the two halves
    // the compiler's wait-count pass sees a path on which the second set is still in flight at the loop head and makes
    // every request wait for it). The second half of the last pair may lie past the range: none of its keys is valid
    // and it leaves the running state as it is.
    float ka[U][DPL], va[U][DPL], kb2[U][DPL], vb2[U][DPL];
    const int k_first = lo + wave * 4;
    if (k_first < hi) request(ka, va, k_first);                 // wave-uniform
    auto pair = [&](int k0, auto cut) __attribute__((always_inline)) {
        request(kb2, vb2, k0 + STEP);                           // past the range: clamped re-reads of the last row
        __builtin_amdgcn_sched_barrier(0);                      // requests are issued where they are written, ahead of the arithmetic
        consume(ka, va, k0, cut);
        request(ka, va, k0 + 2 * STEP);
        __builtin_amdgcn_sched_barrier(0);
        consume(kb2, vb2, k0 + STEP, cut);
    };
    int k0 = k_first;
    if constexpr (MQ) {
        // a pair of passes whose keys all rows attend; a loop of each kind, not a branch inside one (199 instead of 158 registers)
        auto whole = [&] { return k0 >= common_first && k0 + STEP + 16 * (U - 1) + 4 <= min(hi, common_end); };
        for (; k0 < hi && !whole(); k0 += 2 * STEP) pair(k0, std::true_type{});
        for (; whole(); k0 += 2 * STEP) pair(k0, std::false_type{});
    }
    for (; k0 < hi; k0 += 2 * STEP) pair(k0, std::true_type{});

    // Merge the 16 running states of the workgroup (4 lane groups x 4 waves) through LDS: every lane parks its slice,
    // one 16-lane row per head works out the 16 weights 2^(m_s - max) and the weighted sum of the l_s, then each thread
    // sums its output elements over the states. (Merging lane groups by shuffles first cost 80 crossbar round trips and
    // 16 exponentials per lane.) A lane's float4 number j holds elements 64 j + 4 sub .. of the row, so the 16 lanes of
    // a row store 256 contiguous bytes and a state lies in LDS in the row's own element order.
    const int state = wave * 4 + kg;
#pragma unroll
    for (int g = 0; g < GS; ++g) {
#pragma unroll
        for (int j = 0; j < DPL / 4; ++j)
            *reinterpret_cast<float4*>(&wacc[state][g][j * 64 + sub * 4]) =
                make_float4(acc[g][4 * j], acc[g][4 * j + 1], acc[g][4 * j + 2], acc[g][4 * j + 3]);
        if (sub == 0) { wm[g][state] = m[g]; wl[g][state] = l[g]; }
    }
    __syncthreads();
    if (threadIdx.x < 16 * GS) {
        const int g = threadIdx.x >> 4, st = threadIdx.x & 15;
        const float ms = wm[g][st];
        const float mm = row16_max(ms);
        const float c = exp_diff(ms, mm);
        const float ls = row16_sum(c * wl[g][st]);
        cw[g][st] = c;
        if (st == 0) { wmm[g] = mm; wls[g] = ls; }
    }
    __syncthreads();

    constexpr int EPT = GS * D >= 256 ? GS * D / 256 : 1;       // output elements per thread, adjacent inside one head
    if (threadIdx.x * EPT < GS * D) {
        const int g = threadIdx.x * EPT / D, i0 = threadIdx.x * EPT % D;
        float c[16], o[EPT];
#pragma unroll
        for (int q4 = 0; q4 < 4; ++q4) {
            const float4 t = *reinterpret_cast<const float4*>(&cw[g][4 * q4]);
            c[4 * q4] = t.x; c[4 * q4 + 1] = t.y; c[4 * q4 + 2] = t.z; c[4 * q4 + 3] = t.w;
        }
#pragma unroll
        for (int e = 0; e < EPT; ++e) o[e] = 0.f;
#pragma unroll
        for (int st = 0; st < 16; ++st)
#pragma unroll
            for (int e = 0; e < EPT; ++e) o[e] = fmaf(wacc[st][g][i0 + e], c[st], o[e]);
        if (MQ && r0 + g >= rows_kv) return;
        const float mm = wmm[g], ls = wls[g];
        int64_t row = row_of[0];
#pragma unroll
        for (int e = 1; e < GS; ++e) row = g == e ? row_of[e] : row;
        int64_t out_row = row;
        if (MQ && p.out_rows) out_row = ((int64_t)b * p.seq_q + query_of(r0 + g)) * p.heads + kvh * per_kv + head_of(r0 + g);
#pragma unroll
        for (int e = 0; e < EPT; ++e) {
            const int d = i0 + e;                                   // a state's layout in LDS is the row's own element order
            if (!p.part) {
                p.out[out_row * D + d] = ls == 0.f ? 0.f : o[e] / ls;   // an undefined score leaves an undefined sum: no zero for it
            } else {
                p.part[(row * p.splits + split) * D + d] = o[e];
                if (d == 0) *reinterpret_cast<float2*>(p.ml + (row * p.splits + split) * 2) = make_float2(mm, ls);
            }
        }
    }
}

// Merge the per-split (unnormalised output, max, sum) triples of one query row. 4 * D threads: thread (j, d) folds
// splits j, j + 4, ... of output element d (independent loads, all in flight together), LDS folds the four. The
// softmax weights of the splits -- exp(max_s - max) / sum -- are worked out once, by the first wave: one split per
// lane, maximum and sum by wave reductions (splits <= 64), parked in LDS for everyone.
template <int D>
__global__ __launch_bounds__(4 * D) void sdpa_decode_combine_kernel(const float* __restrict__ part, const float* __restrict__ ml,
                                                                    float* __restrict__ out, int splits, int heads, int seq_q, int out_rows) {
    __shared__ float sw[SDPA_DECODE_MAX_SPLITS];
    __shared__ float so[4][D];
    const float* src = part + (int64_t)blockIdx.x * splits * D;
    const float2* src_ml = reinterpret_cast<const float2*>(ml) + (int64_t)blockIdx.x * splits;
    const int d = threadIdx.x % D, j = threadIdx.x / D;
    float pv[SDPA_DECODE_MAX_SPLITS / 4];
#pragma unroll
    for (int i = 0; i < SDPA_DECODE_MAX_SPLITS / 4; ++i) {
        const int sp = j + 4 * i;
        pv[i] = src[min(sp, splits - 1) * D + d];               // clamped: a split past the end gets weight zero below
    }
    if (threadIdx.x < 64) {
        const int sp = threadIdx.x;
        const bool live = sp < splits;
        const float2 st = live ? src_ml[sp] : make_float2(-INFINITY, 0.f);
        const float m = st.x, l = st.y;
        float mm = m;
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) mm = fmaxf(mm, __shfl_xor(mm, off, 64));
        const float w = exp_diff(m, mm);
        const float ls = wave_sum(l * w);
        if (sp < SDPA_DECODE_MAX_SPLITS) sw[sp] = ls == 0.f ? 0.f : w / ls;
    }
    __syncthreads();
    float o = 0.f;
#pragma unroll
    for (int i = 0; i < SDPA_DECODE_MAX_SPLITS / 4; ++i) {
        const int sp = j + 4 * i;
        o = fmaf(pv[i], sp < splits ? sw[sp] : 0.f, o);
    }
    so[j][d] = o;
    __syncthreads();
    int64_t row = blockIdx.x;
    if (out_rows) {
        const int qi = blockIdx.x % seq_q, bh = blockIdx.x / seq_q;
        row = ((int64_t)(bh / heads) * seq_q + qi) * heads + bh % heads;
    }
    if (j == 0) out[row * D + d] = so[0][d] + so[1][d] + so[2][d] + so[3][d];
}

float* sdpa_workspace(size_t bytes);   // shim.hip: per-thread scratch, grown on demand

static std::atomic<int> g_sdpa_decode_split_keys{64};   // least keys per split (a multiple of 16)
void set_sdpa_decode_split_keys(int v) { if (v >= 16) g_sdpa_decode_split_keys = (v + 15) & ~15; }

template <int GS, int DPL, DecodeRows ROWS>
static int launch_decode_variant(const SdpaDecodeParams& p, int subs, bool merge) {
    constexpr int D = 16 * DPL;
    note_kernel("sdpa_decode_kernel");
    if (p.tuples) sdpa_decode_kernel<GS, DPL, ROWS, true><<<dim3((unsigned)((p.tuples + 7) / 8 * 8 * subs)), dim3(256), 0, current_stream()>>>(p);
    else sdpa_decode_kernel<GS, DPL, ROWS, false><<<dim3(p.splits, p.kv_heads * subs, p.batch), dim3(256), 0, current_stream()>>>(p);
    SKH_CHECK(hipGetLastError());
    if (merge) {
        sdpa_decode_combine_kernel<D><<<dim3(p.batch * p.heads * p.seq_q), dim3(4 * D), 0, current_stream()>>>(p.part, p.ml, p.out, p.splits, p.heads, p.seq_q, p.out_rows);
        SKH_CHECK(hipGetLastError());
    }
    return 1;
}
template <int DPL, DecodeRows ROWS>
static int launch_decode_rows(const SdpaDecodeParams& p, int gs, int subs, bool merge) {
    if constexpr (DPL <= 8) { if (gs == 4) return launch_decode_variant<4, DPL, ROWS>(p, subs, merge); }
    if (gs == 2) return launch_decode_variant<2, DPL, ROWS>(p, subs, merge);
    return launch_decode_variant<1, DPL, ROWS>(p, subs, merge);
}
template <int DPL>
static int launch_decode_d(const SdpaDecodeParams& p, int gs, int subs, bool merge) {
    if constexpr (DPL <= 8) { if (p.seq_q >= 16) return launch_decode_rows<DPL, ROWS_PROMPT>(p, gs, subs, merge); }
    return p.seq_q > 1 ? launch_decode_rows<DPL, ROWS_DRAFT>(p, gs, subs, merge) : launch_decode_rows<DPL, ROWS_ONE>(p, gs, subs, merge);
}

static std::atomic<int> g_sdpa_decode_gs{0};            // query heads per workgroup: 0 = chosen from the shape, else 1 / 2 / 4
void set_sdpa_decode_gs(int v) { if (v == 0 || v == 1 || v == 2 || v == 4) g_sdpa_decode_gs = v; }
static std::atomic<int> g_sdpa_decode_dies{1};
void set_sdpa_decode_dies(int v) { g_sdpa_decode_dies = v != 0; }
static std::atomic<int> g_sdpa_decode_prompts{1};       // prompts on this kernel: 0 never, 1 by rule, 2 wherever it fits
void set_sdpa_decode_prompts(int v) { if (v >= 0 && v <= 2) g_sdpa_decode_prompts = v; }
static std::atomic<int> g_sdpa_decode_one_launch{1};
void set_sdpa_decode_one_launch(int v) { g_sdpa_decode_one_launch = v != 0; }
static std::atomic<int> g_attn_merge_max_keys{176};    // most keys per split the unmerged form accepts (a multiple of 16)
void set_attn_merge_max_keys(int v) { if (v >= 16) g_attn_merge_max_keys = (v + 15) & ~15; }
// most splits the unmerged form uses. Measured in a Llama-3-8B decode step at 520 to 650 keys (ms per token): 2 splits 1.637,
// 4: 1.565, 6: 1.540, 8: 1.556; the merge in a launch of its own 1.551 -- every split costs each of the projection's 251
// workgroups another 16 KB of loads, every split less costs the attention workgroups another pass over their keys.
static std::atomic<int> g_attn_merge_splits{6};
void set_attn_merge_splits(int v) { if (v >= 1 && v <= ATTN_MERGE_MAX_SPLITS) g_attn_merge_splits = v; }

double sdpa_prefill_estimate(int batch, int heads, int kv_heads, int seq_q, int seq_kv, int head_dim, int causal, int window, int right_context);   // sdpa_prefill.hip

// Whether a prompt (16 queries and more, no mask) goes to this kernel instead of the matrix-core one, which lays K and V out in a launch of
// its own and sets up a workgroup of eight waves for 32 queries: 8 to 11 us whatever little there is to do. Here a workgroup takes four rows
// straight from the caller's memory, in one launch up to 256 keys and more, with fp32 operands (the other rounds them to bf16). What ends it is the
// K and V that every four rows read for themselves. Both sides by what they do, in us back to back from the host: here the longest workgroup's
// keys and all keys walked over the CUs (whichever is the longer, the fourth root of fourth powers between them), rounds of workgroups, and K and V once;
// fitted to the 42 000 random prompts of the other estimate (12 % rms); this one has to be a sixth below. Of 23 384 other prompts of those ranges
// 11 216 take it, 1.585x, 29 of them more than 5 % slower: 28 queries, one head, D 64 8.9 -> 5.6 us, 60 queries, 16 heads over 2, D 128 12.0 -> 5.7.
// (Straight lines through the keys, fitted up to 2048 earlier ones, took 5 % more, 973 of 21 378 slower, by up to 3.3 times: beyond the fit they
// did not know that the other kernel splits its keys, nor under a window what its workgroups walk.)
bool sdpa_decode_takes_prompt(int batch, int heads, int kv_heads, int seq_q, int seq_kv, int head_dim, int causal, int window, int right_context) {
    if ((head_dim != 64 && head_dim != 128) || seq_q > seq_kv) return false;
    if (g_sdpa_decode_prompts.load() != 1) return g_sdpa_decode_prompts.load() == 2;
    const double cus = num_cus(), groups = (double)batch * kv_heads * (((int64_t)(heads / kv_heads) * seq_q + 3) / 4);
    double keys = causal ? seq_kv - 0.5 * (seq_q - 1) : seq_kv, most = seq_kv, all = seq_kv;       // of a query on average, of a workgroup, of the call
    if (window > 0) {
        keys = fmin(keys, (double)window + right_context);
        most = fmin(most, (double)window + right_context + 3);
        all = fmin(all, (double)window + right_context + seq_q);
    }
    const double splits = fmax(1.0, fmin(ceil(2 * cus / groups), fmin(SDPA_DECODE_MAX_SPLITS, ceil(most / 64)))), rounds = ceil(groups * splits / cus);
    const double chain = most / 64 / splits, walked = groups * keys / 64 / cus, mb = 8e-6 * batch * kv_heads * all * head_dim;
    auto longer = [](double a, double b) { return sqrt(sqrt(a * a * a * a + b * b * b * b)); };
    const double here = head_dim == 64 ? fmax(6.58, 3.08 + longer(1.68 * chain, 0.78 * walked) + 0.98 * rounds + 0.318 * mb)
                                       : fmax(5.83, 5.26 + longer(0.65 * chain, 1.35 * walked) + 0.875 * rounds + 0.095 * mb);
    return 1.2 * here < sdpa_prefill_estimate(batch, heads, kv_heads, seq_q, seq_kv, head_dim, causal, window, right_context);
}

// Returns 1 when this kernel took the call, 0 when the shape is outside its range (the caller uses the general
// kernel), -1 on error. With `leave` the per-split results are left unmerged for a consumer that folds the merge into
// its own activation load (at most ATTN_MERGE_MAX_SPLITS splits, one sequence): `out` is not written, *leave describes
// where the partials are; 0 when the key count would need more splits than that.
int launch_sdpa_decode(const float* q, const float* k, const float* v, float* out, int batch, int heads, int kv_heads,
                       int seq_q, int seq_kv, int kv_capacity, int head_dim, float scale, int causal, int window, int right_context,
                       const int32_t* lengths, AttnMergePrologue* leave, int out_rows) {
    if (seq_q > seq_kv) return 0;
    if (head_dim != 64 && head_dim != 128 && head_dim != 256) return 0;
    if ((reinterpret_cast<uintptr_t>(q) | reinterpret_cast<uintptr_t>(k) | reinterpret_cast<uintptr_t>(v)) & 15) return 0;
    const int per_kv = heads / kv_heads;
    const int gs_max = head_dim == 256 ? 2 : 4;
    int gs = g_sdpa_decode_gs.load() > 0 ? min(g_sdpa_decode_gs.load(), gs_max) : gs_max;
    const bool draft = seq_q > 1;
    // one query: GS divides the heads of a KV head; several: the last workgroup of a KV head may be padded, so a group is
    // only not wider than the rows there are
    while (draft ? gs > 2 && per_kv * seq_q <= gs / 2 : per_kv % gs != 0) gs >>= 1;
    // keys that a query can attend: a window bounds them whatever the cache holds
    // (a prompt: those of a workgroup's rows, at most four neighbouring queries; with all queries' 385 x 1828 under a window of 153 was split and took 21 us)
    const int keys = window > 0 ? (int)min((int64_t)seq_kv, (int64_t)window + right_context + (seq_q < 16 ? seq_q - 1 : 3)) : seq_kv;
    // One split, no merge behind it: the merge is a second launch (2.8 us of a host's time, and about that between two
    // dependent kernels on the device), which buys the parallelism of the splits -- and shorter sums: with one split the error
    // against float64 is up to a third larger (950 keys 1.6e-7 and 2.1e-7). So two estimates in us both have to say that it pays.
    // Measured, 32 heads over 8, D 128, one sequence: 128 keys 7.1 -> 4.6 us, 512 keys 6.8 -> 6.0; 16 sequences at 1024 keys 25.1 -> 20.6;
    // 8950 random calls of 1 to 8 queries take 0.785 of their time with splits, 8 of them more than 5 % longer (by the first estimate
    // alone 0.785 and 107 of 15 500). A key count on the device (a decode step over a growing cache)
    // stays with splits above 256: `keys` is then only a bound, and between a layer's products the cache comes from memory,
    // where a chain of passes waits longer (19 layers at 430 keys: 608 us per step with splits, 664 with one).
    bool single = false;
    const int cols = draft ? per_kv * seq_q : per_kv;           // rows that share a KV head
    if (g_sdpa_decode_one_launch && !leave && g_sdpa_decode_gs.load() == 0 && keys > g_sdpa_decode_split_keys &&
        keys <= (lengths ? 256 : 2048)) {
        const double once = 8e-6 * batch * kv_heads * keys * head_dim, cus = num_cus();       // MB of K and V
        const int gs_most = gs, wide = head_dim > 64, slot[5] = {0, 0, 1, 0, 2};              // slot: 1, 2, 4 rows per workgroup
        auto groups_of = [&](int g) { return (double)((cols + g - 1) / g); };
        auto takes = [&](int g) { return draft ? g == 1 || cols > g / 2 : per_kv % g == 0; };
        // The first: passes of 32 keys (a chain of loads and arithmetic, longer with more rows per workgroup) or the traffic, every
        // group of rows that shares a KV head reading it for itself; with splits the traffic alone.
        static const double pass[2][3] = {{0.137, 0.21, 0.32}, {0.21, 0.30, 0.54}};           // [D 64, 128][slot]
        bool pays = false;
        for (int g = 1; g <= gs_most && takes(g); g *= 2) {
            const double wgs = groups_of(g) * batch * kv_heads, rate = wgs >= 128 ? 7.5 : 6.3 * fmin(1.0, sqrt(wgs / 64));
            const double one = fmax(4.4, 2.7 + fmax((keys + 31) / 32 * pass[wide][slot[g]] * (head_dim == 256 ? 2 : 1), once * groups_of(g) / rate));
            pays |= one < 0.95 * fmax(6.8, 4.9 + once * groups_of(gs_most) / 6.9);
        }
        // The second, fitted to 15 500 random calls with splits (within 5 %) and with one, counts what the first does not: loads of 1
        // and 2 rows that miss the L2s (32 MB together; a group of rows per die keeps a copy of its own), workgroups that leave the CUs
        // uneven shares or crowd the memory from half of them, and the partial outputs. The chains are per 64 keys.
        static const double hit[2][3] = {{0.235, 0.40, 0.75}, {0.395, 0.60, 1.07}}, miss[2][3] = {{0.44, 0.51, 0.75}, {0.64, 0.68, 1.08}};
        auto misses = [&](int g) { return once * fmin(groups_of(g), 8) > 32; };
        auto chain = [&](int g) { return (misses(g) ? miss : hit)[wide][slot[g]] * (head_dim == 256 ? 2 : 1); };
        auto uneven = [&](double wgs) { return wgs > cus ? ceil(wgs / cus) * cus / wgs : 1.0; };
        const int gs_split = gs == 4 && !draft && batch * kv_heads * (per_kv / 4) * fmin(SDPA_DECODE_MAX_SPLITS, (keys + 63) / 64) < cus ? 2 : gs;     // as below
        const double groups_split = groups_of(gs_split) * batch * kv_heads, rows = (double)batch * heads * seq_q;
        const int splits_est = (int)fmin(fmin(SDPA_DECODE_MAX_SPLITS, (keys + 63) / 64), ceil(2 * cus / groups_split));
        const double passes = ((keys + splits_est - 1) / splits_est + 63) / 64, wgs_split = groups_split * splits_est;
        double best = 0.95 * fmax(8.0, 4.9 + fmax(1.26 * chain(gs_split) * passes * ceil(wgs_split / cus),
                                                  once * groups_of(gs_split) * uneven(wgs_split) / (misses(gs_split) ? 9.5 : 34)) +
                                       8.4e-6 * rows * head_dim * splits_est + 8e-4 * rows);
        for (int g = 1; pays && g <= gs_most && takes(g); g *= 2) {
            const double wgs = groups_of(g) * batch * kv_heads, traffic = once * groups_of(g) * uneven(wgs) / (misses(g) ? 7.5 : 20);
            const double crowded = wide && misses(g) && 2 * wgs > cus ? 1.4 : 1.0;
            const double t = fmax(4.4, 3.7 + fmax((keys + 63) / 64 * chain(g) * crowded, traffic));
            if (t < best) { best = t; gs = g; single = true; }
        }
    }
    // Few workgroups (one sequence at a short context, or splits capped for the projection that merges them): two query
    // heads per workgroup instead of four. The K / V rows are then fetched by two workgroups (the second from L2), each
    // with half the arithmetic per pass, and twice as many CUs take part: 1.502 against 1.526 ms per token in a
    // Llama-3-8B decode step at 520 to 650 keys (one head per workgroup: 1.529).
    if (g_sdpa_decode_gs.load() == 0 && gs == 4 && !draft && !single) {
        const int64_t groups4 = (int64_t)batch * kv_heads * (per_kv / 4);
        const int most = leave ? g_attn_merge_splits.load() : SDPA_DECODE_MAX_SPLITS;
        const int splits4 = min(most, (keys + g_sdpa_decode_split_keys - 1) / g_sdpa_decode_split_keys);
        if (groups4 * splits4 < num_cus()) gs = 2;
    }
    const int subs = (cols + gs - 1) / gs;
    if (batch > 65535 || (int64_t)kv_heads * subs > 65535) return 0;
    SdpaDecodeParams p{q, k, v, out, batch, heads, kv_heads, seq_kv, kv_capacity, scale, window, right_context, lengths, 1,
                       nullptr, nullptr, subs, 0, seq_q, causal, out_rows && seq_q > 1};
    // enough workgroups to put every CU on the cache, at least 64 keys per split (measured in the decoder at 500 to 650
    // keys: 32 or 48 keys per split 2.5 % slower per token, 96 and 128 keys the same as 64)
    const int64_t groups = (int64_t)batch * kv_heads * subs;
    int splits = (int)((2 * (int64_t)num_cus() + groups - 1) / groups);
    splits = min(splits, min(SDPA_DECODE_MAX_SPLITS, (keys + g_sdpa_decode_split_keys - 1) / g_sdpa_decode_split_keys));
    if (splits < 1) splits = 1;
    // what the partials of this many splits take is held by the one-split form as well: a cache that grows into splits then
    // does not move the scratch under a graph recorded before
    if (splits > 1 && !sdpa_workspace(sizeof(float) * (size_t)batch * heads * seq_q * splits * (head_dim + 2))) return -1;
    if (single) splits = 1;
    if (leave) {
        if (batch != 1) return 0;
        const int most = g_attn_merge_splits;
        if (splits > most) {
            if ((keys + most - 1) / most > g_attn_merge_max_keys) return 0;
            splits = most;
        }
    }
    p.splits = splits;
    // Workgroups that share keys on one die each, where the dies' own copies of them would not stay in the L2s (32 MB together): 8 queries,
    // 8 heads over 2, three sequences at 3815 keys 37.7 -> 24.1 us, one query, 8 heads over 1, six at 6012 18.8 -> 14.0, 16 over 2, six at 4556,
    // D 64, 18.5 -> 14.6. Of 4733 random calls those with 24 to 32 MB together take 1.00 of their
    // time, 32 to 40 0.96, 64 to 90 0.89, above 140 0.81. Few groups leave the dies uneven shares (3 queries, 4 heads over
    // 1, three at 1720 8.3 -> 9.3).
    const int64_t tuples = (int64_t)batch * kv_heads * splits;
    const double mb = 8e-6 * batch * kv_heads * keys * head_dim;
    if (g_sdpa_decode_dies && mb * min(subs, 8) > 34 && subs > 1 && (tuples >= 24 || (tuples + 7) / 8 * subs <= num_cus() / 8) &&
        (tuples + 7) / 8 * 8 * subs <= 0xFFFFFFFFll / 256)      // a dimension of a grid holds 2^32 work-items
        p.tuples = (int)tuples;
    if (splits > 1 || leave) {
        const size_t rows = (size_t)batch * heads * seq_q;
        p.part = sdpa_workspace(sizeof(float) * rows * splits * (head_dim + 2));
        if (!p.part) return -1;
        p.ml = p.part + rows * splits * head_dim;
    }
    if (leave) *leave = AttnMergePrologue{p.part, p.ml, splits, head_dim};
    const bool merge = splits > 1 && !leave;
    if (head_dim == 64) return launch_decode_d<4>(p, gs, subs, merge);
    if (head_dim == 128) return launch_decode_d<8>(p, gs, subs, merge);
    return launch_decode_d<16>(p, gs, subs, merge);
}

int launch_q4k_gemv_mfma(const uint8_t* w, const float* x, float* y, int k, int n, const float* gain, float eps,
                         const float* residual, int epilogue, const RopeQkvEpilogue* rope_in,
                         const AttnMergePrologue* merge);   // gemv_q4k_mfma.hip
bool q4k_gemv_mfma_accepts_merge(int k, int n, int head_dim);   // gemv_q4k_mfma.hip

static std::atomic<int> g_attn_merge_enable{1};
void set_attn_merge_enable(int v) { g_attn_merge_enable = v; }

// One decode token's attention over the cache and the Q4_K output projection behind it as two launches: the attention
// kernel leaves its per-split results unmerged and the projection's activation load merges them (the merge launch and its
// round trip through memory disappear). out[n] = (residual ? residual : 0) + Wo[n, heads * head_dim] . attention.
// Returns 1 when the pair took the call, 0 when the shapes are outside its range (nothing launched), -1 on error.
int launch_attn_out_proj_q4k(const uint8_t* wo, int n, int k, const float* q, const float* k_cache, const float* v_cache, int heads,
                             int kv_heads, int head_dim, int seq_kv, int kv_capacity, float scale, int window,
                             const int32_t* lengths, const float* residual, float* out) {
    if (!g_attn_merge_enable || k != heads * head_dim || k > 4096 || (k & 1023)) return 0;
    if (heads % kv_heads != 0 || seq_kv < 1 || kv_capacity < seq_kv) return 0;
    // dry checks of the projection first: once the attention kernel has run without a merge there is no way back
    if ((reinterpret_cast<uintptr_t>(wo) & 15) || !q4k_gemv_mfma_accepts_merge(k, n, head_dim)) return 0;
    if (residual && (reinterpret_cast<uintptr_t>(residual) & 3)) return 0;
    AttnMergePrologue am{};
    const int r = launch_sdpa_decode(q, k_cache, v_cache, nullptr, 1, heads, kv_heads, 1, seq_kv, kv_capacity, head_dim, scale, 1, window, 0,
                                     lengths, &am, 0);
    if (r <= 0) return r;
    const int g = launch_q4k_gemv_mfma(wo, nullptr, out, k, n, nullptr, 0.f, residual, residual ? EPI_RESIDUAL : EPI_NONE, nullptr, &am);
    if (g == 0) return set_error("attn_out_proj: the projection refused a shape its checks had passed (n %d, k %d)", n, k);
    return g;
}

}  // namespace skh
