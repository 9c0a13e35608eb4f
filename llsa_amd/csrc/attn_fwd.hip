// Block-sparse flash-attention forward for llsa_l1 / llsa_l2.
//
// One wave owns one or two query blocks (16 queries each).  All products run on the bf16 16x16x32 MFMA
// in the "transposed" orientation, keys on the M axis and queries on the N axis:
//     S^T (16 keys x 16 queries) = K_blk (16x64) . Q^T            A = R tile of K, B = R tile of Q
//     O^T (64 ch  x 16 queries) += V_blk^T (64x32 keys) . P^T     A = T tiles of V, B = P^T
// With this orientation lane l holds, for query l%16, the scores of keys 4*(l/16)..+3 of a
// tile -- which is exactly the B-operand layout of the second product -- and the O^T
// accumulator of lane l belongs to the same query, so the soft-max statistics (running
// max, running sum, rescale factor) never leave the lane that needs them; a row reduction
// is two cross-lane steps (lanes l, l^16, l^32, l^48).
//
// KV order per query block: (l2) the 16*T2 level-1 pooled tokens inside the parent's selected
// coarse blocks, then every token of the coarsest pooled level, then the T selected 16-token
// blocks of K/V (the reference walks the same set fine blocks first; the order only moves
// roundings).  Pooled segments count with weight w1 / w2: the accumulator and the running sum
// are kept in units of the current segment's weight, converted once at each segment boundary.
#include "llsa_device.h"
#include "llsa_host.h"
#include "transpose_device.h"
#include "../../include/llsa_hip.h"

namespace llsa {

constexpr float kMaxSum = 256.f;

struct SoftmaxState {
    float m2;        // reference point of the exponentials (at most log2(kMaxSum) below the running max), log2 units
    f32x4 acc[4];    // O^T: channel 16*dt + 4*(l/16) + e of query l%16, in units of the current weight
    float lsum;      // this lane's share of the running sum of the query's p
};

// Operands of one step = NB 16-key blocks (NB even: a pair of blocks is one K step of the second product), as they sit in
// registers between load and use.
template <int NB> struct KeyRegs { bf16x8 k[NB][2]; };       // K rows (R tile): block j, channel half
template <int NB> struct ValueRegs { bf16x8 v[NB / 2][4]; }; // V (T tiles of a pair of blocks): channel tile dt, keys 4*(l/16)..+3 of the first block, then of the second

__device__ __forceinline__ void init_state(SoftmaxState& st) {
    st.m2 = 0.f;
    st.lsum = 0.f;
#pragma unroll
    for (int dt = 0; dt < 4; dt++) st.acc[dt] = f32x4{0.f, 0.f, 0.f, 0.f};
}

// Changes the unit the accumulator and the running sum are kept in (at a boundary between segments of different weight).
__device__ __forceinline__ void rescale(SoftmaxState& st, float f) {
    st.lsum *= f;
#pragma unroll
    for (int dt = 0; dt < 4; dt++) st.acc[dt] *= f;
}

// The exponentials refer to st.m2, which follows the running maximum lazily: it moves only when p has become large
// (some lane's p of a step -- eight of two fine blocks, sixteen of four pooled ones -- add up to more than kMaxSum; smaller
// ones are harmless in bf16 and in the fp32 sums), so that the accumulator is rescaled a few times per query block instead of at most steps; O = acc / sum and
// lse = m2 + log2(sum) hold for any reference point.  The common path therefore needs no maximum, neither over the quad of
// lanes that share a query nor over a lane's own exponents: the sum that is taken anyway tells (overflow included), and only
// when one in the wave is too large is the reference point moved (for all four lanes of a query alike, by the quad's largest
// exponent) and the step's p taken again.  st.m2 starts at the largest score of the first block (start_reference), so it is
// always finite.
__device__ __forceinline__ void start_reference(SoftmaxState& st, const bf16x8 bq[2], bf16x8 k0, bf16x8 k1) {
    f32x4 z = {0.f, 0.f, 0.f, 0.f};
    const f32x4 s = mfma_bf16(k1, bq[1], mfma_bf16(k0, bq[0], z));
    st.m2 = quad_max(fmaxf(fmaxf(s[0], s[1]), fmaxf(s[2], s[3]))) * kScaleLog2e;
}

// x: the exponents of one step relative to st.m2
template <int NB>
__device__ __forceinline__ void exponents(float x[NB][4], const SoftmaxState& st, const bf16x8 bq[2], const KeyRegs<NB>& t) {
#pragma unroll
    for (int j = 0; j < NB; j++) {
        f32x4 z = {0.f, 0.f, 0.f, 0.f};
        const f32x4 s = mfma_bf16(t.k[j][1], bq[1], mfma_bf16(t.k[j][0], bq[0], z));
#pragma unroll
        for (int e = 0; e < 4; e++) x[j][e] = fmaf(s[e], kScaleLog2e, -st.m2);
    }
}
// p of one step as the B operands of the second product; returns the lane's sum of them.  (pin_in_registers keeps the compiler
// from moving the conversion behind the branch that follows, where the fp32 values would occupy twice the registers.)
template <int NB>
__device__ __forceinline__ float probabilities(bf16x8 bp[NB / 2], const float x[NB][4]) {
    float rs[2];
#pragma unroll
    for (int j = 0; j < NB; j++)
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const float p = exp2_fast(x[j][e]);
            if (j < 2 && e == 0) rs[j] = p;
            else rs[j & 1] += p;
            bp[j >> 1][(j & 1) * 4 + e] = (bf16)p;
        }
#pragma unroll
    for (int c = 0; c < NB / 2; c++) pin_in_registers(bp[c]);
    return rs[0] + rs[1];
}
// in0, in1 (wave-uniform): whether the query block reads the step's first / second block
__device__ __forceinline__ void leave_out(float x[2][4], bool in0, bool in1) {
    if (!in0) x[0][0] = x[0][1] = x[0][2] = x[0][3] = -INFINITY;
    if (!in1) x[1][0] = x[1][1] = x[1][2] = x[1][3] = -INFINITY;
}
// the rare path, from the step's exponents taken once more: moves the reference point of every query whose largest one is above it
template <int NB>
__device__ __forceinline__ float move_reference(SoftmaxState& st, bf16x8 bp[NB / 2], float x[NB][4]) {
    float top = x[0][0];
#pragma unroll
    for (int j = 0; j < NB; j++)
#pragma unroll
        for (int e = 0; e < 4; e++) top = fmaxf(top, x[j][e]);
    const float shift = fmaxf(quad_max(top), 0.f);
    st.m2 += shift;
    rescale(st, exp2_fast(-shift));
#pragma unroll
    for (int j = 0; j < NB; j++)
#pragma unroll
        for (int e = 0; e < 4; e++) x[j][e] -= shift;
    return probabilities<NB>(bp, x);
}
template <int NB>
__device__ __forceinline__ void accumulate(SoftmaxState& st, float rs, const bf16x8 bp[NB / 2], const ValueRegs<NB>& t) {
    st.lsum += rs;
#pragma unroll
    for (int c = 0; c < NB / 2; c++)
#pragma unroll
        for (int dt = 0; dt < 4; dt++)
            st.acc[dt] = mfma_bf16(t.v[c][dt], bp[c], st.acc[dt]);
}

// One step of two blocks for Q query blocks that read the same operands, written as one straight-line piece so that the products of one query block overlap with the
// exponentials of the other (one test for the rare path covers all).
template <int Q>
__device__ __forceinline__ void compute_step(SoftmaxState (&st)[Q], const bf16x8 (&bq)[Q][2], const KeyRegs<2>& k, const ValueRegs<2>& v) {
    bf16x8 bp[Q][1];
    float rs[Q], most = 0.f;
#pragma unroll
    for (int u = 0; u < Q; u++) {
        float x[2][4];
        exponents<2>(x, st[u], bq[u], k);
        rs[u] = probabilities<2>(bp[u], x);
        most = fmaxf(most, rs[u]);
    }
    if (__ballot(most > kMaxSum) != 0)
#pragma unroll
        for (int u = 0; u < Q; u++) {
            float x[2][4];
            exponents<2>(x, st[u], bq[u], k);
            rs[u] = move_reference<2>(st[u], bp[u], x);
        }
#pragma unroll
    for (int u = 0; u < Q; u++) accumulate<2>(st[u], rs[u], bp[u], v);
}
__device__ __forceinline__ void compute_step(SoftmaxState& st, const bf16x8 (&bq)[2], const KeyRegs<2>& k, const ValueRegs<2>& v, bool in0, bool in1) {
    bf16x8 bp[1];
    float x[2][4];
    exponents<2>(x, st, bq, k);
    leave_out(x, in0, in1);
    float rs = probabilities<2>(bp, x);
    if (__ballot(rs > kMaxSum) != 0) {
        exponents<2>(x, st, bq, k);
        leave_out(x, in0, in1);
        rs = move_reference<2>(st, bp, x);
    }
    accumulate<2>(st, rs, bp, v);
}

// Operands out of the workgroup's LDS copy of shared blocks (4 KB per block: R tile of the keys, then T tile of the values).
__device__ __forceinline__ void load_keys_shared(KeyRegs<kGroup>& t, const bf16* blocks, int lane) {
#pragma unroll
    for (int j = 0; j < kGroup; j++) {
        t.k[j][0] = lds_ld16(blocks + j * 2 * kTile + lane * 8);
        t.k[j][1] = lds_ld16(blocks + j * 2 * kTile + 512 + lane * 8);
    }
}
__device__ __forceinline__ void load_values_shared(ValueRegs<kGroup>& t, const bf16* blocks, int lane) {
#pragma unroll
    for (int c = 0; c < kGroup / 2; c++)
#pragma unroll
        for (int dt = 0; dt < 4; dt++) {
            t.v[c][dt] = cat(lds_ld8(blocks + (2 * c) * 2 * kTile + kTile + dt * 256 + lane * 4),
                             lds_ld8(blocks + (2 * c + 1) * 2 * kTile + kTile + dt * 256 + lane * 4));
            __builtin_amdgcn_sched_barrier(0);    // (keeps the two reads one paired LDS read: paired with any other read they need moves)
        }
}
// The values of a pair of fine blocks out of the wave's own copy of their R tiles: the transposing read makes the T operands.
// (So the tokens' values need no T tile in memory, which would be a tenth of all that the pooling pass moves.)
__device__ __forceinline__ void load_values_fine(ValueRegs<2>& t, const bf16* tiles, int lane) {
#pragma unroll
    for (int dt = 0; dt < 4; dt++) t.v[0][dt] = cat(lds_t_operand(tiles, dt, lane), lds_t_operand(tiles + kTile, dt, lane));
}

__device__ __forceinline__ void load_values_fine_rows(ValueRegs<2>& t, const bf16* rows, int lane) {
#pragma unroll
    for (int dt = 0; dt < 4; dt++) t.v[0][dt] = cat(lds_t_operand_rows(rows, dt, lane), lds_t_operand_rows(rows + kTile, dt, lane));
}

// The query blocks' operands out of the rows of q, normalised and rotated here as the pooling pass does it (the sums over a row's chunks
// in its order): the same bits.
template <int Q>
struct QueryRows { bf16x8 x[Q][2], f[Q][2]; };
template <int Q>
__device__ __forceinline__ void request_queries(QueryRows<Q>& qr, const llsa_attn_fwd_args& a, int b, int h, int g, int lane) {
#pragma unroll
    for (int u = 0; u < Q; u++)
#pragma unroll
        for (int i = 0; i < 2; i++) {
            const int64_t tok = (g + u) * kBlk + 8 * i + (lane >> 3);
            qr.x[u][i] = ld16((const bf16*)a.q + b * a.sqb + h * a.sqh + tok * a.sqn + (lane & 7) * 8);
            if (a.freq_q != nullptr) qr.f[u][i] = ld16((const bf16*)a.freq_q + tok * kD + (lane & 7) * 8);
        }
}
template <int Q>
__device__ __forceinline__ void finish_queries(bf16x8 (&bq)[Q][2], const QueryRows<Q>& qr, const llsa_attn_fwd_args& a, int lane, bf16* place) {
#pragma unroll
    for (int u = 0; u < Q; u++) {
        rows_to_operand(bq[u], qr.x[u], place, lane);
        if (a.gamma_q != nullptr) {
            float ss[2];
#pragma unroll
            for (int i = 0; i < 2; i++) {
                ss[i] = 0.f;
#pragma unroll
                for (int e = 0; e < 8; e++) ss[i] += (float)bq[u][i][e] * (float)bq[u][i][e];
                ss[i] = quad_sum(ss[i]);
            }
            const float rstd = rsqrtf((ss[0] + ss[1]) * (1.f / kD) + a.eps_q);
#pragma unroll
            for (int i = 0; i < 2; i++)
#pragma unroll
                for (int e = 0; e < 8; e++) bq[u][i][e] = (bf16)((float)bq[u][i][e] * rstd * a.gamma_q[((lane >> 4) + 4 * i) * 8 + e]);
        }
        if (a.freq_q != nullptr) {
            bf16x8 f[2];
            rows_to_operand(f, qr.f[u], place + kTile, lane);
#pragma unroll
            for (int i = 0; i < 2; i++) bq[u][i] = rope_chunk_fwd(bq[u][i], f[i]);
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
    }
}

__device__ __forceinline__ void finish_query_block(const llsa_attn_fwd_args& a, const SoftmaxState& st, int bh, int b, int h, int g, int lane) {
    const int r = lane & 15, quad = lane >> 4;
    const float L = quad_sum(st.lsum);
    const float inv = 1.f / L;
    bf16x4 o[4];
#pragma unroll
    for (int dt = 0; dt < 4; dt++) o[dt] = cvt4(st.acc[dt] * inv);
    store_rows((bf16*)a.o + b * a.sob + h * a.soh + (int64_t)(g * kBlk + r) * a.son, o, quad, rows_wide(a.o, a.sob, a.soh, a.son));
    if (quad == 0 && a.lse != nullptr) a.lse[(int64_t)bh * a.N + g * kBlk + r] = (st.m2 + __builtin_amdgcn_logf(L)) * kLn2;
}

// One query block's selection among the 64 KEYS blocks of a one-level call, by its wave: the T best pooled keys, best first, as
// topk_dense_kernel finds them.  Result: entry i in lane i, through `scratch` (64 ints of LDS of the wave).
template <int KEYS>
__device__ __forceinline__ int select_blocks(const bf16* pq_row, const bf16* key_tiles, int T, int lane, int* scratch) {
    RankedKeys<KEYS> ranked = rank_keys<KEYS>(pq_row, key_tiles, lane * 8, 512 + lane * 8, 64 * KEYS, lane);
#pragma unroll
    for (int m = 0; m < KEYS; m++)
        if (ranked.rank[m] < T) scratch[ranked.rank[m]] = ranked.index(m, lane);
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    return scratch[min(lane, T - 1)];
}

// Q sibling query blocks per wave, 4 Q consecutive query blocks per workgroup.
//
// The pooled blocks -- the selected blocks of every pooled level below the coarsest and the coarsest level itself -- are
// the same for all query blocks of a 256-token group, hence for the four waves of the workgroup: they are fetched once
// per workgroup, kGroup at a time, straight into LDS (two buffers, the next fetch in flight during the arithmetic).
// The T fine blocks differ from query block to query block, but siblings have many in common (of 2 x 16 entries 24 are
// different on image-like inputs; four siblings per wave would fetch 34 of 64, but leave two long waves per SIMD: 83 against
// 62 us for 12 x 16384 tokens): the wave merges its lists (merge_lists) and walks the union, two blocks per step, every
// block fetched once and multiplied with the query blocks that selected it.  What bounds the fine part is the rate at which
// tiles arrive from the L2, and waves enough to keep the fetches in flight.
// The first `list_rows` rows of the grid make the index transposes of the backward (transpose_device.h): they need the selection
// and nothing else, and are latency for the most part, which the attention's workgroups fill.  In a launch of their own behind this
// one the chip waited for them: step of 12 x 16384 tokens 317 -> 309 us, of 24 x 4096 163 -> 156, of 48 x 16384 1284 -> 1264; both
// kernels of 6 x 65536 157 -> 154, where 67 workgroups a head (66 ranges and the histogram) read all its 65536 entries each.
// That reading is what bounds them on the largest grids: their workgroups then fill the chip by themselves for rounds, and a launch of their own, with
// twice the LDS and so half the ranges, reads less.  Steps behind the forward / riding, us, by entries read over all workgroups (two levels, topk 16/16): 12 x
// 16384 tokens 300.6 / 288.6;  24 x 16384 542.9 / 532.3;  6 x 32768 326 / 313;  65536 tokens, 2 heads 283.7 / 271.6;  6 647.6 / 642.0;  12 (53 M) 1287 / 1284;  16
// (70 M) 1699 / 1682;  20 (88 M) 2115 / 2105;  24 (105 M) 2522 / 2505;  28 (123 M) 2944 / 2950;  32 (141 M) 3315 / 3340;  64 x 32768, 32/16 (76 M) 3973 / 3987;  42 x 49152,
// 20/16 (98 M) 3432 / 3468;  one level, 24 x 49152 5184 / 5216.
constexpr int kTrLdsFwd = 2 * kGroup * 2 * kTile / 2 - 32;    // ints of the kernel's LDS they work in (32 for their scratch)
static_assert(tr_scratch_ints(256) <= 32, "the scratch of a transposing workgroup");
constexpr int64_t kRideMaxReads = (int64_t)88 << 20;          // entries the riding workgroups may read in all
constexpr int kGridRows = 65535;                              // rows a grid can have

// ROWS (no backward will follow): q and v are read as the caller's rows.  Their tiles are then not written, which is a third of all that the pooling pass
// moves; every block of v is still copied into LDS in two loads of whole lines.  8 x 65536 tokens, topk 8:
// pooling 68.7 -> 45.2 us, forward 559 -> 570.
// SELECT (no backward either; 64 SELECT blocks of one level, attn_fwd_selects): a wave selects its own blocks, and the selection's launch goes.
template <int Q, int R, bool ROWS, int SELECT = 0>
__global__ __launch_bounds__(256, Q == 1 ? 4 : 3) void attn_fwd_kernel(llsa_attn_fwd_args a, TrJobs lists, int list_rows) {
    __shared__ __align__(16) bf16 sh[2][kGroup][2 * kTile];
    __shared__ int order[4][R * kWave];
    if (!ROWS && SELECT == 0 && (int)blockIdx.y < list_rows) {
        const int block = (int)(blockIdx.y * gridDim.x + blockIdx.x);
        int* const lds = reinterpret_cast<int*>(&sh[0][0][0]);
        if (block < lists.wgs * ((int)gridDim.y - list_rows)) transpose_block<256>(lists, block, lds, lds + kTrLdsFwd);
        return;
    }
    const int lane = threadIdx.x & 63, unit = r_unit(lane);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int N1 = a.N / kBlk, T = a.T;
    const int lid = xcd_logical_id(list_rows);
    const int g = (lid % (int)gridDim.x) * (4 * Q) + Q * wave;        // query blocks g .. g + Q - 1 (the host checks N1 % 4 Q == 0)
    const int bh = lid / (int)gridDim.x, b = bh / a.H, h = bh % a.H;

    const bf16* kr = (const bf16*)a.kr + (int64_t)bh * N1 * kTile;
    const bf16* vr = ROWS ? (const bf16*)a.v + b * a.svb + h * a.svh + (lane >> 3) * a.svn + row_piece(lane) : (const bf16*)a.vt + (int64_t)bh * N1 * kTile + unit;
    const int64_t v_block = ROWS ? kBlk * a.svn : kTile;
    SharedList sl = shared_list(a.lvl, a.levels, a.N, bh, g, lane);
    bf16* const sh0 = &sh[0][0][0];
    auto issue_group = [&](int grp) __attribute__((always_inline)) {   // this wave brings in block kGroup*grp + wave
        const SharedTiles sb = shared_tiles(sl, a.lvl, bh, kGroup * grp + wave);
        bf16* dst = sh0 + ((grp & 1) * kGroup + wave) * (2 * kTile);
        copy16_global_to_lds(sb.k + lane * 8, dst);
        copy16_global_to_lds<512>(sb.k + lane * 8, dst);
        copy16_global_to_lds(sb.v + lane * 8, dst + kTile);
        copy16_global_to_lds<512>(sb.v + lane * 8, dst + kTile);
    };
    const int n_groups = sl.n_blocks / kGroup;                // every level's count is a multiple of kGroup (host checks)
    QueryRows<Q> rows;
    if constexpr (ROWS) request_queries<Q>(rows, a, b, h, g, lane);
    issue_group(0);
    const int* ip = SELECT > 0 ? nullptr : a.idx + ((int64_t)bh * N1 + g) * T;
    MergedLists<Q, R> ml;
    if constexpr (SELECT > 0) {
        static_assert(Q == 1 && R == 1, "a row of its own per wave");
        ml.packed[0] = select_blocks<SELECT>((const bf16*)a.pq + ((int64_t)bh * N1 + g) * kD, (const bf16*)a.lvl[0].kr + (int64_t)bh * N1 * kD, T, lane, order[wave]) |
                       (1 << kSetShift);
        ml.n = T;
    } else {
        ml = merge_lists<Q, R>(ip, min(T, kWave * R / Q), N1, lane, order[wave]);
    }

    bf16x8 bq[Q][2];               // 1/sqrt(64) is a power of two: scaling q before the product (as the
    SoftmaxState st[Q];            // reference does) equals scaling the fp32 scores, done in the exponent
    if constexpr (ROWS) {
        finish_queries<Q>(bq, rows, a, lane, &sh[1][wave][0]);          // (the second buffer is not filled before the barrier of group 0)
    } else {
#pragma unroll
        for (int u = 0; u < Q; u++) {
            const bf16* qp = (const bf16*)a.qr + ((int64_t)bh * N1 + g + u) * kTile + lane * 8;
            bq[u][0] = ld16(qp);
            bq[u][1] = ld16(qp + 512);
        }
    }
#pragma unroll
    for (int u = 0; u < Q; u++) init_state(st[u]);
    // ---- shared blocks, out of LDS.  The barrier at the top of round grp says two things: every
    // wave's part of group grp has landed, and every wave is done reading the other buffer
    // (group grp - 1), which the next fetch overwrites.  (LDS reads of a group come before the next fetch: the compiler
    // makes every LDS read wait for all copies into LDS that were issued before it.)
    SharedWeight sw = first_weight(a.lvl, a.levels);
    for (int grp = 0; grp < n_groups; grp++) {
        wait_vm0();
        __syncthreads();
        if (grp == sw.next) {
            const float w = sw.w;
            next_weight(sw, a.lvl, a.levels);
#pragma unroll
            for (int u = 0; u < Q; u++) rescale(st[u], w / sw.w);
        }
        const bf16* blk = &sh[grp & 1][0][0];
        if (grp == 0) {
            const bf16x8 k0 = lds_ld16(blk + lane * 8), k1 = lds_ld16(blk + 512 + lane * 8);
#pragma unroll
            for (int u = 0; u < Q; u++) start_reference(st[u], bq[u], k0, k1);
        }
        // All four blocks are one step: one test for the rare path, and the keys' registers are free before the values are used.
        // On long walks (8 x 65536 tokens, topk 8, 256 pooled blocks) the vector ALU is busy 57 % of the time and the matrix
        // cores 37 %, and the instructions per score count: without the maximum, and with one test per four blocks, that forward
        // call went from 850 to 805 us.
        bf16x8 bp[Q][kGroup / 2];
        float rs[Q], most = 0.f;
        ValueRegs<kGroup> v;
        {
            KeyRegs<kGroup> k;
            load_keys_shared(k, blk, lane);
            load_values_shared(v, blk, lane);
            if (grp + 1 < n_groups) issue_group(grp + 1);
#pragma unroll
            for (int u = 0; u < Q; u++) {
                float x[kGroup][4];
                exponents<kGroup>(x, st[u], bq[u], k);
                rs[u] = probabilities<kGroup>(bp[u], x);
                most = fmaxf(most, rs[u]);
            }
        }
        if (__ballot(most > kMaxSum) != 0) {                  // (reads the keys once more rather than keep them for this)
            asm volatile("" ::: "memory");
            KeyRegs<kGroup> k;
            load_keys_shared(k, blk, lane);
#pragma unroll
            for (int u = 0; u < Q; u++) {
                float x[kGroup][4];
                exponents<kGroup>(x, st[u], bq[u], k);
                rs[u] = move_reference<kGroup>(st[u], bp[u], x);
            }
        }
#pragma unroll
        for (int u = 0; u < Q; u++) accumulate<kGroup>(st[u], rs[u], bp[u], v);
    }
#pragma unroll
    for (int u = 0; u < Q; u++) rescale(st[u], sw.w);         // fine tokens weigh 1
    __syncthreads();                                          // the shared copy is dead: its LDS becomes private slots

    // ---- fine blocks, two per step: the keys of step s + 1 are loaded into registers and its values copied into the wave's other
    // LDS slot while step s is worked on.  (The LDS reads of a step come before the next fetch, see above; the products with
    // the keys do not wait for them.)  Nothing may be in flight when the wave ends (a copy landing in LDS that already
    // belongs to another workgroup), so the last step fetches nothing.
    bf16* const slots = sh0 + wave * (4 * kTile);             // two slots of the V tiles of two blocks
    auto fine = [&]() __attribute__((always_inline)) {
        const int n_steps = (ml.n + 1) / 2;
        auto fetch = [&](int s, KeyRegs<2>& dst) __attribute__((always_inline)) {
            bf16* slot = slots + (s & 1) * (2 * kTile);
#pragma unroll
            for (int j = 0; j < 2; j++) {
                const int64_t blk = ml.block(min(2 * s + j, ml.n - 1));
                const bf16 *kb = kr + blk * kTile, *vb = vr + blk * v_block;
                dst.k[j][0] = ld16(kb + lane * 8);
                dst.k[j][1] = ld16(kb + lane * 8 + 512);
                copy16_global_to_lds(vb, slot + j * kTile);
                if constexpr (ROWS) copy16_global_to_lds(vb + 8 * a.svn, slot + j * kTile + 512);
                else copy16_global_to_lds<512>(vb, slot + j * kTile);
            }
        };
        auto work = [&](int s, KeyRegs<2>& cur, KeyRegs<2>& nxt) __attribute__((always_inline)) {
            const unsigned m0 = ml.rows(2 * s), m1 = 2 * s + 1 < ml.n ? ml.rows(2 * s + 1) : 0u;
            wait_vm0();
            ValueRegs<2> v;
            if constexpr (ROWS) load_values_fine_rows(v, slots + (s & 1) * (2 * kTile), lane);
            else load_values_fine(v, slots + (s & 1) * (2 * kTile), lane);
            if (s + 1 < n_steps) fetch(s + 1, nxt);
            if ((m0 & m1) == (1u << Q) - 1u) {
                compute_step<Q>(st, bq, cur, v);
            } else {
#pragma unroll
                for (int u = 0; u < Q; u++) {
                    const bool in0 = (m0 >> u) & 1u, in1 = (m1 >> u) & 1u;
                    if (in0 || in1) compute_step(st[u], bq[u], cur, v, in0, in1);
                }
            }
        };
        KeyRegs<2> ra, rb;
        fetch(0, ra);
        for (int s = 0; s < n_steps; s += 2) {
            work(s, ra, rb);
            if (s + 1 < n_steps) work(s + 1, rb, ra);
        }
    };
    fine();
    if constexpr (Q == 1 && SELECT == 0) {                        // longer lists: 64 entries at a time
        for (int c0 = kWave * R; c0 < T; c0 += kWave * R) {
            ml = merge_lists<Q, R>(ip + c0, min(T - c0, kWave * R), N1, lane, order[wave]);
            fine();
        }
    }
#pragma unroll
    for (int u = 0; u < Q; u++) finish_query_block(a, st[u], bh, b, h, g + u, lane);
}

}  // namespace llsa

using namespace llsa;

// Rows of a grid of `width` workgroups that the index transposes take in front of the attention's, or -1: launches of their own
static int64_t plan_list_rows(const llsa_transpose_job* jobs, int n_jobs, int B, int H, int width, TrJobs& lists) {
    if (!plan_transpose(jobs, n_jobs, B, H, kTrLdsFwd, lists)) return -1;
    const int64_t BH = (int64_t)B * H, rows = (lists.wgs * BH + width - 1) / width;
    int64_t reads = 0;
    for (int i = 0; i < lists.n_jobs; i++) reads += (lists.job[i].parts + 1) * BH * lists.job[i].Mb * lists.job[i].T;
    return reads > kRideMaxReads || BH + rows > kGridRows ? -1 : rows;
}
static int forward_width(int N, bool pairs) { return N / (pairs ? 128 : 64); }   // workgroups of a (b,h); a multiple of 8: N is one of 1024

// Whether the forward selects by itself where no backward follows.  A wave ranks 64 keys in 0.4 us and 128 in 1.2, which waves in the same SIMD add up
// to, where the launch it saves takes 6 to 10 and its gap.  A pass, us, launch of its own / in the forward:
//   1024 tokens, topk 8: 6 heads 18.7 / 14.9;  24 25.6 / 22.3;  96 38.8 / 35.3;  128 44.4 / 41.4;  topk 64: 6 34.6 / 24.9;  128 107 / 95
//   2048 tokens, topk 8: 1 head 18.6 / 16.8;  6 20.9 / 18.5;  24 30.6 / 29.7;  48 40.2 / 40.8;  64 45.8 / 48.5;  topk 32: 6 26.6 / 23.0;  64 70.9 / 69.2
//   3072 and 4096 tokens, 192 and 256 keys, topk 8: 1 head 20.4 / 21.8 and 21.3 / 25.7
static bool attn_fwd_selects(int64_t BH, int N, int T, int levels) {
    const int32_t topk[1] = {T};
    if (levels != 1 || (N != 1024 && N != 2048) || T < 4 || T > 64 || T % 4 != 0 || two_blocks_per_wave(BH, N, topk, 1, true)) return false;
    return BH * (N / kBlk) <= (N == 1024 || T >= 32 ? 8192 : 3072);
}

// jobs: the index transposes that ride along, or nullptr
static int attn_fwd(const llsa_attn_fwd_args* a, const llsa_transpose_job* jobs, int n_jobs, void* stream) {
    LLSA_REQUIRE(a != nullptr, "attn_fwd: null args");
    LLSA_REQUIRE(a->levels >= 1 && a->levels <= LLSA_MAX_LEVELS, "attn_fwd: levels must be 1..%d", LLSA_MAX_LEVELS);
    LLSA_REQUIRE(a->B > 0 && a->H > 0 && a->N > 0, "attn_fwd: bad B/H/N");
    const bool rows_form = a->q != nullptr, selects = a->pq != nullptr;
    LLSA_REQUIRE(a->kr && (a->idx || selects) && a->o && (rows_form ? a->v != nullptr : a->qr && a->vt && a->lse), "attn_fwd: null tensor");
    LLSA_REQUIRE(!rows_form || jobs == nullptr, "attn_fwd: no index transposes beside a forward on rows");
    if (rows_form) {
        LLSA_REQUIRE(aligned16(a->q) && aligned16(a->v) && aligned16(a->freq_q), "attn_fwd: tensors must be 16-byte aligned");
        for (const int64_t st : {a->sqb, a->sqh, a->sqn, a->svb, a->svh, a->svn}) LLSA_REQUIRE(stride_ok(st), "attn_fwd: rows must be 16-byte aligned");
        LLSA_REQUIRE(a->gamma_q == nullptr || a->eps_q >= 0.f, "attn_fwd: eps must be >= 0");
    }
    LLSA_REQUIRE(!selects || (aligned16(a->pq) && !rows_form && jobs == nullptr && attn_fwd_selects((int64_t)a->B * a->H, a->N, a->T, a->levels)),
                 "attn_fwd: these sizes are not selected in the forward");
    LLSA_REQUIRE(a->T >= 4 && a->T % 4 == 0 && a->T <= a->N / 16, "attn_fwd: topk=%d must be a multiple of 4 and <= N/16", a->T);
    const int64_t mult = coarsest_multiple(a->levels);
    LLSA_REQUIRE(a->N % mult == 0,
                 "attn_fwd: %d level(s) need N %% %lld == 0 (N=%d): the coarsest level is walked in 64-token tiles of its N/16^levels pooled tokens",
                 a->levels, (long long)mult, a->N);
    int listed = 0;
    int32_t topk[LLSA_MAX_LEVELS] = {a->T};
    int64_t span = 256;                                       // tokens under one block of level l
    for (int l = 1; l <= a->levels; l++, span *= 16) {
        const llsa_fwd_level& lv = a->lvl[l - 1];
        LLSA_REQUIRE(lv.kr && lv.vt && aligned16(lv.kr) && aligned16(lv.vt), "attn_fwd: tiles of level %d missing or not 16-byte aligned", l);
        LLSA_REQUIRE(lv.w > 0.f, "attn_fwd: the weight of level %d must be > 0", l);
        if (l < a->levels) {
            LLSA_REQUIRE(lv.sel != nullptr, "attn_fwd: selection of level %d missing", l);
            LLSA_REQUIRE(lv.T >= 4 && lv.T % 4 == 0 && lv.T <= a->N / span, "attn_fwd: topk of level %d (%d) must be a multiple of 4 and <= N/%lld",
                         l, lv.T, (long long)span);
            listed += lv.T;
            topk[l] = lv.T;
        }
    }
    LLSA_REQUIRE(listed <= LLSA_POOLED_TOPK_MAX, "attn_fwd: the topk of the pooled levels together (%d) must not exceed %d", listed,
                 LLSA_POOLED_TOPK_MAX);
    LLSA_REQUIRE(aligned16(a->qr) && aligned16(a->kr) && aligned16(a->vt) && aligned16(a->o), "attn_fwd: tensors must be 16-byte aligned");
    LLSA_REQUIRE((a->sob % 4 == 0) && (a->soh % 4 == 0) && (a->son % 4 == 0), "attn_fwd: rows of o must be 8-byte aligned");
    const int BH = a->B * a->H;
    // Two query blocks per wave halve the LDS reads of the pooled blocks and save a quarter of the fine fetches; one per wave
    // leaves more and shorter waves.  Two win where the pooled blocks are most of the walk (11 x 32768 tokens, topk 8,
    // 128 pooled blocks: 227 against 267 us) and on large grids (16 x 16384, topk 16: 78.2 against 83.7; 48 x 16384: 228 against 271; 6 x
    // 262144: 929 against 1057), one on smaller ones (12 x 16384: 58.5 against 64.6; 24 x 4096: 30.1 against 31.2; 3 x 49152 at topk 64
    // even) and where the last round would be mostly empty (see pairs_pay).
    const bool pairs = two_blocks_per_wave(BH, a->N, topk, a->levels, true);
    TrJobs lists{};
    const int width = forward_width(a->N, pairs);
    const int64_t list_rows = jobs != nullptr ? plan_list_rows(jobs, n_jobs, a->B, a->H, width, lists) : -1;
    const bool ride = list_rows >= 0;
    const int rows = ride ? (int)list_rows : 0;
    const dim3 grid(width, BH + rows);
    const hipStream_t st = (hipStream_t)stream;
#define LLSA_FWD(Q, R)                                                                                                                    \
    do {                                                                                                                                  \
        if (rows_form) hipLaunchKernelGGL(HIP_KERNEL_NAME(attn_fwd_kernel<Q, R, true>), grid, dim3(256), 0, st, *a, lists, rows);         \
        else hipLaunchKernelGGL(HIP_KERNEL_NAME(attn_fwd_kernel<Q, R, false>), grid, dim3(256), 0, st, *a, lists, rows);                  \
    } while (0)
    if (selects && a->N == 1024) hipLaunchKernelGGL(HIP_KERNEL_NAME(attn_fwd_kernel<1, 1, false, 1>), grid, dim3(256), 0, st, *a, lists, rows);
    else if (selects) hipLaunchKernelGGL(HIP_KERNEL_NAME(attn_fwd_kernel<1, 1, false, 2>), grid, dim3(256), 0, st, *a, lists, rows);
    else if (!pairs) LLSA_FWD(1, 1);
    else if (a->T <= 32) LLSA_FWD(2, 1);
    else LLSA_FWD(2, 2);
#undef LLSA_FWD
    const int rc = launch_status("attn_fwd");
    if (rc != 0 || jobs == nullptr || ride) return rc;
    return llsa_transpose_indices_multi(jobs, n_jobs, a->B, a->H, stream);
}

static int check_plan_query(const char* what, int B, int H, int N, const int32_t* topk, int levels) {
    LLSA_REQUIRE(topk != nullptr && levels >= 1 && levels <= LLSA_MAX_LEVELS, "%s: levels must be 1..%d", what, LLSA_MAX_LEVELS);
    LLSA_REQUIRE(B > 0 && H > 0 && N > 0 && N % coarsest_multiple(levels) == 0, "%s: bad B/H/N", what);
    for (int l = 0; l < levels; l++) LLSA_REQUIRE(topk[l] > 0, "%s: topk must be > 0", what);
    return 0;
}

extern "C" int llsa_query_blocks_per_wave(int B, int H, int N, const int32_t* topk, int levels, int backward) {
    if (const int rc = check_plan_query("query_blocks_per_wave", B, H, N, topk, levels)) return rc;
    return two_blocks_per_wave((int64_t)B * H, N, topk, levels, backward == 0) ? 2 : 1;
}

extern "C" int llsa_attn_fwd_selects(int B, int H, int N, int T, int levels) {
    return B > 0 && H > 0 && N > 0 && attn_fwd_selects((int64_t)B * H, N, T, levels);
}

extern "C" int llsa_lists_ride(int B, int H, int N, const int32_t* topk, int levels) {
    if (const int rc = check_plan_query("lists_ride", B, H, N, topk, levels)) return rc;
    llsa_transpose_job jobs[LLSA_MAX_LEVELS];
    int32_t* const some = reinterpret_cast<int32_t*>(16);     // (the plan only looks whether there are lists and inverse positions: of the pooled levels there are)
    for (int l = 0, m = N / 16; l < levels; l++, m /= 16)
        jobs[l] = llsa_transpose_job{some, some, some, nullptr, l == 0 ? nullptr : some, m, m, topk[l], 1, nullptr};
    TrJobs lists{};
    return plan_list_rows(jobs, levels, B, H, forward_width(N, two_blocks_per_wave((int64_t)B * H, N, topk, levels, true)), lists) >= 0;
}

extern "C" int llsa_attn_fwd(const llsa_attn_fwd_args* a, void* stream) { return attn_fwd(a, nullptr, 0, stream); }

extern "C" int llsa_attn_fwd_lists(const llsa_attn_fwd_args* a, const llsa_transpose_job* jobs, int n_jobs, void* stream) {
    LLSA_REQUIRE(jobs != nullptr && n_jobs >= 1 && n_jobs <= LLSA_MAX_LEVELS, "attn_fwd_lists: 1..%d jobs, got %d", LLSA_MAX_LEVELS, n_jobs);
    return attn_fwd(a, jobs, n_jobs, stream);
}
