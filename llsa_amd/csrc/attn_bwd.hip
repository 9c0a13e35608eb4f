// Backward of the block-sparse attention: delta pre-pass, dQ per query block, and the
// K-side gradients (dK/dV of the fine tokens through the transposed index, the sparse
// level-1 pooled gradients of llsa_l2, and the dense coarsest pooled gradients).
//
// MFMA orientations (bf16 16x16x32, see llsa_device.h for the register layout):
//   dQ pass, per key block (keys on M, queries on N, like the forward):
//       S^T  = K . Q^T          dP^T = V . dO^T          dS^T = P^T o (dP^T - delta)
//       dQ^T (64 ch x 16 q) += K_blk^T (64 x 32 keys) . dS^T      A = block-transposed K
//   K-side pass, per key block and per pair of query blocks (queries on M, keys on N):
//       S    = Q . K^T          dP   = dO . V^T          dS   = P o (dP - delta)
//       dV^T (64 ch x 16 keys) += dO_blk^T (64 x 32 q) . P        A = block-transposed dO
//       dK^T (64 ch x 16 keys) += Q_blk^T  (64 x 32 q) . dS       A = block-transposed Q
// In both passes the score tile leaves the MFMA in exactly the operand layout the next
// product needs, so P and dS go from registers to registers.
#include "llsa_device.h"
#include "llsa_host.h"
#include "../../include/llsa_hip.h"
#include <algorithm>

namespace llsa {

// ---------------------------------------------------------------------------------------
// dQ: Q query blocks per wave, 4 Q consecutive query blocks per workgroup, key blocks taken
// two at a time (32 keys = one MFMA K step).
//
// K and V always reach the MFMA from R tiles.  K is needed twice: as the A operand of S^T (a plain
// 16-byte read per lane) and, read back with the transposing LDS load, as the A operand of
// dQ^T += K^T.dS^T -- so K goes through LDS in any case, copied there straight from global memory.
//  * pooled blocks (level-1 pooled tokens of the parent's coarse blocks, the coarsest level) are
//    the same for all query blocks of the workgroup: one copy per workgroup, kGroup blocks
//    of K and V at a time, two buffers;
//  * fine blocks are private: afterwards each wave re-uses a quarter of the same LDS as two slots
//    for the K tiles of a pair (the copy of pair t+1 in flight during pair t), V stays in registers.
// ---------------------------------------------------------------------------------------
struct PairR {
    bf16x8 k[2][2], v[2][2];       // block j, channel half
};
struct PairT {
    bf16x4 t[2][4];                // block j, channel tile dt
};

__device__ __forceinline__ void read_k_r(PairR& o, const bf16* k0, const bf16* k1, int lane) {
    o.k[0][0] = lds_ld16(k0 + r_unit(lane));
    o.k[0][1] = lds_ld16(k0 + 512 + r_unit(lane));
    o.k[1][0] = lds_ld16(k1 + r_unit(lane));
    o.k[1][1] = lds_ld16(k1 + 512 + r_unit(lane));
}
__device__ __forceinline__ void read_v_r(PairR& o, const bf16* v0, const bf16* v1, int lane) {
    o.v[0][0] = lds_ld16(v0 + r_unit(lane));
    o.v[0][1] = lds_ld16(v0 + 512 + r_unit(lane));
    o.v[1][0] = lds_ld16(v1 + r_unit(lane));
    o.v[1][1] = lds_ld16(v1 + 512 + r_unit(lane));
}
__device__ __forceinline__ void read_k_t(PairT& o, const bf16* k0, const bf16* k1, int lane) {
#pragma unroll
    for (int dt = 0; dt < 4; dt++) {
        o.t[0][dt] = lds_t_operand(k0, dt, lane);
        o.t[1][dt] = lds_t_operand(k1, dt, lane);
    }
}
// dS^T of a pair of key blocks, as the B operand of the dQ product
// (nlse2w: log2 of the segment's weight minus the query's log-sum-exp, log2 units: the weight rides in the exponent; ndl:
// -delta in all four places, what the product dP starts from, which saves a subtraction per score)
__device__ __forceinline__ bf16x8 dq_scores(const PairR& p, const bf16x8 bq[2], const bf16x8 bdo[2], float nlse2w,
                                            const f32x4& ndl) {
    bf16x8 bds;
#pragma unroll
    for (int j = 0; j < 2; j++) {
        f32x4 s = {0.f, 0.f, 0.f, 0.f}, dp = ndl;
        s = mfma_bf16(p.k[j][0], bq[0], s);
        s = mfma_bf16(p.k[j][1], bq[1], s);
        dp = mfma_bf16(p.v[j][0], bdo[0], dp);
        dp = mfma_bf16(p.v[j][1], bdo[1], dp);
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const float pe = exp2_fast(fmaf(s[e], kScaleLog2e, nlse2w));
            bds[j * 4 + e] = (bf16)(pe * dp[e]);
        }
    }
    return bds;
}
__device__ __forceinline__ void dq_accum(f32x4 dq[4], const PairT& p, bf16x8 bds) {
#pragma unroll
    for (int dt = 0; dt < 4; dt++) dq[dt] = mfma_bf16(cat(p.t[0][dt], p.t[1][dt]), bds, dq[dt]);
}

// A gradient block (16 tokens x 64 channels, one lane: channels 16 dt + 4 (l/16) ..+3 of token l%16) back through the RMS norm of
// its rows x, as rmsnorm_bwd_kernel does it: with xn = x rstd and g = dy gamma, dx = rstd (g - xn mean(g xn)).  contrib: dy xn,
// added up for the weights' gradient.  x: the lane's channels of its token; gamma: its channels' weights.
// Inside the kernels that write dq and dk because a pass of its own is bound by memory: it reads the finished gradient and x and
// writes the gradient again (300 MB for q and k of 8 x 6 x 16384 tokens, plus four launches).  Here x is all that is read, by
// waves that have their arithmetic still to do: 1368 -> 1298 us for that step, 215 -> 200 us at 4 x 6 x 4096.
__device__ __forceinline__ void norm_back(bf16x4 (&dy)[4], const bf16x4 (&x)[4], const f32x4 (&gamma)[4], float eps, float (&contrib)[16]) {
    float ss = 0.f;
#pragma unroll
    for (int dt = 0; dt < 4; dt++)
#pragma unroll
        for (int e = 0; e < 4; e++) ss += (float)x[dt][e] * (float)x[dt][e];
    const float rstd = rsqrtf(quad_sum(ss) * (1.f / kD) + eps);
    float dot = 0.f;
#pragma unroll
    for (int dt = 0; dt < 4; dt++)
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const float xn = (float)x[dt][e] * rstd, g = (float)dy[dt][e];
            dot += g * gamma[dt][e] * xn;
            contrib[dt * 4 + e] += g * xn;
        }
    dot = quad_sum(dot) * (1.f / kD);
#pragma unroll
    for (int dt = 0; dt < 4; dt++)
#pragma unroll
        for (int e = 0; e < 4; e++)
            dy[dt][e] = (bf16)(rstd * ((float)dy[dt][e] * gamma[dt][e] - (float)x[dt][e] * rstd * dot));
}
__device__ __forceinline__ void norm_gamma(f32x4 (&gamma)[4], const llsa_norm_back& nb, int quad) {
#pragma unroll
    for (int dt = 0; dt < 4; dt++)
#pragma unroll
        for (int e = 0; e < 4; e++) gamma[dt][e] = nb.gamma[dt * 16 + quad * 4 + e];
}
__device__ __forceinline__ void norm_load(bf16x4 (&x)[4], f32x4 (&gamma)[4], const llsa_norm_back& nb, int b, int h, int tok, int quad) {
    load_rows(x, (const bf16*)nb.x + b * nb.sxb + h * nb.sxh + (int64_t)tok * nb.sxn, quad);
    norm_gamma(gamma, nb, quad);
}
// Sum of the sixteen contrib[] over the sixteen tokens of a quad, by exchanging halves: lane l ends with the sum for
// channel 16 (i/4) + 4 (l/16) + i%4, i = the lane's low four bits.  (Exchanges with i^8, i^7, i^2 and i^1 reach all sixteen.  With moves inside the
// vector instructions instead of fifteen shuffles, and dQ's rows requested together, the training step of 48 x 16384 tokens with the norm 1197 -> 1186 us.)
__device__ __forceinline__ float norm_contrib_sum(const float (&contrib)[16], int lane, int& channel) {
    float a8[8], a4[4], a2[2];
    const bool b3 = lane & 8, b2 = lane & 4, b1 = lane & 2, b0 = lane & 1;
#pragma unroll
    for (int i = 0; i < 8; i++) a8[i] = (b3 ? contrib[8 + i] : contrib[i]) + across<8>(b3 ? contrib[i] : contrib[8 + i]);
#pragma unroll
    for (int i = 0; i < 4; i++) a4[i] = (b2 ? a8[4 + i] : a8[i]) + across<7>(b2 ? a8[i] : a8[4 + i]);
#pragma unroll
    for (int i = 0; i < 2; i++) a2[i] = (b1 ? a4[2 + i] : a4[i]) + across<2>(b1 ? a4[i] : a4[2 + i]);
    const float s = (b0 ? a2[1] : a2[0]) + across<1>(b0 ? a2[0] : a2[1]);
    const int i = lane & 15;
    channel = 16 * (i >> 2) + 4 * (lane >> 4) + (i & 3);
    return s;
}

// What the K-side kernels need of a query block besides its tiles, as their products take it: minus the log-sum-exp (log2
// units) of its 16 queries, then minus their deltas, one 128-byte line per block.
// (The products dP start from minus delta and the exponent is one multiply-add: no subtraction per score, no product per query
// and pass.  The vector ALU is busy 37 % of the time in the dense K side and 50 % in the dQ kernel at 6 x 262144 tokens; with
// the forward's soft-max without a maximum that step went from 4404 to 4263 us, of 12 x 16384 337 -> 330.)
constexpr int kStats = 2 * kBlk;

// What a wave keeps per query block
struct DqSide {
    bf16x8 bq[2], bdo[2];          // R operands of q and dO
    float nlse2;                   // -log-sum-exp (log2 units) of query l%16
    f32x4 ndl;                     // -delta of query l%16, four times
    f32x4 dq[4];                   // dQ^T: channel 16*dt + 4*(l/16) + e of query l%16
};

// dO comes straight from the caller's tensor, as R operand (lane l: row l%16, channels 8*(l/16)..+7 and
// 32 + 8*(l/16)..+7).  The wave also does the pre-pass the K-side kernels need: delta = rowsum(O * dO) in fp32 (the reference sums in the
// tensor dtype, sparse_attention_res_1.py:153-177) and dO as an R tile.
// The rows of dO and O arrive whole and change into the operand layout through LDS (rows_to_operand; `place`: 2 KB of the wave's own for each).
// With the normalised rows and rotations of the epilogues in 16-byte pieces (load_rows) 12 x 16384 tokens 74.4 -> 70.0 us, 48 x 16384 with the
// qk norm 335.6 -> 310.4 and its K side 306.5 -> 301.5, 24 x 4096 33.5 -> 31.2, 15 x 7168 44.3 -> 42.3, 6 x 1024 8.2 -> 7.3; 3 x 49152 at topk 64 even.
struct DqRows { bf16x8 g[2], o[2]; };
__device__ __forceinline__ void dq_request(DqRows& rows, const llsa_attn_bwd_args& a, int b, int h, int g, int lane) {
#pragma unroll
    for (int i = 0; i < 2; i++) {
        const int64_t tok = g * kBlk + 8 * i + (lane >> 3);
        rows.g[i] = ld16((const bf16*)a.dout + b * a.sdob + h * a.sdoh + tok * a.sdon + (lane & 7) * 8);
        rows.o[i] = ld16((const bf16*)a.o + b * a.sob + h * a.soh + tok * a.son + (lane & 7) * 8);
    }
}
__device__ __forceinline__ void dq_begin(DqSide& sd, const DqRows& rows, const llsa_attn_bwd_args& a, float* __restrict__ stats, bf16* __restrict__ dor,
                                         int bh, int g, int lane, bf16* place) {
    const int N1 = a.N / kBlk, r = lane & 15, quad = lane >> 4, tok = g * kBlk + r;
    const bf16* qp = (const bf16*)a.qr + ((int64_t)bh * N1 + g) * kTile + lane * 8;
    sd.bq[0] = ld16(qp);
    sd.bq[1] = ld16(qp + 512);
    bf16x8 o[2];
    rows_to_operand(sd.bdo, rows.g, place, lane);
    rows_to_operand(o, rows.o, place + kTile, lane);
    float acc = 0.f;
#pragma unroll
    for (int e = 0; e < 8; e++) acc += (float)o[0][e] * (float)sd.bdo[0][e];
#pragma unroll
    for (int e = 0; e < 8; e++) acc += (float)o[1][e] * (float)sd.bdo[1][e];
    const float ndl = -quad_sum(acc);
    sd.ndl = f32x4{ndl, ndl, ndl, ndl};
    bf16* tile = dor + ((int64_t)bh * N1 + g) * kTile + lane * 8;
    st16(tile, sd.bdo[0]);
    st16(tile + 512, sd.bdo[1]);
    sd.nlse2 = -a.lse[(int64_t)bh * a.N + tok] * kLog2e;
    if (quad < 2) stats[((int64_t)bh * N1 + g) * kStats + lane] = quad == 0 ? sd.nlse2 : ndl;
#pragma unroll
    for (int dt = 0; dt < 4; dt++) sd.dq[dt] = f32x4{0.f, 0.f, 0.f, 0.f};
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}
// x, f: rows of the norm's input and of the rotation's entries, as request_rows leaves them
template <bool NORM>
__device__ __forceinline__ void dq_end(const DqSide& sd, const llsa_attn_bwd_args& a, int b, int h, int g, int lane, const bf16x8 (&x_raw)[2],
                                       const bf16x8 (&f_raw)[2], const f32x4 (&gamma)[4], float (&contrib)[16]) {
    const int r = lane & 15, quad = lane >> 4, tok = g * kBlk + r;
    bf16x4 o[4];
#pragma unroll
    for (int dt = 0; dt < 4; dt++) o[dt] = cvt4(sd.dq[dt] * kScale);
    if (a.freq_dq != nullptr) {                               // rotate the gradient back
        bf16x4 f[4];
        arrange_rows(f, f_raw);
#pragma unroll
        for (int dt = 0; dt < 4; dt++) o[dt] = rope_bwd4(o[dt], f[dt]);
    }
    if (NORM) {
        bf16x4 x[4];
        arrange_rows(x, x_raw);
        norm_back(o, x, gamma, a.norm_q.eps, contrib);
    }
    store_rows((bf16*)a.dq + b * a.sdqb + h * a.sdqh + (int64_t)tok * a.sdqn, o, quad, rows_wide(a.dq, a.sdqb, a.sdqh, a.sdqn));
}
__device__ __forceinline__ void dq_pair_of_blocks(DqSide& sd, const PairR& r, const PairT& t, float log2w) {
    dq_accum(sd.dq, t, dq_scores(r, sd.bq, sd.bdo, sd.nlse2 + log2w, sd.ndl));
}
// in0, in1 (wave-uniform): whether the query block reads the pair's first / second block.  What it does not read is cleared by one AND
// per two values: selects of 16-bit values cost 18 vector instructions beside the 28 of the arithmetic (dQ at 24 x 4096 tokens, topk 16:
// 35.1 -> 33.9 us, 12 x 16384: 83 -> 79 in the step).
__device__ __forceinline__ void dq_pair_of_blocks(DqSide& sd, const PairR& r, const PairT& t, bool in0, bool in1) {
    u32x4 ds = __builtin_bit_cast(u32x4, dq_scores(r, sd.bq, sd.bdo, sd.nlse2, sd.ndl));
    const unsigned keep0 = in0 ? ~0u : 0u, keep1 = in1 ? ~0u : 0u;
    ds &= u32x4{keep0, keep0, keep1, keep1};
    dq_accum(sd.dq, t, __builtin_bit_cast(bf16x8, ds));
}

// Q sibling query blocks per wave (see attn_fwd_kernel): the pooled blocks and the fine blocks both rows selected are read once
// -- from memory and, what weighs more here, from LDS, where every key block is read three times (K rows, V rows, K
// transposed) -- and multiplied twice.
template <int Q, int R, bool NORM>
__global__ __launch_bounds__(256, Q == 1 ? 4 : 3) void attn_dq_kernel(llsa_attn_bwd_args a, float* __restrict__ stats,
                                                                      bf16* __restrict__ dor) {
    __shared__ __align__(16) bf16 sh[2][kGroup][2 * kTile];   // per block: R tile of K, R tile of V
    __shared__ int order[4][R * kWave];
    const int lane = threadIdx.x & 63, unit = r_unit(lane);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int N1 = a.N / kBlk, T = a.T;
    const int lid = xcd_logical_id();
    const int g = (lid % (int)gridDim.x) * (4 * Q) + Q * wave;        // query blocks g .. g + Q - 1 (the host checks N1 % 4 Q == 0)
    const int bh = lid / (int)gridDim.x, b = bh / a.H, h = bh % a.H;

    const bf16* kr = (const bf16*)a.kr + (int64_t)bh * N1 * kTile;
    const bf16* vr = (const bf16*)a.vr + (int64_t)bh * N1 * kTile;
    const int* ip = a.idx + ((int64_t)bh * N1 + g) * T;

    // shared list: the selected blocks of every pooled level below the coarsest, then every block of the coarsest
    SharedList sl = shared_list(a.lvl, a.levels, a.N, bh, g, lane);
    const int n_groups = sl.n_blocks / kGroup;
    bf16* const sh0 = &sh[0][0][0];
    auto issue_group = [&](int grp) __attribute__((always_inline)) {   // this wave brings in block kGroup*grp + wave
        const SharedTiles sb = shared_tiles(sl, a.lvl, bh, kGroup * grp + wave);
        bf16* dst = sh0 + ((grp & 1) * kGroup + wave) * (2 * kTile);
        copy16_global_to_lds(sb.k + unit, dst);
        copy16_global_to_lds<512>(sb.k + unit, dst);
        copy16_global_to_lds(sb.v + unit, dst + kTile);
        copy16_global_to_lds<512>(sb.v + unit, dst + kTile);
    };
    DqRows rows[Q];
#pragma unroll
    for (int u = 0; u < Q; u++) dq_request(rows[u], a, b, h, g + u, lane);
    issue_group(0);

    DqSide sd[Q];                                             // (the second buffer is not filled before the barrier of group 0)
#pragma unroll
    for (int u = 0; u < Q; u++) dq_begin(sd[u], rows[u], a, stats, dor, bh, g + u, lane, &sh[1][wave][0]);
    MergedLists<Q, R> ml = merge_lists<Q, R>(ip, min(T, kWave * R / Q), N1, lane, order[wave]);

    // ---- pooled blocks out of the shared copy.  The barrier at the top of round grp says: every
    // wave's part of group grp has landed, and every wave is done reading the other buffer.  All
    // LDS reads of a round come before the next fetch is issued (the compiler makes an LDS read
    // wait for every copy into LDS issued before it).
    // (two groups per trip: the buffer a group sits in is then a constant and every LDS address a lane-invariant
    // base plus an immediate)
    SharedWeight sw = first_weight(a.lvl, a.levels);
    auto shared_group = [&](int grp, const bf16* blk) __attribute__((always_inline)) {
        wait_vm0();
        __syncthreads();
        if (grp == sw.next) next_weight(sw, a.lvl, a.levels);
        const float w = __builtin_amdgcn_logf(sw.w);          // log2
        PairR r0;
        PairT t0;
        read_k_r(r0, blk, blk + 2 * kTile, lane);
        read_v_r(r0, blk + kTile, blk + 3 * kTile, lane);
        read_k_t(t0, blk, blk + 2 * kTile, lane);
#pragma unroll
        for (int u = 0; u < Q; u++) dq_pair_of_blocks(sd[u], r0, t0, w);
        read_k_r(r0, blk + 4 * kTile, blk + 6 * kTile, lane);
        read_v_r(r0, blk + 5 * kTile, blk + 7 * kTile, lane);
        read_k_t(t0, blk + 4 * kTile, blk + 6 * kTile, lane);
        if (grp + 1 < n_groups) issue_group(grp + 1);
#pragma unroll
        for (int u = 0; u < Q; u++) dq_pair_of_blocks(sd[u], r0, t0, w);
    };
    for (int grp = 0; grp < n_groups; grp += 2) {
        shared_group(grp, sh0);
        if (grp + 1 < n_groups) shared_group(grp + 1, sh0 + kGroup * (2 * kTile));
    }
    __syncthreads();                                          // the shared copy is dead: its LDS becomes private slots

    // ---- fine blocks: K of step t+1 is copied into the wave's other slot and V of step t+1 loaded
    // into registers while step t is worked on.  Nothing may be in flight when the wave ends (a copy
    // landing in LDS that already belongs to another workgroup), so the last step fetches nothing.
    bf16* const priv = sh0 + wave * (4 * kTile);              // two slots of two K tiles
    auto fine = [&]() __attribute__((always_inline)) {
        const int n_steps = (ml.n + 1) / 2;
        PairR ra, rb;
        auto fetch = [&](int t, PairR& dst) __attribute__((always_inline)) {
            bf16* slot = priv + (t & 1) * (2 * kTile);
#pragma unroll
            for (int j = 0; j < 2; j++) {
                const int64_t at = (int64_t)ml.block(min(2 * t + j, ml.n - 1)) * kTile;
                const bf16 *kb = kr + at, *vb = vr + at;
                copy16_global_to_lds(kb + unit, slot + j * kTile);
                copy16_global_to_lds<512>(kb + unit, slot + j * kTile);
                dst.v[j][0] = ld16(vb + lane * 8);
                dst.v[j][1] = ld16(vb + lane * 8 + 512);
            }
        };
        auto work = [&](int t, PairR& cur, PairR& nxt) __attribute__((always_inline)) {
            const unsigned m0 = ml.rows(2 * t), m1 = 2 * t + 1 < ml.n ? ml.rows(2 * t + 1) : 0u;
            wait_vm0();
            const bf16* slot = priv + (t & 1) * (2 * kTile);
            PairT tt;
            read_k_r(cur, slot, slot + kTile, lane);
            read_k_t(tt, slot, slot + kTile, lane);
            if (t + 1 < n_steps) fetch(t + 1, nxt);
#pragma unroll
            for (int u = 0; u < Q; u++) {
                const bool in0 = (m0 >> u) & 1u, in1 = (m1 >> u) & 1u;
                if (in0 || in1) dq_pair_of_blocks(sd[u], cur, tt, in0, in1);
            }
        };
        fetch(0, ra);
        for (int t = 0; t < n_steps; t += 2) {
            work(t, ra, rb);
            if (t + 1 < n_steps) work(t + 1, rb, ra);
        }
    };
    fine();
    if constexpr (Q == 1) {                                   // longer lists: 64 entries at a time
        for (int c0 = kWave * R; c0 < T; c0 += kWave * R) {
            ml = merge_lists<Q, R>(ip + c0, min(T - c0, kWave * R), N1, lane, order[wave]);
            fine();
        }
    }
    // what the way out reads, requested for all query blocks before the first store, which the compiler would not move a load across
    bf16x8 x[Q][2], f[Q][2];
    f32x4 gamma[4];
#pragma unroll
    for (int u = 0; u < Q; u++) {
        const int64_t tok = (g + u) * kBlk + (lane & 15);
        if (NORM) request_rows(x[u], (const bf16*)a.norm_q.x + b * a.norm_q.sxb + h * a.norm_q.sxh + tok * a.norm_q.sxn, lane >> 4);
        if (a.freq_dq != nullptr) request_rows(f[u], (const bf16*)a.freq_dq + tok * kD, lane >> 4);
    }
    if (NORM) norm_gamma(gamma, a.norm_q, lane >> 4);
    float contrib[16];
#pragma unroll
    for (int i = 0; i < 16; i++) contrib[i] = 0.f;
#pragma unroll
    for (int u = 0; u < Q; u++) dq_end<NORM>(sd[u], a, b, h, g + u, lane, x[u], f[u], gamma, contrib);
    if (NORM) {                                               // one row of partial sums per workgroup
        float* const red = reinterpret_cast<float*>(sh0);     // (the private slots: every wave is done with its own only after the barrier)
        __syncthreads();
        int ch;
        const float s = norm_contrib_sum(contrib, lane, ch);
        red[wave * kD + ch] = s;
        __syncthreads();
        if (threadIdx.x < kD) {
            const int t = threadIdx.x;
            a.norm_q.partials[((int64_t)bh * gridDim.x + lid % (int)gridDim.x) * kD + t] = (red[t] + red[kD + t]) + (red[2 * kD + t] + red[3 * kD + t]);
        }
    }
}

// ---------------------------------------------------------------------------------------
// K-side gradients.  A "unit" is 16 key rows (a fine K block, 16 pooled tokens of one coarse
// block, or 16 tokens of the dense coarsest level).  Three kernels: attn_kside_kernel walks the
// transposed selection of the fine blocks (unit-major: a unit and the list of query blocks that
// selected it), attn_kside_group_kernel the pooled levels under an ancestor's selection
// (query-group-major), attn_kside_dense_kernel the dense coarsest level and, on large grids, the lists that
// sixteen groups or more share (llsa_l3 and above).
// ---------------------------------------------------------------------------------------

// Optional last step of the fine dK / dV: add the pooled gradients the token's block received
// (what the backward of the two mean pools and autograd's accumulation do in the reference:
// every sum and every division by 16 rounded to bf16) and rotate dK back through the RoPE.
struct PoolFold {
    const bf16* gk[LLSA_MAX_LEVELS];              // gradients of the pooled k per level, (BH, N/16^l, 64); depth == 0: no folding
    const bf16* gv[LLSA_MAX_LEVELS];
    const bf16* freq;                             // (N, 64) or nullptr
    int depth;                                    // pooled levels to fold in
};
// What a token receives from its pooled ancestors, level by level, coarsest first (pool_bwd_accum_kernel applied down the
// chain): below = the running sum of the level above, g = the gradient of this level's own pooled token.
__device__ __forceinline__ bf16x4 fold_step(bf16x4 g, bf16x4 below) {
#pragma clang fp contract(off)
#pragma unroll
    for (int e = 0; e < 4; e++) g[e] = (bf16)((float)g[e] + rn_bf16((float)below[e] * 0.0625f));
    return g;
}
// x: four channels of one token; c: the same channels of the chain's sum at its level-1 ancestor; f: their [sin, cos] entries
__device__ __forceinline__ bf16x4 fold_math(bf16x4 x, bf16x4 c, bool has_f, bf16x4 f) {
    x = fold_step(x, c);
    return has_f ? rope_bwd4(x, f) : x;
}
// x: channels c0..c0+3 of token `tok` of (b,h) `bh`; which = 0 for dK, 1 for dV
__device__ __forceinline__ bf16x4 fold_pooled(bf16x4 x, const PoolFold& f, int which, int64_t bh, int N, int tok, int c0) {
    bf16x4 acc = x;
#pragma nounroll
    for (int l = f.depth - 1; l >= 0; l--) {
        const int sh = 4 * (l + 1);
        const bf16x4 g = ld8((which ? f.gv[l] : f.gk[l]) + (bh * (N >> sh) + (tok >> sh)) * kD + c0);
        acc = (l == f.depth - 1) ? g : fold_step(g, acc);
    }
    const bool rot = which == 0 && f.freq != nullptr;
    bf16x4 fr = x;
    if (rot) fr = ld8(f.freq + (int64_t)tok * kD + c0);
    return fold_math(x, acc, rot, fr);
}
constexpr int kFoldRows = 2 * LLSA_MAX_LEVELS * kD;   // LDS copy of a unit's fold operands: per level its dk and dv row, then 16 freq rows
constexpr int kFoldElems = kFoldRows + kBlk * kD;

struct KSideParams {
    const bf16* qr;  const bf16* dor;             // R tiles of q and dO, (BH, N1, 1024)
    const float* stats;                           // (BH, N1, kStats)
    const bf16* kk;  const bf16* vv;              // R tiles the unit's 16 key rows come from, (BH, n_units, 1024)
    const int* off;  const int* flat;             // CSR of the transposed selection (per K block)
    const int* work;                              // work list over that CSR (see transpose.hip)
    bf16* dk; int64_t sdkb, sdkh, sdkn;           // bf16 outputs
    bf16* dv; int64_t sdvb, sdvh, sdvn;
    f32x4* part;                                  // fp32 partials: slots (fine pass) or chunks (dense pass)
    int H, N, n_units, chunk_len;
    int64_t flat_stride;                          // entries of `flat` per (b,h)
    int64_t work_stride;                          // ints of `work` per (b,h)
    int64_t slot_stride;                          // partial slots per (b,h)
    float w;
    PoolFold fold;                                // fine pass only
    llsa_norm_back norm;                          // fine pass: the norm of k (x: nullptr without)
    int stripes, stripe_len;                      // fine pass: how the items are dealt to the XCDs (see kside_item)
};

// Two query blocks against the unit's 16 key rows, operands out of a wave-private piece of LDS: `stage` holds the
// R tiles of Q and dO of the two blocks (block u: Q at 2u, dO at 2u + 1), `stats` their statistics (kStats each).  The tiles
// are read twice, plainly as the A operands of S = Q.K^T and dP = dO.V^T and with the transposing read as the T
// operands of dV^T += dO^T.P and dK^T += Q^T.dS.
struct KsideOperands {
    bf16x8 aq[2][2], ag[2][2];
    bf16x4 tq[2][4], tg[2][4];
    f32x4 l4[2], d4[2];
};
__device__ __forceinline__ void kside_read(KsideOperands& o, const bf16* stage, const float* stats, int lane) {
    const int quad = lane >> 4;
#pragma unroll
    for (int u = 0; u < 2; u++) {
        const bf16* q = stage + (2 * u) * kTile;
        const bf16* g = stage + (2 * u + 1) * kTile;
        o.aq[u][0] = lds_ld16(q + r_unit(lane));
        o.aq[u][1] = lds_ld16(q + 512 + r_unit(lane));
        o.ag[u][0] = lds_ld16(g + r_unit(lane));
        o.ag[u][1] = lds_ld16(g + 512 + r_unit(lane));
#pragma unroll
        for (int dt = 0; dt < 4; dt++) {
            o.tq[u][dt] = lds_t_operand(q, dt, lane);
            o.tg[u][dt] = lds_t_operand(g, dt, lane);
        }
        o.l4[u] = *reinterpret_cast<const f32x4*>(stats + u * kStats + quad * 4);
        o.d4[u] = *reinterpret_cast<const f32x4*>(stats + u * kStats + kBlk + quad * 4);
    }
}
__device__ __forceinline__ void kside_pair(f32x4 dk[4], f32x4 dv[4], const bf16x8 bk[2], const bf16x8 bv[2], const KsideOperands& o,
                                           bool second_valid) {
    bf16x8 bp, bds;
#pragma unroll
    for (int u = 0; u < 2; u++) {
        f32x4 s = {0.f, 0.f, 0.f, 0.f}, dp = o.d4[u];
        s = mfma_bf16(o.aq[u][0], bk[0], s);
        s = mfma_bf16(o.aq[u][1], bk[1], s);
        dp = mfma_bf16(o.ag[u][0], bv[0], dp);
        dp = mfma_bf16(o.ag[u][1], bv[1], dp);
#pragma unroll
        for (int e = 0; e < 4; e++) {
            float pe = exp2_fast(fmaf(s[e], kScaleLog2e, o.l4[u][e]));
            if (u == 1 && !second_valid) pe = 0.f;
            bp[u * 4 + e] = (bf16)pe;
            bds[u * 4 + e] = (bf16)(pe * dp[e]);
        }
    }
#pragma unroll
    for (int dt = 0; dt < 4; dt++) {
        dv[dt] = mfma_bf16(cat(o.tg[0][dt], o.tg[1][dt]), bp, dv[dt]);
        dk[dt] = mfma_bf16(cat(o.tq[0][dt], o.tq[1][dt]), bds, dk[dt]);
    }
}

// A partial sum of one unit (16 key rows x 64 channels, dK and dV) is kept in the MFMA
// accumulator layout: 8 f32x4 registers per lane (4 channel tiles of dK, then 4 of dV).
__device__ __forceinline__ f32x4* part_slot(f32x4* part, int64_t slot) { return part + slot * (8 * kWave); }

// The items of the fine pass over the XCDs.  A (b,h)'s list is [long items | short items | places no item took], so XCDs that
// get contiguous pieces of the lists' storage (1.5 lists each for 12 (b,h)) get unequal work: nearly all long items and
// more items here, short ones and empty places there.  Every list is cut into `stripes` = 8 / gcd(BH, 8) stripes instead, each a
// contiguous share of its long and one of its short items, and every XCD gets the same number of stripes, neighbours in
// the list of (b,h)s.  (Shares dealt out in small turns are as even, but neighbouring key blocks, which are selected by the same
// queries, then sit on different XCDs: 6 x 32768 tokens 1.5 % of a step slower than the contiguous pieces.)
__device__ __forceinline__ bool kside_item(const KSideParams& p, int& bh, int& item) {
    const int xcd = (int)blockIdx.x % kXcds, slot = (int)blockIdx.x / kXcds;
    const int per_xcd = (int)gridDim.x / kXcds / p.stripe_len;                 // stripes per XCD
    const int stripe = xcd * per_xcd + slot / p.stripe_len, at = slot % p.stripe_len;
    bh = stripe / p.stripes;
    const int c = stripe % p.stripes;
    const int* work = p.work + (int64_t)bh * p.work_stride;
    const int n_long = work[3], n_short = work[0] - n_long;
    const int l0 = n_long * c / p.stripes, nl = n_long * (c + 1) / p.stripes - l0;
    const int s0 = n_short * c / p.stripes, ns = n_short * (c + 1) / p.stripes - s0;
    item = at < nl ? l0 + at : n_long + s0 + at - nl;
    return at < nl + ns;
}

// One work item of the fine pass: a key block and a piece (at most LLSA_CHUNK_FINE_MAX entries) of its list.
// One wave = one workgroup per item (items differ a lot in length; a wave that shared its workgroup
// with a longer one would keep its registers and LDS allocated while idle).
template <bool NORM>
__global__ __launch_bounds__(64) void attn_kside_kernel(KSideParams p) {
    __shared__ __align__(16) bf16 stage[4 * kTile];           // 2 query blocks x {Q, dO} R tiles
    __shared__ __align__(16) float stats[64];                 // their statistics
    __shared__ __align__(16) bf16 fold_buf[kFoldElems];
    int bh, item;
    if (!kside_item(p, bh, item)) return;
    const int lane = threadIdx.x & 63;
    const int N1 = p.N / kBlk;
    const int b = bh / p.H, h = bh % p.H;
    const int r = lane & 15, quad = lane >> 4;

    // which 16 key rows, which part of their query-block list, and where the result goes
    int unit, start, cnt;
    int64_t slot = -1;                                        // >= 0: write an fp32 partial
    const int* fl = nullptr;
    {
        const int* rec = p.work + (int64_t)bh * p.work_stride + 4 + 4 * item;
        unit = rec[0];
        start = rec[1];
        cnt = rec[2];
        const int sl = rec[3];
        if (sl >= 0) slot = (int64_t)bh * p.slot_stride + sl;
        fl = p.flat + (int64_t)bh * p.flat_stride;
    }
    // What the fold on the way out needs (the unit's pooled-gradient rows, its tokens' RoPE entries)
    // is copied into LDS now, without registers, so that no load waits at the end of the wave.
    const bool folding = p.fold.depth > 0 && slot < 0;
    if (folding) {
        const int row = lane >> 3, piece = lane & 7;          // rows: dk, dv of level 1, of level 2, ...; 8 x 16 bytes each
        if (row < 2 * p.fold.depth) {
            const int lvl = row >> 1;
            int n = N1, u = unit;
            for (int l = 0; l < lvl; l++) {
                n /= kBlk;
                u /= kBlk;
            }
            const bf16* src = ((row & 1) ? p.fold.gv[lvl] : p.fold.gk[lvl]) + ((int64_t)bh * n + u) * kD;
            copy16_global_to_lds(src + piece * 8, fold_buf);
        }
        if (p.fold.freq != nullptr) {
            const bf16* fr = p.fold.freq + (int64_t)unit * kBlk * kD;
            copy16_global_to_lds(fr + lane * 8, fold_buf + kFoldRows);
            copy16_global_to_lds(fr + 512 + lane * 8, fold_buf + kFoldRows + 512);
        }
    }
    // The item's list entries (at most LLSA_CHUNK_FINE_MAX query blocks) are fetched once, entry i into lane i % 64 of
    // register i / 64, and handed out with readlane: the walk below then has no load that depends on a load.  (Lanes behind the last entry have the last.)
    constexpr int kEntryRegs = LLSA_CHUNK_FINE_MAX / kWave;
    int mine[kEntryRegs];
#pragma unroll
    for (int k = 0; k < kEntryRegs; k++) mine[k] = k * kWave < cnt ? clampi(fl[start + min(k * kWave + lane, cnt - 1)], 0, N1 - 1) : 0;

    f32x4 dk[4], dv[4];
#pragma unroll
    for (int dt = 0; dt < 4; dt++) {
        dk[dt] = f32x4{0.f, 0.f, 0.f, 0.f};
        dv[dt] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    {
        bf16x8 bk[2], bv[2];
        const bf16* kp = p.kk + ((int64_t)bh * p.n_units + unit) * kTile + lane * 8;
        const bf16* vp = p.vv + ((int64_t)bh * p.n_units + unit) * kTile + lane * 8;
        bk[0] = ld16(kp);
        bk[1] = ld16(kp + 512);
        bv[0] = ld16(vp);
        bv[1] = ld16(vp + 512);
        const bf16* qrb = p.qr + (int64_t)bh * N1 * kTile;
        const bf16* dorb = p.dor + (int64_t)bh * N1 * kTile;
        const float* stb = p.stats + (int64_t)bh * N1 * kStats;
        // The operands of entries i, i + 1 are copied straight into LDS (no registers) while entries i - 2, i - 1 are
        // worked on: a round reads everything it needs out of LDS first, then starts the next copy into the same
        // place, then does its arithmetic.
        int g0 = 0, g1 = 0;                                   // the next two
        auto next_entries = [&](int i) __attribute__((always_inline)) {       // i: even, from 0 on in steps of two
            if (i > 0 && i % kWave == 0)                      // the next register moves up to the front
#pragma unroll
                for (int k = 1; k < kEntryRegs; k++) mine[k - 1] = mine[k];
            g0 = __builtin_amdgcn_readlane(mine[0], i % kWave);
            g1 = __builtin_amdgcn_readlane(mine[0], i % kWave + 1);
        };
        auto fetch = [&]() __attribute__((always_inline)) {
            const int at = r_unit(lane);
            const bf16 *q0 = qrb + (int64_t)g0 * kTile, *d0 = dorb + (int64_t)g0 * kTile;
            const bf16 *q1 = qrb + (int64_t)g1 * kTile, *d1 = dorb + (int64_t)g1 * kTile;
            copy16_global_to_lds(q0 + at, stage);
            copy16_global_to_lds<512>(q0 + at, stage);
            copy16_global_to_lds(d0 + at, stage + kTile);
            copy16_global_to_lds<512>(d0 + at, stage + kTile);
            copy16_global_to_lds(q1 + at, stage + 2 * kTile);
            copy16_global_to_lds<512>(q1 + at, stage + 2 * kTile);
            copy16_global_to_lds(d1 + at, stage + 3 * kTile);
            copy16_global_to_lds<512>(d1 + at, stage + 3 * kTile);
            if (lane < 16) {                                  // four floats a lane: the statistics of g0, of g1
                const float* src = stb + (int64_t)((lane & 8) ? g1 : g0) * kStats + (lane & 7) * 4;
                copy16_global_to_lds(reinterpret_cast<const bf16*>(src), reinterpret_cast<bf16*>(stats));
            }
        };
        next_entries(0);
        if (cnt > 0) fetch();
        for (int i = 0; i < cnt; i += 2) {
            wait_vm0();
            KsideOperands o;
            kside_read(o, stage, stats, lane);
            next_entries(i + 2);                              // (while the reads arrive)
            wait_all_mem();                                   // every lane has its operands: the next copy may land
            __builtin_amdgcn_wave_barrier();
            if (i + 2 < cnt) fetch();
            kside_pair(dk, dv, bk, bv, o, i + 1 < cnt);
        }
    }

    if (slot >= 0) {
        f32x4* ps = part_slot(p.part, slot);
#pragma unroll
        for (int dt = 0; dt < 4; dt++) {
            ps[dt * kWave + lane] = dk[dt];
            ps[(4 + dt) * kWave + lane] = dv[dt];
        }
        return;
    }
    bf16* kp = p.dk + b * p.sdkb + h * p.sdkh + (int64_t)(unit * kBlk + r) * p.sdkn;
    bf16* vp = p.dv + b * p.sdvb + h * p.sdvh + (int64_t)(unit * kBlk + r) * p.sdvn;
    bf16x4 nx[4];
    f32x4 ngamma[4];
    if (NORM) norm_load(nx, ngamma, p.norm, b, h, unit * kBlk + r, quad);
    if (folding) {
        wait_vm0();                                           // the copies into fold_buf (long since done)
        // the chain of pooled levels collapses into one row for dk and one for dv, left where level 1's rows were:
        // lane (which, four channels) reads its channels of every level and is the only one to write them
        if (lane < 32) {
            const int which = lane >> 4, c0 = (lane & 15) * 4;
            bf16x4 acc = lds_ld8(fold_buf + (2 * (p.fold.depth - 1) + which) * kD + c0);
#pragma nounroll
            for (int l = p.fold.depth - 2; l >= 0; l--) acc = fold_step(lds_ld8(fold_buf + (2 * l + which) * kD + c0), acc);
            lds_st8(fold_buf + which * kD + c0, acc);
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
    bf16x4 ok[4], ov[4];
#pragma unroll
    for (int dt = 0; dt < 4; dt++) {
        ok[dt] = cvt4(dk[dt] * kScale);
        ov[dt] = cvt4(dv[dt]);
        if (folding) {
            const int c0 = dt * 16 + quad * 4;
            ok[dt] = fold_math(ok[dt], lds_ld8(fold_buf + c0), p.fold.freq != nullptr, lds_ld8(fold_buf + kFoldRows + r * kD + c0));
            ov[dt] = fold_math(ov[dt], lds_ld8(fold_buf + kD + c0), false, ov[dt]);
        }
    }
    store_rows(vp, ov, quad, rows_wide(p.dv, p.sdvb, p.sdvh, p.sdvn));
    if (NORM) {
        float contrib[16];
#pragma unroll
        for (int i = 0; i < 16; i++) contrib[i] = 0.f;
        norm_back(ok, nx, ngamma, p.norm.eps, contrib);
        int ch;
        const float s = norm_contrib_sum(contrib, lane, ch);
        p.norm.partials[((int64_t)bh * p.n_units + unit) * kD + ch] = s;       // (a unit cut into pieces: kside_reduce_kernel's row)
    }
    store_rows(kp, ok, quad, rows_wide(p.dk, p.sdkb, p.sdkh, p.sdkn));
}

// ---------------------------------------------------------------------------------------
// Dense coarsest level.  Every unit (16 pooled tokens) meets every query block, so the Q / dO
// tiles are the same for all units: a workgroup takes WAVES * UPW units (UPW per wave) and one piece
// of the query range and streams that piece through LDS, a pair of query blocks (8 KB) per
// round, once for all of its units.  The stream is three rounds deep: the tiles of round t + 3 are requested from memory (every
// wave its share, into registers) while those of round t + 1 move from registers into the other LDS buffer and round t is worked on,
// so a tile has two rounds of arithmetic to arrive.  (Copies straight into LDS cannot be run ahead like that: the compiler
// waits for all of them before any LDS read.)  Each wave ends with the partial sums of its units over this piece of the range.
//
// What bounds it is the instruction stream of a SIMD.  A round of two units is 32 MFMAs of 16 cycles, which keep vector instructions
// from being issued for 8 of them, 48 vector instructions of 4 cycles and 16 exponentials of 8: 576 cycles if nothing waits.  Waves
// that run alike read LDS at the same time and then multiply at the same time: four waves of two units took 1009 cycles a round at 6 x
// 262144 tokens (51 % of the matrix cores' cycles busy).  So
//  * the vector instructions of one unit are placed between the products of the other (interleave): 960, and
//  * eight waves take turns: four of them, one per SIMD, fetch their operands from LDS while the other four multiply (862 cycles, 59 %;
//    820 -> 715 us).  A barrier ends each half; the second four start half a round late.
// (Tried: the row operands of the next round fetched under the products, exponentials in the half of the LDS reads: both slower;
// products of 32 x 32, which block vector instructions half as long, with a ring of eight pairs in LDS: 1058, their operands are
// all needed before the first exponential.)
// ---------------------------------------------------------------------------------------
// Everything one unit's products of a round (two query blocks) need of the round's tiles and statistics
struct DenseOps {
    bf16x8 q[2][2], g[2][2];       // R operands of Q and dO
    bf16x4 tq[2][4], tg[2][4];     // T operands
    f32x4 l[2], d[2];              // statistics
};

// ... read out of LDS (tiles of the two query blocks, `stats` of the first, the second's behind them)
__device__ __forceinline__ void dense_operands(DenseOps& o, const bf16* q0, const bf16* g0, const bf16* q1, const bf16* g1, const float* stats,
                                               int lane) {
    const int quad = lane >> 4;
#pragma unroll
    for (int u = 0; u < 2; u++) {
        const bf16 *q = u ? q1 : q0, *g = u ? g1 : g0;
        o.q[u][0] = lds_ld16(q + r_unit(lane));
        o.q[u][1] = lds_ld16(q + 512 + r_unit(lane));
        o.g[u][0] = lds_ld16(g + r_unit(lane));
        o.g[u][1] = lds_ld16(g + 512 + r_unit(lane));
        o.l[u] = *reinterpret_cast<const f32x4*>(stats + u * kStats + quad * 4);
        o.d[u] = *reinterpret_cast<const f32x4*>(stats + u * kStats + kBlk + quad * 4);
    }
#pragma unroll
    for (int u = 0; u < 2; u++)
#pragma unroll
        for (int dt = 0; dt < 4; dt++) {
            o.tq[u][dt] = lds_t_operand(u ? q1 : q0, dt, lane);
            o.tg[u][dt] = lds_t_operand(u ? g1 : g0, dt, lane);
        }
}
// A round's products of UPW units (a weight is left out of the exponentials: it multiplies the sums at the end)
template <int UPW>
__device__ __forceinline__ void dense_products(f32x4 (*dk)[4], f32x4 (*dv)[4], const bf16x8 (*bk)[2], const bf16x8 (*bv)[2], const DenseOps& o) {
    f32x4 sc[UPW][2], dp[UPW][2];
    bf16x8 bp[UPW], bds[UPW];
    auto scores = [&](int j) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < 2; u++) {
            const f32x4 z = {0.f, 0.f, 0.f, 0.f};
            sc[j][u] = mfma_bf16(o.q[u][0], bk[j][0], z);
            dp[j][u] = mfma_bf16(o.g[u][0], bv[j][0], o.d[u]);
        }
#pragma unroll
        for (int u = 0; u < 2; u++) {
            sc[j][u] = mfma_bf16(o.q[u][1], bk[j][1], sc[j][u]);
            dp[j][u] = mfma_bf16(o.g[u][1], bv[j][1], dp[j][u]);
        }
    };
    auto exponentials = [&](int j) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < 2; u++)
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const float pe = exp2_fast(fmaf(sc[j][u][e], kScaleLog2e, o.l[u][e]));
                bp[j][u * 4 + e] = (bf16)pe;
                bds[j][u * 4 + e] = (bf16)(pe * dp[j][u][e]);
            }
    };
    auto sums = [&](int j) __attribute__((always_inline)) {
#pragma unroll
        for (int dt = 0; dt < 4; dt++) {
            dv[j][dt] = mfma_bf16(cat(o.tg[0][dt], o.tg[1][dt]), bp[j], dv[j][dt]);
            dk[j][dt] = mfma_bf16(cat(o.tq[0][dt], o.tq[1][dt]), bds[j], dk[j][dt]);
        }
    };
    // the vector instructions of one unit between the products of the other, in this order
    auto interleave = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < 8; i++) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);      // one MFMA
            __builtin_amdgcn_sched_group_barrier(0x002, 4, 0);      // four vector ALU instructions (and the exponentials among them)
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    scores(0);
    if constexpr (UPW == 2) {
        __builtin_amdgcn_sched_barrier(0);
        scores(1);
        exponentials(0);
        interleave();
        sums(0);
        exponentials(1);
        interleave();
        sums(1);
    } else {
        exponentials(0);
        sums(0);
    }
}

// With LISTS the units are those of a selection (level 2 of llsa_l3 and above): piece i of the query range belongs to owner i >> chunk_shift,
// the common ancestor of its query blocks, whose list names the units; the partial sum of an entry and a piece is left where the
// transposed selection puts the entry, 1 << chunk_shift of them side by side.
struct KSideLists {
    const int* sel; const int* inv;               // (BH, owners, cnt)
    int cnt, chunk_shift;
};
template <int WAVES, int UPW, bool LISTS>
__global__ __launch_bounds__(64 * WAVES, UPW == 2 ? 2 : 3) void attn_kside_dense_kernel(KSideParams p, KSideLists ls) {
    static_assert(WAVES == 4 || WAVES == 8, "a wave moves one or two of the eight half tiles of a pair");
    __shared__ __align__(16) bf16 sh[2][4 * kTile];           // per pair: Q0, dO0, Q1, dO1 as R tiles
    __shared__ __align__(16) float sh_stats[2][64];           // per pair: the statistics of its two query blocks
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int N1 = p.N / kBlk;
    // Workgroups that stream the same piece of the query range (one per group of units) get neighbouring logical ids,
    // which xcd_logical_id keeps on one XCD: the piece then comes out of that XCD's L2 for all but the first of them.
    const int n_met = LISTS ? ls.cnt : p.n_units;              // units that meet a piece
    const int unit_groups = (n_met + WAVES * UPW - 1) / (WAVES * UPW);
    const int lid = xcd_logical_id();                          // grid: (unit_groups * pieces, BH)
    const int piece = (lid % (int)gridDim.x) / unit_groups;
    const int bh = lid / (int)gridDim.x;
    const int unit0 = (((lid % (int)gridDim.x) % unit_groups) * WAVES + wave) * UPW;
    const bool active = unit0 < n_met;                        // (n_met is a multiple of UPW; a wave past the end only moves tiles)
    const int64_t entry0 = LISTS ? ((int64_t)bh * (((int)gridDim.x / unit_groups) >> ls.chunk_shift) + (piece >> ls.chunk_shift)) * ls.cnt : 0;
    const int start = piece * p.chunk_len;
    const int n_pairs = min(p.chunk_len, N1 - start) / 2;     // even: chunk_len and N1 are multiples of 4
    if (n_pairs <= 0) return;                                 // uniform over the workgroup
    const bf16* qrb = p.qr + ((int64_t)bh * N1 + start) * kTile;
    const bf16* dorb = p.dor + ((int64_t)bh * N1 + start) * kTile;
    const float* stb = p.stats + ((int64_t)bh * N1 + start) * kStats;

    // The four tiles of a pair are eight half tiles: tile i/2 (query block i/4; Q for even tiles, dO for odd ones), half i%2.  Wave w
    // moves half tile w (of eight waves) or 2 w and 2 w + 1 (of four); the first 16 lanes of wave 0 also the pair's 64 statistics.
    // Rounds past the end re-read the last pair (no branch around loads).
    constexpr int HALVES = 8 / WAVES;
    struct Stage { bf16x8 h[HALVES]; f32x4 s; };
    const bool stat_lane = wave == 0 && lane < 16;
    const int half0 = wave * HALVES;
    auto request = [=](int t, Stage& st) __attribute__((always_inline)) {
        t = min(t, n_pairs - 1);
        const bf16* src = (((half0 >> 1) & 1) ? dorb : qrb) + (int64_t)(2 * t + (half0 >> 2)) * kTile + (half0 & 1) * 512;
#pragma unroll
        for (int i = 0; i < HALVES; i++) st.h[i] = ld16(src + i * 512 + lane * 8);
        // (every lane of every wave loads, lanes 16.. the same as lane % 16: a load inside a branch makes the compiler lose
        // count of the loads in flight, after which it waits for all of them in every round)
        st.s = *reinterpret_cast<const f32x4*>(stb + (int64_t)(2 * t) * kStats + (lane & 15) * 4);
    };
    auto deposit = [&](int t, const Stage& st) __attribute__((always_inline)) {
        bf16* dst = &sh[t & 1][half0 * 512];
#pragma unroll
        for (int i = 0; i < HALVES; i++) st16(dst + i * 512 + r_unit(lane), st.h[i]);
        if (stat_lane) *reinterpret_cast<f32x4*>(&sh_stats[t & 1][lane * 4]) = st.s;
    };
    Stage s0, s1;
    request(0, s0);
    request(1, s1);
    bf16x8 bk[UPW][2], bv[UPW][2];
#pragma unroll
    for (int j = 0; j < UPW; j++) {
        int unit = min(unit0 + j, n_met - 1);
        if (LISTS) unit = clampi(ls.sel[entry0 + unit], 0, p.n_units - 1);
        const bf16* kp = p.kk + ((int64_t)bh * p.n_units + unit) * kTile + lane * 8;
        const bf16* vp = p.vv + ((int64_t)bh * p.n_units + unit) * kTile + lane * 8;
        bk[j][0] = ld16(kp);
        bk[j][1] = ld16(kp + 512);
        bv[j][0] = ld16(vp);
        bv[j][1] = ld16(vp + 512);
    }
    deposit(0, s0);
    request(2, s0);
    f32x4 dk[UPW][4], dv[UPW][4];
#pragma unroll
    for (int j = 0; j < UPW; j++)
#pragma unroll
        for (int dt = 0; dt < 4; dt++) {
            dk[j][dt] = f32x4{0.f, 0.f, 0.f, 0.f};
            dv[j][dt] = f32x4{0.f, 0.f, 0.f, 0.f};
        }

    DenseOps o;
    // First half of a round: this wave's operands out of LDS, its share of the next pair into the other buffer, the request for
    // the pair after the next but one.
    auto gather = [&](int t, Stage& nxt) __attribute__((always_inline)) {
        const bf16* b = &sh[t & 1][0];
        dense_operands(o, b, b + kTile, b + 2 * kTile, b + 3 * kTile, sh_stats[t & 1], lane);
        deposit(t + 1, nxt);
        request(t + 3, nxt);
    };
    auto multiply = [&]() __attribute__((always_inline)) {
        __builtin_amdgcn_sched_barrier(0);
        dense_products<UPW>(dk, dv, bk, bv, o);
        __builtin_amdgcn_sched_barrier(0);
    };
    if constexpr (WAVES == 8) {
        // Buffer (t + 1) & 1 is refilled in the first half of round t, by the first four waves while the others multiply round t - 1
        // and by those while the first multiply round t: nobody reads it then, and it is whole before anybody reads round t + 1.
        // The halves are half a round apart, so the barrier that ends one half's products ends the other's fetches: they stand at
        // different places.  Both arrive 2 n_pairs + 2 times, the second four waves one time more in front and one time less behind.
        auto round = [&](int t, Stage& nxt) __attribute__((always_inline)) {
            gather(t, nxt);
            counted_barrier();
            if (active) multiply();
            counted_barrier();
        };
        counted_barrier();
        if (wave >= 4) counted_barrier();
        for (int t = 0; t < n_pairs; t += 2) {
            round(t, s1);
            round(t + 1, s0);
        }
        if (wave < 4) counted_barrier();
    } else {
        auto round = [&](int t, Stage& nxt) __attribute__((always_inline)) {
            __syncthreads();
            gather(t, nxt);
            if (active) multiply();
        };
        // (two rounds per trip without a branch between them: n_pairs is even, and with a conditional second round the
        // compiler loses count of the loads in flight where the loop closes and waits for all of them)
        for (int t = 0; t < n_pairs; t += 2) {
            round(t, s1);
            round(t + 1, s0);
        }
    }
    if (!active) return;
#pragma unroll
    for (int j = 0; j < UPW; j++) {
        int64_t slot = ((int64_t)piece * gridDim.y + bh) * p.n_units + unit0 + j;
        if (LISTS) {
            const int pos = clampi(ls.inv[entry0 + unit0 + j], 0, (int)(p.slot_stride >> ls.chunk_shift) - 1);
            slot = (int64_t)bh * p.slot_stride + ((int64_t)pos << ls.chunk_shift) + (piece & ((1 << ls.chunk_shift) - 1));
        }
        f32x4* ps = part_slot(p.part, slot);
#pragma unroll
        for (int dt = 0; dt < 4; dt++) {
            const f32x4 k = dk[j][dt] * p.w, v = dv[j][dt] * p.w;      // (the weight, left out of the exponentials)
            if constexpr (LISTS) {                           // (large grids only: past the caches, see kGroupStreamBytes)
                __builtin_nontemporal_store(k, &ps[dt * kWave + lane]);
                __builtin_nontemporal_store(v, &ps[(4 + dt) * kWave + lane]);
            } else {
                ps[dt * kWave + lane] = k;
                ps[(4 + dt) * kWave + lane] = v;
            }
        }
    }
}

// ---------------------------------------------------------------------------------------
// Pooled levels whose keys come from an ancestor's selection (the level-1 pooled tokens of
// llsa_l2 / llsa_l3 under the parent's coarse blocks, the level-2 pooled tokens of llsa_l3 under
// the grand-parent's), "group-major": a workgroup owns one group of 16 consecutive query blocks
// -- the children of one parent, which all read the same pooled key blocks -- copies their Q and
// dO tiles into LDS once (64 KB) and meets every key block of the group's lists there; a wave
// takes its share of the key blocks, two at a time, and ends each with that block's dK / dV summed
// over the group's 256 queries.  A key block selected by several ancestors receives one such
// partial sum per selecting group, written where pooled_reduce_kernel finds the partial sums of a
// key block side by side: at the position the transposed selection gives the (ancestor, entry)
// pair.  Walking the transposed lists instead (key block major, the reference's order,
// sparse_attention_res_2.py:492-575) fetches the 64 KB of a group once per key block that
// selected it, T2 times in all.
// With few tokens on the dense coarsest level its blocks are appended to the lists (every group
// meets all of them), which saves that level a pass of its own over Q and dO.
// What bounds it is the instruction stream, as in the dense pass, and the waits at both ends of a wave's pass over the queries: two
// workgroups a CU (64 KB of tiles each) fill them for one another.  The vector instructions of one key block stand between the
// products of the other, the statistics lie in LDS beside the tiles, and a pass's key blocks are requested before the sums of the pass before
// it are rounded and stored: 163 -> 148 us at 48 x 16384 tokens (20 blocks a group), 255 -> 225 at 6 x 262144 (16), 490 -> 441 with 36 blocks;
// 45 at 12 x 16384 either way (768 workgroups, 512 places).  (Tried: one workgroup of eight waves per CU that stays, the next
// group's tiles copied into a second buffer meanwhile and the halves taking turns as in the dense pass: 186, 254, 588.)
// ---------------------------------------------------------------------------------------
constexpr int kGroupWaves = 4;
constexpr int kGroupSegs = LLSA_MAX_LEVELS;
constexpr int kGroupMaxBlocks = 64;               // key blocks per group over all its lists (their ids live in one lane each)
constexpr int kGroupDenseMax = 8;                 // dense blocks are appended up to this many
// From this many bytes of partial sums on, and with this many key blocks a group, they are stored past the caches (STREAM): they are read once, by a
// later kernel, and push the tiles of q and dO that the fine pass gathers out of the caches meanwhile.  Training steps, us, through the
// caches / past them, read past them either way (kReduceStreamBytes):
//   20 key blocks: 16 x 16384 tokens, 80 MiB, 392 / 385;  18 x 16384 443 / 436;  24 x 16384 581 / 568.5;  48 x 16384 1159 / 1147
//   24: 8 x 32768, 96 MiB, 424 / 421;  12 x 32768 620 / 612.5     36: 12 x 16384, 108 MiB, 372 / 366     16: 6 x 65536, 96 MiB, 682 / 677;  8 x 65536 909 /
//   906;  36 x 16384, 144 MiB, 838 / 830.5;  24 x 16384, 96 MiB, 535 / 538;  48 x 16384, 16 x 65536 and 3 x 262144 even;  24 x 32768 1092 / 1096
//   12: 30 x 16384, 90 MiB, 644.5 / 647;  48 x 16384 1019 / 1024;  72 x 16384 1494 / 1505;  24 x 32768 1014 / 1022
//   three levels: 3 x 262144 even, but 1 x 262144, 36 key blocks, 144 MiB, 691 / 699
// The number of key blocks is a multiple of 4 (topk and coarsest blocks are), so 12 and 16 are neighbours.  Below the byte line, 64 to 80 MiB: 13 x
// 16384 338 / 336, 6 x 32768 335 / 330.5, but 6 x 49152 510 / 512, 3 x 49152 with 32 key blocks 678 / 679; 10 x 16384, 50 MiB, 267.9 / 268.2.
constexpr int64_t kGroupStreamBytes = (int64_t)80 << 20;
constexpr int kGroupStreamBlocks = 16;
static_assert(LLSA_POOLED_TOPK_MAX + kGroupDenseMax <= kGroupMaxBlocks, "a group's lists must fit one lane per key block");

struct GroupSeg {
    const bf16* kk; const bf16* vv;               // R tiles of this level's pooled k, v: (BH, n_units, 1024)
    const int* sel;                               // (BH, n_groups >> owner_shift, cnt) blocks selected by the group's ancestor;
                                                  // nullptr: blocks 0..cnt-1 (dense level)
    const int* inv;                               // (BH, n_groups >> owner_shift, cnt) position of each entry in the transposed selection
    bf16x8* part;                                 // partial sums, the accumulators of part_slot rounded to bf16, two registers (16 bytes)
                                                  // per lane side by side: slot = [4 register pairs][64 lanes] bf16x8.  The
                                                  // group-major pass writes one per (group, key block), 8 KB each in fp32, which at
                                                  // 16384 tokens is more memory traffic than everything else the pass moves; a group's
                                                  // sum over its 256 queries is taken in fp32 and rounded once (2^-9 relative), and the
                                                  // reduction adds the rounded sums of a key block's groups in fp32
    int n_units, owner_shift, cnt;
    int64_t slots;                                // partial slots per (b,h) (sparse) -- positions are clamped into them
    float w;
};
struct GroupParams {
    const bf16* qr; const bf16* dor;              // R tiles of q and dO, (BH, N1, 1024)
    const float* stats;                           // (BH, N1, kStats)
    int BH, N, n_segs, n_blocks;
    int whole, parts;                             // see GroupSplit
    GroupSeg seg[kGroupSegs];
};

// Workgroups of the group-major pass over an XCD's `groups` groups.  32 CUs take two each; where that leaves a last round at most half full, the key blocks
// of its groups are dealt out to `parts` workgroups, each with the group's tiles in LDS, and the first `whole` groups are as before.  Every key block is
// still met by one wave, so the results are the same.  Training steps of two levels, topk 16/16, us, whole / dealt out: 1 x 16384 tokens (8 groups an XCD) 91.0 /
// 84.8;  at 16/32 106.6 / 95.2;  10 x 16384 (80) 250.4 / 246.3;  17 x 16384 at 16/12 (136) 374.1 / 370.3;  9 x 16384 at 16/32 (72) 293.0 / 284.2;  1 x 32768 119.1 /
// 113.7;  3 x 49152 at 64/32 (72) 635.3 / 625.3;  just half full 4 x 16384 (32) and 12 x 16384 (96) even.
struct GroupSplit { int whole, parts; };
// key blocks of a wave of a group that `parts` workgroups share
__host__ __device__ inline int group_wave_blocks(int n_blocks, int parts) { return (n_blocks + kGroupWaves * parts - 1) / (kGroupWaves * parts); }
constexpr int kGroupSlots = 2 * 256 / kXcds;
// key blocks to a part, on the average over a group's parts, at least.  3 / 4 / 6 / 8 / 12, us: 1 x 16384 84.9 / 84.9 / 84.8 / 87.3 / 90.9;  17 x 16384 at 16/12 369.8 / 369.4 /
// 370.3 / 369.2 / 374.6;  9 x 16384 at 16/32 284.4 / 284.8 / 284.2 / 281.6 / 281.8;  3 x 49152 at 64/32 629.6 / 629.6 / 625.3 / 625.2 / 627.4
constexpr int kGroupPartBlocks = 6;
static GroupSplit group_split(int groups, int n_blocks) {
    const int rest = groups % kGroupSlots;
    int parts = rest == 0 ? 1 : std::min(kGroupSlots / rest, n_blocks / kGroupPartBlocks);
    if (parts < 2) return {groups, 1};
    const int share = kGroupWaves * group_wave_blocks(n_blocks, parts);       // of every part but the last
    parts = (n_blocks + share - 1) / share;                                   // (none of them empty; the shares are the same)
    return {groups - rest, parts};
}

// UPW key blocks against the group's 16 query blocks, two query blocks per step, operands out of LDS.  `next` starts the loads of the
// wave's next key blocks, into bk and bv, where these are no longer needed: they arrive while the sums are rounded and stored.
template <int UPW, bool STREAM, typename NEXT>
__device__ __forceinline__ void group_pass(const bf16x8 (&bk)[2][2], const bf16x8 (&bv)[2][2], const float (&weights)[2], bf16x8* const (&slots)[2],
                                           const bf16* shq, const bf16* shg, const float* sh_stats, int lane, NEXT&& next) {
    f32x4 dk[UPW][4], dv[UPW][4];
#pragma unroll
    for (int j = 0; j < UPW; j++)
#pragma unroll
        for (int dt = 0; dt < 4; dt++) {
            dk[j][dt] = f32x4{0.f, 0.f, 0.f, 0.f};
            dv[j][dt] = f32x4{0.f, 0.f, 0.f, 0.f};
        }
#pragma unroll 1
    for (int t = 0; t < kBlk / 2; t++) {
        DenseOps o;
        dense_operands(o, shq + 2 * t * kTile, shg + 2 * t * kTile, shq + (2 * t + 1) * kTile, shg + (2 * t + 1) * kTile,
                       sh_stats + 2 * t * kStats, lane);
        dense_products<UPW>(dk, dv, bk, bv, o);
    }
    float w[UPW];
    bf16x8* dst[UPW];
#pragma unroll
    for (int j = 0; j < UPW; j++) {
        w[j] = weights[j];
        dst[j] = slots[j];
    }
    next();
    // The partial sums of this pass leave as bf16 (see GroupSeg::part): the sum over the group's 256 queries was
    // taken in fp32, and the result the reduction makes of them is a bf16 tensor.
#pragma unroll
    for (int j = 0; j < UPW; j++)
#pragma unroll
        for (int pr = 0; pr < 2; pr++) {                      // registers 2 pr, 2 pr + 1 of dK, then of dV: 16 bytes a lane and store
            const bf16x8 k = cat(cvt4(dk[j][2 * pr] * w[j]), cvt4(dk[j][2 * pr + 1] * w[j]));
            const bf16x8 v = cat(cvt4(dv[j][2 * pr] * w[j]), cvt4(dv[j][2 * pr + 1] * w[j]));
            if constexpr (STREAM) {
                __builtin_nontemporal_store(k, &dst[j][pr * kWave + lane]);
                __builtin_nontemporal_store(v, &dst[j][(2 + pr) * kWave + lane]);
            } else {
                dst[j][pr * kWave + lane] = k;
                dst[j][(2 + pr) * kWave + lane] = v;
            }
        }
}

template <bool STREAM>
__global__ __launch_bounds__(64 * kGroupWaves, 2) void attn_kside_group_kernel(GroupParams p) {
    __shared__ __align__(16) bf16 sh[2][kBlk * kTile];        // R tiles of the group's 16 query blocks: Q, then dO
    __shared__ __align__(16) float sh_stats[kBlk * kStats];   // their statistics
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int N1 = p.N / kBlk, n_groups = N1 / kBlk;
    const int slot = (int)blockIdx.x / kXcds, behind = slot - p.whole;        // (an XCD's workgroups are every eighth)
    const int part = behind < 0 ? 0 : behind % p.parts, parts = behind < 0 ? 1 : p.parts;
    const int lid = (int)blockIdx.x % kXcds * (n_groups * p.BH / kXcds) + (behind < 0 ? slot : p.whole + behind / p.parts);
    const int G = lid % n_groups;                              // group of query blocks 16 G .. 16 G + 15
    const int bh = lid / n_groups;

    {   // 32 KB of Q tiles and 32 KB of dO tiles, contiguous in memory, 1 KB per wave and copy
        const bf16* qsrc = p.qr + ((int64_t)bh * N1 + (int64_t)G * kBlk) * kTile;
        const bf16* gsrc = p.dor + ((int64_t)bh * N1 + (int64_t)G * kBlk) * kTile;
#pragma unroll
        for (int i = 0; i < 2 * kBlk / kGroupWaves; i++) {
            const int piece = i * kGroupWaves + wave;
            copy16_global_to_lds(qsrc + piece * 512 + r_unit(lane), &sh[0][piece * 512]);
            copy16_global_to_lds(gsrc + piece * 512 + r_unit(lane), &sh[1][piece * 512]);
        }
        const float* ssrc = p.stats + ((int64_t)bh * N1 + (int64_t)G * kBlk) * kStats;
        if (wave < 2) copy16_global_to_lds(reinterpret_cast<const bf16*>(ssrc + wave * 256 + lane * 4), reinterpret_cast<bf16*>(sh_stats + wave * 256));
    }
    // Key block j of the group's lists lives in lane j: which tile, which weight, where its partial sum goes.
    int my_unit = 0, my_seg = 0;
    int64_t my_slot = 0;
    {
        int j = lane, sgi = 0;
        while (sgi < p.n_segs - 1 && j >= p.seg[sgi].cnt) {
            j -= p.seg[sgi].cnt;
            sgi++;
        }
        const GroupSeg& sg = p.seg[sgi];
        if (lane < p.n_blocks) {
            my_seg = sgi;
            if (sg.sel != nullptr) {
                const int64_t e = ((int64_t)bh * (n_groups >> sg.owner_shift) + (G >> sg.owner_shift)) * sg.cnt + j;
                my_unit = clampi(sg.sel[e], 0, sg.n_units - 1);
                const int64_t pos = ((int64_t)clampi(sg.inv[e], 0, (int)((sg.slots >> sg.owner_shift) - 1)) << sg.owner_shift) +
                                    (G & ((1 << sg.owner_shift) - 1));
                my_slot = (int64_t)bh * sg.slots + pos;
            } else {
                my_unit = j;
                my_slot = ((int64_t)G * p.BH + bh) * sg.n_units + j;      // [group][bh][unit]: what the dense reduction walks
            }
        }
    }
    // this wave's key blocks: a contiguous share, taken two at a time (the last alone if the share is odd)
    const int per = group_wave_blocks(p.n_blocks, parts);
    const int lo = min((part * kGroupWaves + wave) * per, p.n_blocks), hi = min(lo + per, p.n_blocks);

    bf16x8 bk[2][2], bv[2][2];
    float w[2];
    bf16x8* dst[2];
    auto fetch = [&](int j, int u) __attribute__((always_inline)) {    // K, V tiles of key block j into register set u
        const int sgi = __builtin_amdgcn_readlane(my_seg, j);
        const int unit = __builtin_amdgcn_readlane(my_unit, j);
        const int slo = __builtin_amdgcn_readlane((int)(my_slot & 0xffffffff), j), shi = __builtin_amdgcn_readlane((int)(my_slot >> 32), j);
        const GroupSeg& sg = p.seg[sgi];
        const bf16* kp = sg.kk + ((int64_t)bh * sg.n_units + unit) * kTile + lane * 8;
        const bf16* vp = sg.vv + ((int64_t)bh * sg.n_units + unit) * kTile + lane * 8;
        bk[u][0] = ld16(kp);
        bk[u][1] = ld16(kp + 512);
        bv[u][0] = ld16(vp);
        bv[u][1] = ld16(vp + 512);
        w[u] = sg.w;
        dst[u] = sg.part + (((int64_t)(unsigned)slo) | ((int64_t)shi << 32)) * (4 * kWave);
    };
    if (lo < hi) fetch(lo, 0);
    if (lo + 1 < hi) fetch(lo + 1, 1);
    wait_vm0();
    __syncthreads();                                          // the copies into LDS are everybody's
    for (int j = lo; j < hi; j += 2) {
        auto next = [&]() __attribute__((always_inline)) {
            if (j + 2 < hi) fetch(j + 2, 0);
            if (j + 3 < hi) fetch(j + 3, 1);
        };
        if (j + 1 < hi) group_pass<2, STREAM>(bk, bv, w, dst, &sh[0][0], &sh[1][0], sh_stats, lane, next);
        else group_pass<1, STREAM>(bk, bv, w, dst, &sh[0][0], &sh[1][0], sh_stats, lane, next);
    }
}

// The gradients of the pooled levels out of their partial sums: a workgroup of 1024 threads per unit.  A bf16 partial sum (group-major
// pass) is 16 bytes a thread of 256, an fp32 one (dense pass) of 512: four or two slices of the workgroup take every fourth or every
// second one, four loads in flight a thread, and their sums meet in LDS in slice order, so that the result does not depend on
// scheduling.  The kernel is a few round trips to memory one after the other: with one workgroup of 256 threads a unit and sixteen
// loads in flight it took 17 us at 12 x 16384 tokens (14 now), 110 at 6 x 262144 (102, and 98 past the caches), 53 at 48 x 16384 (45.5); eight loads in
// flight, or 512 threads, 2 to 5 % more.
struct PooledJob {
    const void* part;        // fp32 (f32x4[8][64] a slot) or, with half_part, bf16 (bf16x8[4][64] a slot) partial sums
    int half_part;
    const int* off;          // the partial sums of unit u are slots [off[u] << csr_shift, off[u + 1] << csr_shift) of its (b,h), or ...
    int csr_shift;
    int64_t slot_stride;     // slots per (b,h)
    int n_chunks;            // ... (off == nullptr) this many at stride BH * n_units slots
    int n_units;
    bf16* dk; bf16* dv;      // (B,H,16 n_units,64), contiguous
};
struct PooledJobs {
    PooledJob job[LLSA_MAX_LEVELS];
    int n_jobs;
};
constexpr int kReduceThreads = 1024;
// With STREAM the partial sums are read past the caches: they are read once, and what they push out of the caches the fine pass behind this
// kernel needs.  Few of them push out little.  Training steps, through the caches / past them, us: two levels, 14 x 16384 tokens, 73 MB, 356 / 352;
// 18 x 16384, 94 MB, 442.5 / 432; 24 x 16384 575 / 561; 48 x 16384, 252 MB, 1146 / 1143; 6 x 65536, 133 MB, 686 / 672; 4 x 49152, topk 32, 126 MB,
// 429 / 423; three levels of 262144 704 / 694; 3 x 49152, topk 32, 98 MB, and 6 x 262144 with two (0.5 GB) and three levels (0.6) even.  Below the
// line either may win by a little: 2 x 131072, 67 MB, 457 / 458.5, 12 x 16384, 63 MB, 306 / 304.5, one level of 6 x 16384, 31 MB, 246.5 / 247.4, of
// 4 x 6 x 4096, 31 MB, 163.0 / 163.4, of 8 x 6 x 4096, 31 MB, 266.3 / 265.0, of 64 x 6 x 1024, 25 MB, 439 / 434.
constexpr int64_t kReduceStreamBytes = (int64_t)64 << 20;
template <bool STREAM>
__global__ __launch_bounds__(kReduceThreads, 8) void pooled_reduce_kernel(PooledJobs jobs) {
    __shared__ __align__(16) float sums[3 * 256 * 8];         // of all slices but the first
    // grid.x: the units of all jobs, the coarsest level's first: they have the most partial sums
    int u = blockIdx.x, ji = jobs.n_jobs - 1;
    while (u >= jobs.job[ji].n_units) u -= jobs.job[ji--].n_units;
    const PooledJob& jb = jobs.job[ji];
    const int bh = blockIdx.y, width = jb.half_part ? 256 : 512, slices = kReduceThreads / width;
    const int slice = (int)threadIdx.x / width, pos = (int)threadIdx.x % width;
    int64_t first, stride;
    int n;
    if (jb.off != nullptr) {
        const int* o = jb.off + (int64_t)bh * (jb.n_units + 1) + u;
        const int o0 = o[0];
        n = (o[1] - o0) << jb.csr_shift;
        first = (int64_t)bh * jb.slot_stride + ((int64_t)o0 << jb.csr_shift);
        stride = 1;
    } else {
        n = jb.n_chunks;
        first = (int64_t)bh * jb.n_units + u;
        stride = (int64_t)gridDim.y * jb.n_units;
    }
    constexpr int kBatch = 4;
    f32x4 acc = {0.f, 0.f, 0.f, 0.f}, acc2 = {0.f, 0.f, 0.f, 0.f};
    const i32x4* ps = reinterpret_cast<const i32x4*>(jb.part) + first * width + pos;
    for (int c0 = slice; c0 < n; c0 += kBatch * slices) {
        i32x4 v[kBatch];
#pragma unroll
        for (int k = 0; k < kBatch; k++) {
            const i32x4* at = ps + (int64_t)min(c0 + k * slices, n - 1) * stride * width;
            v[k] = STREAM ? __builtin_nontemporal_load(at) : *at;
        }
#pragma unroll
        for (int k = 0; k < kBatch; k++)
            if (c0 + k * slices < n) {
                if (jb.half_part) {
                    const bf16x8 x = __builtin_bit_cast(bf16x8, v[k]);
                    acc += f32x4{(float)x[0], (float)x[1], (float)x[2], (float)x[3]};
                    acc2 += f32x4{(float)x[4], (float)x[5], (float)x[6], (float)x[7]};
                } else {
                    acc += __builtin_bit_cast(f32x4, v[k]);
                }
            }
    }
    if (slice > 0) {
        f32x4* dst = reinterpret_cast<f32x4*>(sums);
        dst[(slice - 1) * width + pos] = acc;
        if (jb.half_part) dst[(3 + slice - 1) * width + pos] = acc2;
    }
    __syncthreads();
    if (slice > 0) return;
    const f32x4* src = reinterpret_cast<const f32x4*>(sums);
    for (int i = 0; i + 1 < slices; i++) {
        acc += src[i * width + pos];
        if (jb.half_part) acc2 += src[(3 + i) * width + pos];
    }
    const int lane = pos & 63, r = lane & 15, quad = lane >> 4, reg = jb.half_part ? 2 * (pos >> 6) : pos >> 6;       // (bf16: registers reg, reg + 1)
    const int dt = reg & 3;
    const bool is_k = reg < 4;
    bf16* dst = (is_k ? jb.dk : jb.dv) + (((int64_t)bh * jb.n_units + u) * kBlk + r) * kD + dt * 16 + quad * 4;
    st8(dst, cvt4(is_k ? acc * kScale : acc));
    if (jb.half_part) st8(dst + 16, cvt4(is_k ? acc2 * kScale : acc2));
}

// Finishes the fine units whose list was cut into several pieces: the result is the sum of the
// unit's fp32 partial slots, added in piece order, so it does not depend on scheduling.
struct ReduceParams {
    const f32x4* part;
    const int* work;         // work list
    bf16* dk; int64_t sdkb, sdkh, sdkn;
    bf16* dv; int64_t sdvb, sdvh, sdvn;
    int n_units, max_units, H, N;        // max_units: upper bound of units that can have several pieces per (b,h)
    int64_t work_stride, slot_stride;
    PoolFold fold;
    llsa_norm_back norm;     // the norm of k (x: nullptr without)
};

// Unit positions per (b,h) that are walked in parallel: a quarter of the most units there can be,
// between 32 and 256.  Usually a few per cent of the units have several pieces, and every position beyond
// them is a pair of workgroups that starts, reads one record and leaves (at 256 positions for a job of at
// most 257 units that cost 4 us per launch).
__host__ __device__ inline int reduce_slots(int max_units) {
    if (max_units <= 32) return max_units;
    const int q = max_units / 4;
    return q < 32 ? 32 : (q > 256 ? 256 : q);
}

__global__ __launch_bounds__(256) void kside_reduce_kernel(ReduceParams p) {
    // Two workgroups per unit (dK, dV); every thread owns one f32x4 of the unit's 8 x 64 accumulator registers and streams that
    // position of all partials, sixteen loads in flight.  The workgroups (reduce_slots pairs of them) walk the units with that
    // stride: the number of units with several pieces is known only on the device and usually small, and a grid sized for the worst
    // case would be mostly workgroups that start, look and leave.
    __shared__ float row_ss[4][kBlk], row_dot[4][kBlk];
    const int bh = blockIdx.y, b = bh / p.H, h = bh % p.H;
    const int u0 = blockIdx.x >> 1;
    const int which = blockIdx.x & 1;                         // 0: dK, 1: dV
    const int dt = (int)(threadIdx.x >> 6), lane = (int)(threadIdx.x & 63);
    const int r = lane & 15, quad = lane >> 4;
    const int step = reduce_slots(p.max_units);
    const int* work = p.work + (int64_t)bh * p.work_stride;
    const int max_items = (int)(p.work_stride - work_tail_len(p.n_units) - 4 - 4 * p.max_units) / 4;
    // the unit's record is fetched together with the count it is checked against (u0 is always
    // inside the list's storage): one memory round trip instead of two
    const int* multi = work + 4 + 4 * max_items;
    int rec_unit = multi[4 * u0], rec_first = multi[4 * u0 + 1], rec_n = multi[4 * u0 + 2];
    const int count = min(work[2], p.max_units);
    for (int u = u0; u < count; u += step) {
        if (u != u0) {
            rec_unit = multi[4 * u];
            rec_first = multi[4 * u + 1];
            rec_n = multi[4 * u + 2];
        }
        const int unit = rec_unit, n = rec_n;
        const int64_t first = (int64_t)bh * p.slot_stride + rec_first;
        f32x4 acc = {0.f, 0.f, 0.f, 0.f};
        const f32x4* ps = p.part + first * (8 * kWave) + (4 * which + dt) * kWave + lane;
        for (int c0 = 0; c0 < n; c0 += 16) {
            f32x4 v[16];
#pragma unroll
            for (int k = 0; k < 16; k++) v[k] = ps[(int64_t)min(c0 + k, n - 1) * (8 * kWave)];
#pragma unroll
            for (int k = 0; k < 16; k++)
                if (c0 + k < n) acc += v[k];
        }
        bf16* dst = which ? p.dv + b * p.sdvb + h * p.sdvh + (int64_t)(unit * kBlk + r) * p.sdvn
                          : p.dk + b * p.sdkb + h * p.sdkh + (int64_t)(unit * kBlk + r) * p.sdkn;
        bf16x4 out = cvt4(which ? acc : acc * kScale);
        if (p.fold.depth > 0)
            out = fold_pooled(out, p.fold, which, bh, p.N, unit * kBlk + r, dt * 16 + quad * 4);
        if (p.norm.x != nullptr && which == 0) {              // (uniform over the workgroup)
            // wave dt holds channels 16 dt .. of the unit's rows: norm_back with the sums over a row's channels through LDS
            const llsa_norm_back& nb = p.norm;
            const int c0 = dt * 16 + quad * 4;
            const bf16x4 x = ld8((const bf16*)nb.x + b * nb.sxb + h * nb.sxh + (int64_t)(unit * kBlk + r) * nb.sxn + c0);
            const f32x4 gamma = {nb.gamma[c0], nb.gamma[c0 + 1], nb.gamma[c0 + 2], nb.gamma[c0 + 3]};
            float ss = 0.f, dot = 0.f;
#pragma unroll
            for (int e = 0; e < 4; e++) {
                ss += (float)x[e] * (float)x[e];
                dot += (float)out[e] * gamma[e] * (float)x[e];
            }
            ss = quad_sum(ss);
            dot = quad_sum(dot);
            __syncthreads();                                  // (the previous unit's sums have been read)
            if (quad == 0) {
                row_ss[dt][r] = ss;
                row_dot[dt][r] = dot;
            }
            __syncthreads();
            const float rstd = rsqrtf(((row_ss[0][r] + row_ss[1][r]) + (row_ss[2][r] + row_ss[3][r])) * (1.f / kD) + nb.eps);
            dot = ((row_dot[0][r] + row_dot[1][r]) + (row_dot[2][r] + row_dot[3][r])) * rstd * (1.f / kD);
            f32x4 contrib;
#pragma unroll
            for (int e = 0; e < 4; e++) {
                contrib[e] = (float)out[e] * (float)x[e] * rstd;
                out[e] = (bf16)(rstd * ((float)out[e] * gamma[e] - (float)x[e] * rstd * dot));
            }
#pragma unroll
            for (int d = 1; d < 16; d <<= 1)
#pragma unroll
                for (int e = 0; e < 4; e++) contrib[e] += __shfl_xor(contrib[e], d);
            if (r == 0) *reinterpret_cast<f32x4*>(nb.partials + ((int64_t)bh * p.n_units + unit) * kD + c0) = contrib;
        }
        st8(dst + quad * 4 + dt * 16, out);
    }
}

// The weights' gradients of the norms: dgamma = column sums of the rows of partial sums.  Two launches for both norms (blockIdx.y):
// workgroup x of X adds rows x, x + X, ... of `in` into row x of `out`, then one workgroup adds those.  With out == in a
// workgroup overwrites a row that only it has read.
struct NormSums {
    const float* in[2]; float* out[2];
    int64_t rows[2];
};
__global__ __launch_bounds__(1024) void norm_sums_kernel(NormSums p) {
    __shared__ float red[16][kD];
    const int ch = threadIdx.x & 63, j = threadIdx.x >> 6;
    const float* in = p.in[blockIdx.y];
    float s = 0.f;
#pragma unroll 4
    for (int64_t r = blockIdx.x + (int64_t)j * gridDim.x; r < p.rows[blockIdx.y]; r += 16 * (int64_t)gridDim.x) s += in[r * kD + ch];
    red[j][ch] = s;
    __syncthreads();
    if (j == 0) {
#pragma unroll
        for (int k = 1; k < 16; k++) s += red[k][ch];
        p.out[blockIdx.y][(int64_t)blockIdx.x * kD + ch] = s;
    }
}

struct DensePlan {
    int n_tok;       // tokens of the dense coarsest level per (b,h)
    int wg_units;    // units per workgroup: 16 (eight waves of two), 8 (four waves of two) or 4 (four waves of one)
    int chunks;      // query range split
    int chunk_len;   // query blocks per chunk (a multiple of 4)
    bool merged;     // the dense blocks ride on the group-major pass (one partial sum per group of 16 query blocks)
};

static DensePlan dense_plan(int B, int H, int N, int levels) {
    const int N1 = N / 16;
    DensePlan d;
    d.n_tok = N1;                                             // tokens of pooled level `levels`
    for (int l = 1; l < levels; l++) d.n_tok /= 16;
    const int n_units = d.n_tok / 16;
    // Eight waves of two units, unless their last workgroup would be at most half full and there are few of them (N = 5120, 12
    // heads: 20 units as two workgroups of sixteen 19.8 us, as three of eight 18.5; 28 units, N = 7168: 32 against 35 us).
    const int last = n_units % 16;
    d.wg_units = n_units < 16 ? 4 : (last == 0 || last > 8 || n_units > 64 ? 16 : 8);
    const int groups = (n_units + d.wg_units - 1) / d.wg_units * B * H;   // workgroups per piece of the query range
    // The query range is cut so that the workgroups fill the chip's resident slots (256 CUs x the workgroups the
    // registers allow per CU) a whole number of times: a count just above a multiple of the slots leaves a last round in
    // which a few workgroups run alone.  Once, for the fewest partial sums; where the pieces are long and once leaves more than a
    // fifth of the slots empty, twice or three times.  Training steps cut for one / two / three rounds, us, in brackets how full:
    //   4 x 8 x 16384 1078 (1.00) / 1090 / 1104;  8 x 32768 788 (1.00) / 796 / 807;  3 x 49152 693 (.98) / 701 / 711;  2 x 65536 769 (1.00) / 777 / 788
    //   3 x 6 x 16384 630 (.84) / 637 (.98) / 651 (.94);  7 x 65536 2350 (.88) / 2364 / 2384;  two levels: 8 x 131072 1666 (1.00) / 1675 / 1691
    //   3 x 262144 2031 (.98) / 2046 / 2043;  6 x 262144 even;  but 4 x 6 x 16384 743 (.75) / 738 (.94) / 745 (1.00);  6 x 65536 2129 (.75) / 2037 (.94) /
    //   2041 (1.00);  5 x 8 x 16384 1256 (.62) / 1200 (.94) / 1228 (.83);  8 x 6 x 16384 1460 (.75) / 1476 (.75) / 1441 (1.00)
    //   short pieces: 3 x 5 x 7168 191 (.94) / 197 / 205;  4 x 6 x 4096 162.5 (.94) / 169 / 169
    const int slots = 256 * (d.wg_units == 16 ? 1 : d.wg_units == 8 ? 2 : 3);
    int chunks = slots / groups;
    for (int rounds = 2; rounds <= 3 && (chunks < 1 || (N1 / chunks > 256 && (int64_t)chunks * groups * 5 < (int64_t)(rounds - 1) * slots * 4)); rounds++)
        chunks = rounds * slots / groups;
    if (chunks > N1 / 16) chunks = N1 / 16;
    if (chunks < 1) chunks = 1;
    int len = (N1 + chunks - 1) / chunks;
    len = (len + 3) & ~3;
    d.chunk_len = len;
    d.chunks = (N1 + len - 1) / len;
    d.merged = levels >= 2 && n_units <= kGroupDenseMax;
    if (d.merged) {
        d.chunks = N1 / 16;
        d.chunk_len = 16;
    }
    return d;
}

// A pooled level whose lists belong to `owners` ancestors of `range` query blocks each (a power of 16): into how many pieces, as a power of
// two, the list form of the dense kernel cuts every owner's range, or -1 for the group-major pass.  The list form leaves one partial
// sum per piece, in fp32, where the other leaves one per 16 query blocks, in bf16; but its workgroup is sixteen entries and a whole CU: it is taken
// for full workgroups, three rounds of the chip and pieces of 128 query blocks or more.  Both passes and the reduction, us, group-major / list
// (llsa_l3 at 262144 tokens): 6 heads, T3 = 16: 724 / 682; 12 heads: 1374 / 1273; but 2 heads (512 workgroups) 284 / 291, 3 heads with T3 = 12
// 294 / 318, one head with T3 = 20 170 / 186.
static int list_chunk_shift(int BH, int owners, int range, int T) {
    constexpr int kMinWorkgroups = 3 * 256, kMinPiece = 128;
    if (range < kMinPiece || T % 16 != 0) return -1;
    const int64_t lists = (int64_t)BH * owners * (T / 16);
    int shift = 0;
    while ((lists << shift) < kMinWorkgroups && (range >> shift) > kMinPiece) shift++;
    return (lists << shift) >= kMinWorkgroups ? shift : -1;
}

static int64_t align256(int64_t x) { return (x + 255) & ~(int64_t)255; }
constexpr int64_t kSlotBytes = 8 * kWave * sizeof(f32x4);     // one partial: 16 rows x 64 ch x (dK, dV) fp32

struct BwdWorkspace {
    int64_t stats, dor, part_fine, part_dense, total;
    int64_t part_level[LLSA_MAX_LEVELS];                        // partial sums of pooled level l (below the coarsest) at [l - 1]
    int64_t slots_fine, slots_level[LLSA_MAX_LEVELS];           // per (b,h)
};

// topk[0] = T of the fine blocks, topk[l] = T of pooled level l (l < levels)
static BwdWorkspace bwd_workspace(int B, int H, int N, const int32_t* topk, int levels) {
    const int64_t BH = (int64_t)B * H, N1 = N / 16, N2 = N1 / 16;
    const DensePlan d = dense_plan(B, H, N, levels);
    BwdWorkspace w;
    // a key block has several chunks only if it has more than `chunk` entries, so at most
    // E/chunk such blocks with at most E/chunk + E/chunk chunks in total (fine_chunk_for: the shortest chunk a call may use)
    w.slots_fine = 2 * (N1 * topk[0] / fine_chunk_for(BH, N, topk[0])) + 2;
    int64_t o = 0;
    w.stats = o;        o += align256(BH * N / kBlk * kStats * 4);
    w.dor = o;          o += align256(BH * N * 64 * 2);
    w.part_fine = o;    o += align256(BH * w.slots_fine * kSlotBytes);
    // group-major pooled passes: one partial sum per (group of 16 query blocks, entry of its ancestor's list)
    for (int l = 1; l <= LLSA_MAX_LEVELS; l++) {
        w.slots_level[l - 1] = (l < levels) ? N2 * topk[l] : 0;
        w.part_level[l - 1] = o;
        o += align256(BH * w.slots_level[l - 1] * kSlotBytes);
    }
    w.part_dense = o;   o += align256((int64_t)d.chunks * BH * (d.n_tok / 16) * kSlotBytes);
    w.total = o;
    return w;
}

}  // namespace llsa

using namespace llsa;

extern "C" int64_t llsa_attn_bwd_workspace_bytes(int B, int H, int N, const int32_t* topk, int levels) {
    if (B <= 0 || H <= 0 || N <= 0 || topk == nullptr || levels < 1 || levels > LLSA_MAX_LEVELS) return -1;
    if (N % coarsest_multiple(levels) != 0) return -1;       // what llsa_attn_bwd asks of N: whole 64-token tiles of the coarsest level
    for (int l = 0; l < levels; l++)
        if (topk[l] <= 0) return -1;
    return bwd_workspace(B, H, N, topk, levels).total;
}

extern "C" int llsa_attn_bwd(const llsa_attn_bwd_args* a, void* stream) {
    LLSA_REQUIRE(a != nullptr, "attn_bwd: null args");
    LLSA_REQUIRE(a->levels >= 1 && a->levels <= LLSA_MAX_LEVELS, "attn_bwd: levels must be 1..%d", LLSA_MAX_LEVELS);
    LLSA_REQUIRE(a->B > 0 && a->H > 0 && a->N > 0, "attn_bwd: bad B/H/N");
    LLSA_REQUIRE(a->dout && a->o && a->lse && a->qr && a->kr && a->vr && a->idx && a->off && a->flat && a->dq && a->dk && a->dv &&
                     a->workspace,
                 "attn_bwd: null tensor");
    LLSA_REQUIRE(a->T >= 4 && a->T % 4 == 0 && a->T <= a->N / 16, "attn_bwd: topk=%d must be a multiple of 4 and <= N/16", a->T);
    const int64_t mult = coarsest_multiple(a->levels);
    LLSA_REQUIRE(a->N % mult == 0, "attn_bwd: %d level(s) need N %% %lld == 0 (N=%d)", a->levels, (long long)mult, a->N);
    int32_t topk[LLSA_MAX_LEVELS] = {a->T, 0, 0, 0};
    int listed = 0;
    int64_t span = 256;
    for (int l = 1; l <= a->levels; l++, span *= 16) {
        const llsa_bwd_level& lv = a->lvl[l - 1];
        LLSA_REQUIRE(lv.kr && lv.vr && lv.dk && lv.dv, "attn_bwd: tensors of level %d missing", l);
        LLSA_REQUIRE(aligned16(lv.kr) && aligned16(lv.vr) && aligned16(lv.dk) && aligned16(lv.dv), "attn_bwd: tensors must be 16-byte aligned");
        LLSA_REQUIRE(lv.w > 0.f && lv.gw > 0.f, "attn_bwd: the weights of level %d must be > 0", l);
        if (l < a->levels) {
            LLSA_REQUIRE(lv.sel && lv.off && lv.inv, "attn_bwd: selection of level %d or its transpose missing", l);
            LLSA_REQUIRE(lv.T >= 4 && lv.T % 4 == 0 && lv.T <= a->N / span, "attn_bwd: topk of level %d (%d) must be a multiple of 4 and <= N/%lld",
                         l, lv.T, (long long)span);
            topk[l] = lv.T;
            listed += lv.T;
        }
    }
    LLSA_REQUIRE(listed <= LLSA_POOLED_TOPK_MAX, "attn_bwd: the topk of the pooled levels together (%d) must not exceed %d", listed,
                 LLSA_POOLED_TOPK_MAX);
    const void* al[] = {a->dout, a->o, a->qr, a->kr, a->vr, a->dq, a->dk, a->dv, a->workspace, a->freq_dq, a->lse};
    for (const void* p : al) LLSA_REQUIRE(aligned16(p), "attn_bwd: tensors must be 16-byte aligned");
    const int64_t st[] = {a->sdob, a->sdoh, a->sdon, a->sob, a->soh, a->son};
    for (int64_t s : st) LLSA_REQUIRE(stride_ok(s), "attn_bwd: input row strides must keep rows 16-byte aligned");
    const int64_t so[] = {a->sdqb, a->sdqh, a->sdqn, a->sdkb, a->sdkh, a->sdkn, a->sdvb, a->sdvh, a->sdvn};
    for (int64_t s : so) LLSA_REQUIRE(s % 4 == 0, "attn_bwd: output row strides must keep rows 8-byte aligned");
    const BwdWorkspace wsp = bwd_workspace(a->B, a->H, a->N, topk, a->levels);
    LLSA_REQUIRE(a->workspace_bytes >= wsp.total, "attn_bwd: workspace too small (%lld < %lld)", (long long)a->workspace_bytes,
                 (long long)wsp.total);
    LLSA_REQUIRE(a->work != nullptr, "attn_bwd: work list missing");
    const int chunk_fine = a->chunk != 0 ? a->chunk : fine_chunk(a->N), least_chunk = fine_chunk_for((int64_t)a->B * a->H, a->N, a->T);
    LLSA_REQUIRE(chunk_fine >= least_chunk && chunk_fine <= LLSA_CHUNK_FINE_MAX, "attn_bwd: chunk=%d must be in %d..%d", chunk_fine, least_chunk,
                 LLSA_CHUNK_FINE_MAX);

    hipStream_t s = (hipStream_t)stream;
    const int B = a->B, H = a->H, N = a->N, N1 = N / 16, N2 = N1 / 16, BH = B * H, L = a->levels;
    const DensePlan d = dense_plan(B, H, N, L);
    char* ws = (char*)a->workspace;
    float* stats = (float*)(ws + wsp.stats);
    bf16* dor = (bf16*)(ws + wsp.dor);
    const bool fold = a->fold_pooled != 0;
    LLSA_REQUIRE(fold || a->freq_dk == nullptr, "attn_bwd: freq_dk needs fold_pooled");
    LLSA_REQUIRE(fold || a->norm_k.x == nullptr, "attn_bwd: norm_k needs fold_pooled");
    for (const llsa_norm_back* nb : {&a->norm_q, &a->norm_k}) {
        if (nb->x == nullptr) continue;
        LLSA_REQUIRE(nb->gamma && nb->dgamma && nb->partials && nb->eps >= 0.f, "attn_bwd: norm without gamma, dgamma or partials");
        LLSA_REQUIRE(aligned16(nb->x) && stride_ok(nb->sxb) && stride_ok(nb->sxh) && stride_ok(nb->sxn) && aligned16(nb->partials),
                     "attn_bwd: rows of the norm's input must be 16-byte aligned");
    }
    NormSums sums;
    int n_sums = 0;

    const int stages = a->stages ? a->stages : (0x7fffffff & ~LLSA_BWD_NO_REDUCE);
    if (stages & LLSA_BWD_DQ) {
        const bool pairs = two_blocks_per_wave(BH, N, topk, L, false);
        const dim3 grid(N1 / (pairs ? 8 : 4), BH);
#define LLSA_DQ(Q, R)                                                                                                                  \
    do {                                                                                                                               \
        if (a->norm_q.x) hipLaunchKernelGGL(HIP_KERNEL_NAME(attn_dq_kernel<Q, R, true>), grid, dim3(256), 0, s, *a, stats, dor);       \
        else hipLaunchKernelGGL(HIP_KERNEL_NAME(attn_dq_kernel<Q, R, false>), grid, dim3(256), 0, s, *a, stats, dor);                  \
    } while (0)
        if (!pairs) LLSA_DQ(1, 1);
        else if (a->T <= 32) LLSA_DQ(2, 1);
        else LLSA_DQ(2, 2);
#undef LLSA_DQ
        if (a->norm_q.x) {
            sums.in[n_sums] = a->norm_q.partials;
            sums.out[n_sums] = a->norm_q.dgamma;
            sums.rows[n_sums++] = (int64_t)grid.x * BH;
        }
    }

    PooledJobs pooled;
    pooled.n_jobs = 0;
    PoolFold no_fold;
    for (int l = 0; l < LLSA_MAX_LEVELS; l++) no_fold.gk[l] = no_fold.gv[l] = nullptr;
    no_fold.freq = nullptr;
    no_fold.depth = 0;
    // the finished gradients of the pooled levels
    auto reduce_pooled = [&]() {
        if (pooled.n_jobs == 0 || (stages & LLSA_BWD_NO_REDUCE)) return;     // (profiling: time the K-side kernels alone)
        int units = 0;
        int64_t bytes = 0;
        for (int i = 0; i < pooled.n_jobs; i++) {
            const PooledJob& j = pooled.job[i];
            units += j.n_units;
            bytes += BH * (j.off != nullptr ? j.slot_stride : (int64_t)j.n_chunks * j.n_units) * (j.half_part ? kSlotBytes / 2 : kSlotBytes);
        }
        if (bytes > kReduceStreamBytes) hipLaunchKernelGGL(pooled_reduce_kernel<true>, dim3(units, BH), dim3(kReduceThreads), 0, s, pooled);
        else hipLaunchKernelGGL(pooled_reduce_kernel<false>, dim3(units, BH), dim3(kReduceThreads), 0, s, pooled);
    };
    KSideParams base;
    base.qr = (const bf16*)a->qr; base.dor = dor;
    base.stats = stats;
    base.H = H; base.N = N; base.chunk_len = 0;
    base.fold = no_fold;
    base.norm = llsa_norm_back{};
    // pooled level l: N / 16^l tokens per (b,h), contiguous (B,H,n,64) gradients
    auto level_tokens = [&](int l) {
        int n = N;
        for (int i = 0; i < l; i++) n /= 16;
        return n;
    };

    auto run_fine = [&]() {                                   // dK / dV of the fine tokens
        if (!(stages & LLSA_BWD_DKV)) return;
        KSideParams p = base;
        p.kk = (const bf16*)a->kr; p.vv = (const bf16*)a->vr;
        p.off = a->off; p.flat = a->flat; p.flat_stride = (int64_t)N1 * a->T;
        const int chunk = chunk_fine;
        p.work = a->work; p.work_stride = llsa_work_list_len(N1, N1, a->T, chunk);
        p.part = (f32x4*)(ws + wsp.part_fine); p.slot_stride = wsp.slots_fine;
        p.dk = (bf16*)a->dk; p.sdkb = a->sdkb; p.sdkh = a->sdkh; p.sdkn = a->sdkn;
        p.dv = (bf16*)a->dv; p.sdvb = a->sdvb; p.sdvh = a->sdvh; p.sdvn = a->sdvn;
        p.n_units = N1; p.w = 1.f;
        if (fold) {
            for (int l = 0; l < L; l++) {
                p.fold.gk[l] = (const bf16*)a->lvl[l].dk;
                p.fold.gv[l] = (const bf16*)a->lvl[l].dv;
            }
            p.fold.freq = (const bf16*)a->freq_dk;
            p.fold.depth = L;
        }
        const int max_items = N1 * a->T / chunk + N1;
        int g = 8;                                            // gcd(BH, 8)
        while (BH % g != 0) g /= 2;
        p.stripes = kXcds / g;
        p.stripe_len = max_items / p.stripes + 2;             // ceil(long / stripes) + ceil(short / stripes) at most
        p.norm = a->norm_k;
        const dim3 grid((unsigned)(p.stripe_len * p.stripes * BH));
        if (p.norm.x) {
            hipLaunchKernelGGL(HIP_KERNEL_NAME(attn_kside_kernel<true>), grid, dim3(64), 0, s, p);
            sums.in[n_sums] = p.norm.partials;
            sums.out[n_sums] = p.norm.dgamma;
            sums.rows[n_sums++] = (int64_t)N1 * BH;
        } else {
            hipLaunchKernelGGL(HIP_KERNEL_NAME(attn_kside_kernel<false>), grid, dim3(64), 0, s, p);
        }
        if (stages & LLSA_BWD_NO_REDUCE) return;
        ReduceParams r;
        r.part = p.part; r.work = p.work;
        r.dk = p.dk; r.sdkb = p.sdkb; r.sdkh = p.sdkh; r.sdkn = p.sdkn;
        r.dv = p.dv; r.sdvb = p.sdvb; r.sdvh = p.sdvh; r.sdvn = p.sdvn;
        r.n_units = p.n_units; r.max_units = N1 * a->T / chunk + 1; r.H = H; r.N = N;
        r.work_stride = p.work_stride; r.slot_stride = p.slot_stride;
        r.fold = p.fold;
        r.norm = p.norm;
        hipLaunchKernelGGL(kside_reduce_kernel, dim3(2 * reduce_slots(r.max_units), BH), dim3(256), 0, s, r);
    };
    // pooled levels under an ancestor's selection, group-major (one launch for all of them, plus the dense level when it is small)
    auto run_groups = [&]() {
        if (L < 2 || !(stages & LLSA_BWD_DPKV1)) return;
        GroupParams g;
        g.qr = (const bf16*)a->qr; g.dor = dor; g.stats = stats;
        g.BH = BH; g.N = N; g.n_segs = 0; g.n_blocks = 0;
        auto add_seg = [&](const void* kk, const void* vv, const int* sel, const int* inv, int64_t part_off, int n_units, int shift,
                           int cnt, int64_t slots, float w) {
            GroupSeg& sgm = g.seg[g.n_segs++];
            sgm.kk = (const bf16*)kk; sgm.vv = (const bf16*)vv; sgm.sel = sel; sgm.inv = inv;
            sgm.part = (bf16x8*)(ws + part_off); sgm.n_units = n_units; sgm.owner_shift = shift; sgm.cnt = cnt; sgm.slots = slots; sgm.w = w;
            g.n_blocks += cnt;
        };
        for (int l = 1; l < L; l++) {                         // level l: blocks N / 16^(l+1), one list per 16^(l-1) groups
            const llsa_bwd_level& lv = a->lvl[l - 1];
            PooledJob& j = pooled.job[pooled.n_jobs++];
            j.part = ws + wsp.part_level[l - 1]; j.off = lv.off; j.n_chunks = 0; j.n_units = level_tokens(l + 1);
            j.dk = (bf16*)lv.dk; j.dv = (bf16*)lv.dv;
            const int owners = N2 >> (4 * (l - 1)), shift = list_chunk_shift(BH, owners, N1 / owners, lv.T);
            j.half_part = shift < 0;
            j.csr_shift = shift < 0 ? 4 * (l - 1) : shift;
            j.slot_stride = shift < 0 ? wsp.slots_level[l - 1] : (int64_t)owners * lv.T << shift;
            if (shift < 0) {
                add_seg(lv.kr, lv.vr, lv.sel, lv.inv, wsp.part_level[l - 1], j.n_units, j.csr_shift, lv.T, j.slot_stride, lv.gw);
                continue;
            }
            KSideParams p = base;
            p.kk = (const bf16*)lv.kr; p.vv = (const bf16*)lv.vr; p.w = lv.gw;
            p.off = nullptr; p.flat = nullptr; p.flat_stride = 0; p.work = nullptr; p.work_stride = 0; p.slot_stride = j.slot_stride;
            p.part = (f32x4*)(ws + wsp.part_level[l - 1]); p.n_units = j.n_units; p.chunk_len = (N1 / owners) >> shift;
            const dim3 grid(lv.T / 16 * (owners << shift), BH);
            hipLaunchKernelGGL(HIP_KERNEL_NAME(attn_kside_dense_kernel<8, 2, true>), grid, dim3(512), 0, s, p,
                               KSideLists{lv.sel, lv.inv, lv.T, shift});
        }
        if (d.merged && (stages & LLSA_BWD_DENSE))
            add_seg(a->lvl[L - 1].kr, a->lvl[L - 1].vr, nullptr, nullptr, wsp.part_dense, d.n_tok / 16, 0, d.n_tok / 16, 0, a->lvl[L - 1].gw);
        const int64_t bytes = (int64_t)BH * N2 * g.n_blocks * (kSlotBytes / 2);
        const int per_xcd = N2 * BH / kXcds;                  // (two levels need N2 to be a multiple of 64)
        const GroupSplit split = group_split(per_xcd, g.n_blocks);
        g.whole = split.whole;
        g.parts = split.parts;
        const dim3 grid((unsigned)(kXcds * (split.whole + (per_xcd - split.whole) * split.parts)));
        if (bytes > kGroupStreamBytes && g.n_blocks >= kGroupStreamBlocks) hipLaunchKernelGGL(attn_kside_group_kernel<true>, grid, dim3(64 * kGroupWaves), 0, s, g);
        else hipLaunchKernelGGL(attn_kside_group_kernel<false>, grid, dim3(64 * kGroupWaves), 0, s, g);
    };
    // dense coarsest level: every unit (16 pooled tokens) meets every query block; the query
    // range is cut into d.chunks pieces whose partial sums are added afterwards
    auto run_dense = [&]() {
        if (!(stages & LLSA_BWD_DENSE)) return;
        KSideParams p = base;
        const llsa_bwd_level& lv = a->lvl[L - 1];
        p.kk = (const bf16*)lv.kr; p.vv = (const bf16*)lv.vr;
        p.w = lv.gw;
        p.off = nullptr; p.flat = nullptr; p.flat_stride = 0; p.work = nullptr; p.work_stride = 0; p.slot_stride = 0;
        p.part = (f32x4*)(ws + wsp.part_dense);
        p.n_units = d.n_tok / 16; p.chunk_len = d.chunk_len;
        PooledJob& j = pooled.job[pooled.n_jobs++];           // (merged: the group-major pass has written one bf16 partial sum per group)
        j.part = p.part; j.half_part = d.merged; j.off = nullptr; j.csr_shift = 0; j.slot_stride = 0;
        j.n_chunks = d.chunks; j.n_units = p.n_units;
        j.dk = (bf16*)lv.dk; j.dv = (bf16*)lv.dv;
        if (d.merged) return;
        const dim3 grid((p.n_units + d.wg_units - 1) / d.wg_units * d.chunks, BH);
        const KSideLists none{nullptr, nullptr, 0, 0};
        if (d.wg_units == 16) hipLaunchKernelGGL(HIP_KERNEL_NAME(attn_kside_dense_kernel<8, 2, false>), grid, dim3(512), 0, s, p, none);
        else if (d.wg_units == 8) hipLaunchKernelGGL(HIP_KERNEL_NAME(attn_kside_dense_kernel<4, 2, false>), grid, dim3(256), 0, s, p, none);
        else hipLaunchKernelGGL(HIP_KERNEL_NAME(attn_kside_dense_kernel<4, 1, false>), grid, dim3(256), 0, s, p, none);
    };

    if (fold) {
        // the fine pass adds the finished pooled gradients on its way out, so they come first
        run_groups();
        run_dense();
        reduce_pooled();
        run_fine();
    } else {
        run_fine();
        run_groups();
        run_dense();
        reduce_pooled();
    }
    if (n_sums > 0) {
        // (rows of the first stage's results: at most as many as there are rows)
        constexpr int kSumGroups = 128;
        NormSums first = sums;
        int groups = kSumGroups;
        for (int i = 0; i < n_sums; i++) {
            first.out[i] = const_cast<float*>(sums.in[i]);
            groups = (int)std::min<int64_t>(groups, sums.rows[i]);
        }
        hipLaunchKernelGGL(norm_sums_kernel, dim3(groups, n_sums), dim3(1024), 0, s, first);
        for (int i = 0; i < n_sums; i++) sums.rows[i] = groups;
        hipLaunchKernelGGL(norm_sums_kernel, dim3(1, n_sums), dim3(1024), 0, s, sums);
    }
    return launch_status("attn_bwd");
}
