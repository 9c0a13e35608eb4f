// Block selection: dense coarsest-level top-k and parent-guided fine top-k.
//
// A tile of 16 pooled queries is scored against 16-key tiles with the bf16 MFMA in the S^T orientation: lane l gets the
// scores of query l%16, so a query's scores live in the registers of four lanes (l, l^16, l^32, l^48) and never leave
// them.  All sixteen rows of a wave are selected side by side: bisection narrows every row down to a few more than its T
// best keys -- a compare and an add-with-carry per score and step and two lane swaps per step for the row's count --, and
// those are ranked among each other in LDS.  (One row per wave at a time, spread over the 64 lanes with a ballot and a
// scalar population count per score, issues about three times the instructions per row and step, half of them on the one
// scalar unit.  Bisecting down to exactly T keys takes 20 to 30 steps instead of 2 to 5: the T-th and the next best key of
// the worst of sixteen rows agree in most of their bits.)
//
// The order is total -- higher score first, equal scores by smaller key index -- so the result does not depend on how the
// work is split.
#include <algorithm>
#include "llsa_device.h"
#include "llsa_host.h"
#include "../../include/llsa_hip.h"

namespace llsa {

constexpr int kMaxT = 64;        // largest supported top-k
constexpr int kMaxCand = 512;    // candidates per parent in the sparse kernel (T2 * 16)

// Any score, any index: the same order in 64 bits.
__device__ __forceinline__ unsigned long long wide_key(unsigned score_key, int idx) {
    return ((unsigned long long)score_key << 32) | (unsigned)(0x7FFFFFFF - idx);
}

// sum / largest / smallest over the four lanes that share a query
__device__ __forceinline__ int quad_sum_i(int v) {
    u32x2 a = __builtin_amdgcn_permlane16_swap((unsigned)v, (unsigned)v, false, false);
    const unsigned w = a[0] + a[1];
    u32x2 b = __builtin_amdgcn_permlane32_swap(w, w, false, false);
    return (int)(b[0] + b[1]);
}
__device__ __forceinline__ unsigned quad_max_u(unsigned v) {
    u32x2 a = __builtin_amdgcn_permlane16_swap(v, v, false, false);
    const unsigned w = max(a[0], a[1]);
    u32x2 b = __builtin_amdgcn_permlane32_swap(w, w, false, false);
    return max(b[0], b[1]);
}
__device__ __forceinline__ unsigned quad_min_u(unsigned v) { return ~quad_max_u(~v); }
__device__ __forceinline__ unsigned long long quad_max_u(unsigned long long v) {
    const unsigned hi = quad_max_u((unsigned)(v >> 32));
    const unsigned lo = quad_max_u((unsigned)(v >> 32) == hi ? (unsigned)v : 0u);
    return ((unsigned long long)hi << 32) | lo;
}

// Where a lane's two pieces of sixteen keys are: in rows of 64 channels, or in an R tile, which is the same sixteen keys in the same place in
// the order the lanes read them.  Out of rows each of the 64 pieces of a load is an access of its own in the L1, whose rate the selection of
// long rows then runs at; out of tiles a load is one contiguous kilobyte: 8 x 4096 rows
// of 4096 keys, T = 8, 71.5 -> 48.9 us; 6 x 1024 of 1024, in registers, 19.3 -> 14.6; 24 x 256 8.2 -> 7.0; parent-guided, 6 x 16384 rows, 54.4 -> 49.3.
struct KeyPieces {
    int first, second;                                        // elements from the sixteen keys' start
    __device__ __forceinline__ KeyPieces(int tiled, int lane)
        : first(tiled ? lane * 8 : (lane & 15) * kD + (lane >> 4) * 8), second(first + (tiled ? kTile / 2 : kD / 2)) {}
};

// S^T tiles: rows = 16 keys starting at row_of(a) * kD elements into `keys`, columns = the wave's 16 queries (bq).  Lane l
// gets the scores of query l%16 against keys 4*(l/16) .. +3 of tile a.  No branch around the loads, so that they are all in
// flight together: the caller clamps the rows of tiles that do not exist and drops their scores.
template <int TILES, typename RowOf>
__device__ __forceinline__ void score_tiles(f32x4 (&s)[TILES], const bf16* keys, RowOf row_of, const bf16x8 bq[2], const KeyPieces& pieces) {
    constexpr int kBatch = TILES < 8 ? TILES : 8;
#pragma unroll
    for (int a0 = 0; a0 < TILES; a0 += kBatch) {
        bf16x8 k[kBatch][2];
#pragma unroll
        for (int a = 0; a < kBatch; a++) {
            const bf16* p = keys + (int64_t)row_of(a0 + a) * kD;
            k[a][0] = ld16(p + pieces.first);
            k[a][1] = ld16(p + pieces.second);
        }
#pragma unroll
        for (int a = 0; a < kBatch; a++) {
            f32x4 z = {0.f, 0.f, 0.f, 0.f};
            s[a0 + a] = mfma_bf16(k[a][1], bq[1], mfma_bf16(k[a][0], bq[0], z));
        }
    }
}

// What the W waves of a workgroup that hold parts of the same sixteen rows use to add their counts; W = 1 needs none of it.
template <int W>
struct RowShare {
    int part[2][W][16];
};
template <int W>
__device__ __forceinline__ int rows_sum(int v, RowShare<W>* sh, int& turn, int wave, int lane) {
    v = quad_sum_i(v);
    if (W > 1) {
        // (two buffers in turn: a wave that is through the barrier may write the next counts while another still reads these)
        if (lane < 16) sh->part[turn][wave][lane] = v;
        __syncthreads();
        v = 0;
#pragma unroll
        for (int w = 0; w < W; w++) v += sh->part[turn][w][lane & 15];
        turn ^= 1;
    }
    return v;
}

// A key near the middle of the scores of two keys (it need not lie between them: a NaN, an overflow).
__device__ __forceinline__ float key_score(unsigned k) { return __uint_as_float((k & 0x80000000u) ? (k ^ 0x80000000u) : ~k); }
__device__ __forceinline__ unsigned middle_key(unsigned a, unsigned b) { return ordered_key(0.5f * (key_score(a) + key_score(b))); }
__device__ __forceinline__ unsigned long long middle_key(unsigned long long a, unsigned long long b) {
    return (unsigned long long)middle_key((unsigned)(a >> 32), (unsigned)(b >> 32)) << 32;
}

// A threshold that leaves a few more than the T best keys of every row: count(key >= t) is at least T and at most T + kSpare,
// or t is a key so often repeated that no threshold comes closer.  key[0..E): this lane's keys of its row (0: empty).  lo: a lower bound with
// count(key >= lo) >= T; top: the row's largest key.  T may differ from row to row (it is the same in a row's lanes).  Returns
// t; n_ge: the count at t.  The rows of a wave (of all W waves) run until the last one is decided.
// The first steps halve the interval of scores, not of keys: half of all keys between 0.01 and 16 belong to scores below 0.4.
constexpr int kSpare = 8, kScoreSteps = 10;
template <int E, int W, typename Key>
__device__ __forceinline__ Key row_threshold(const Key (&key)[E], int T, Key lo, Key top, RowShare<W>* sh, int& turn, int wave, int lane,
                                             int& n_ge) {
    Key mid = lo, hi = top + 1;                               // (top is below the largest integer: an index part is never all ones)
    bool open = true;
    n_ge = 0;
    for (int step = 0;; step++) {
        int c = 0;
#pragma unroll
        for (int i = 0; i < E; i++) c += (key[i] >= mid) ? 1 : 0;
        c = rows_sum<W>(c, sh, turn, wave, lane);
        if (open) {
            if (c >= T) {
                lo = mid;
                n_ge = c;
            } else {
                hi = mid;
            }
            open = n_ge > T + kSpare && hi - lo > 1;
        }
        if (__ballot(open) == 0) return lo;
        const Key half = lo + ((hi - lo) >> 1), of_score = middle_key(lo, hi);
        mid = !open ? lo : (step < kScoreSteps && of_score > lo && of_score < hi) ? of_score : half;
    }
}

// The T best of a row's m (>= T) keys in LDS, in order: a key's rank is the number of larger ones, 64 * W threads for sixteen rows.
// keys[row][slot]: wide keys, no two of a row equal.  index_of(low word) is what goes to out + row * out_stride + rank.
constexpr int kWin = kMaxT + kSpare, kWinStride = kWin + 1;       // (odd: the rows start in different banks; what is no winner goes to the last place)
template <int W, typename IndexOf>
__device__ __forceinline__ void write_winners(unsigned long long (*keys)[kWinStride], const int* n_keys, int T, int* out, int64_t out_stride, int tid,
                                              IndexOf index_of) {
    constexpr int kSub = 4 * W;                   // threads per row
    const int row = tid / kSub, sub = tid % kSub, m = min(n_keys[row], kWin);
    for (int j0 = sub; j0 < m; j0 += 4 * kSub) {
        unsigned long long own[4];
        int rank[4];
#pragma unroll
        for (int u = 0; u < 4; u++) {
            own[u] = keys[row][min(j0 + u * kSub, m - 1)];
            rank[u] = 0;
        }
#pragma unroll 4
        for (int j = 0; j < m; j++) {
            const unsigned long long o = keys[row][j];
#pragma unroll
            for (int u = 0; u < 4; u++) rank[u] += o > own[u] ? 1 : 0;
        }
#pragma unroll
        for (int u = 0; u < 4; u++)
            if (j0 + u * kSub < m && rank[u] < T) out[row * out_stride + rank[u]] = index_of((unsigned)own[u]);
    }
}
__device__ __forceinline__ int wide_index(unsigned low) { return 0x7FFFFFFF - (int)low; }

// t again, in a way the compiler cannot see through (slot is a small non-negative number out of LDS): the comparisons that
// counted the winners are made a second time when they are written, instead of being kept as dozens of lane masks, for which
// the scalar registers do not suffice.
template <typename Key>
__device__ __forceinline__ Key compare_again(Key t, int slot) { return t + (Key)((unsigned)slot >> 31); }

// A lower bound of the T-th best key of every row (0 < bound): the keys are cut into disjoint groups, and the smallest of
// the groups' largest keys has at least as many keys at or above it as there are groups.  tiles: key tiles there are (tile a * W +
// wave is in registers 4 a ..); no group may be without any.
template <int TPW, int W>
__device__ __forceinline__ unsigned row_bound(const unsigned (&key)[4 * TPW], int tiles, int T, unsigned& top, RowShare<W>* sh, int& turn,
                                              int wave, int lane) {
    constexpr int kFew = TPW < 4 ? TPW : 4;                   // groups per lane: all its keys, kFew groups, or one per tile
    unsigned tile_max[TPW], few[kFew];
#pragma unroll
    for (int g = 0; g < kFew; g++) few[g] = 0;
#pragma unroll
    for (int a = 0; a < TPW; a++) {
        tile_max[a] = max(max(key[4 * a], key[4 * a + 1]), max(key[4 * a + 2], key[4 * a + 3]));
        few[a % kFew] = max(few[a % kFew], tile_max[a]);
    }
    top = 0;
#pragma unroll
    for (int g = 0; g < kFew; g++) top = max(top, few[g]);
    unsigned lo = top;                                        // the fewer groups the closer the bound
    if (T > 4 * W || tiles < W) {
        lo = 0xFFFFFFFFu;
        if (T <= 4 * W * kFew && tiles >= W * kFew) {
#pragma unroll
            for (int g = 0; g < kFew; g++) lo = min(lo, few[g]);
        } else if (T <= 4 * W * TPW && tiles == W * TPW) {
#pragma unroll
            for (int a = 0; a < TPW; a++) lo = min(lo, tile_max[a]);
        } else {                                              // the row's smallest key
#pragma unroll
            for (int i = 0; i < 4 * TPW; i++) lo = key[i] != 0u ? min(lo, key[i]) : lo;
        }
    }
    top = quad_max_u(top);
    lo = quad_min_u(lo);
    if (W > 1) {
        if (lane < 16) {
            sh->part[0][wave][lane] = (int)top;
            sh->part[1][wave][lane] = (int)lo;
        }
        __syncthreads();
#pragma unroll
        for (int w = 0; w < W; w++) {
            top = max(top, (unsigned)sh->part[0][w][lane & 15]);
            lo = min(lo, (unsigned)sh->part[1][w][lane & 15]);
        }
        __syncthreads();
        turn = 0;
    }
    return max(lo, 1u);
}

constexpr int kRegMaxN = 1024;        // keys per row the register kernel takes: 4 waves x 16 tiles

// Dense selection for n <= kRegMaxN: 16 query rows per workgroup, four waves that take every fourth key tile each.
// PACK: scores rounded to bf16, score and index in one 32-bit key; otherwise fp32 scores with a second bisection over the
// index where scores are equal.  Latency decides here (a few hundred workgroups of a few thousand cycles each); with
// one row per wave and a ballot per score it took 17 us at n = 256, 24 rows of heads, and 44 us at n = 1024, 6.
template <int TPW, int W, bool PACK>
__global__ __launch_bounds__(64 * W) void topk_dense_kernel(const bf16* __restrict__ pq, const bf16* __restrict__ pk, int* __restrict__ out,
                                                         int n, int T, int tiled) {
    constexpr int E = 4 * TPW;
    __shared__ RowShare<W> share;
    __shared__ unsigned long long win[16][kWinStride];
    __shared__ int n_win[16];
    const int tid = threadIdx.x, lane = tid & 63, wave = W == 1 ? 0 : __builtin_amdgcn_readfirstlane(tid >> 6), quad = lane >> 4, r = lane & 15;
    const int bh = blockIdx.y, q0 = blockIdx.x * 16;
    const bf16* pqb = pq + ((int64_t)bh * n + q0) * kD;
    const bf16* pkb = pk + (int64_t)bh * n * kD;
    if (tid < 16) n_win[tid] = 0;
    bf16x8 bq[2];
    bq[0] = ld16(pqb + r * kD + quad * 8);
    bq[1] = ld16(pqb + r * kD + quad * 8 + 32);
    unsigned key[E];
    f32x4 s[TPW];
    score_tiles<TPW>(s, pkb, [=](int a) { return min(a * W + wave, n / 16 - 1) * 16; }, bq, KeyPieces(tiled, lane));
#pragma unroll
    for (int a = 0; a < TPW; a++) {
        const int tile = a * W + wave;
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const unsigned k = PACK ? packed_key(s[a][e], tile * 16 + 4 * quad + e) : ordered_key(s[a][e]);
            key[4 * a + e] = tile < n / 16 ? k : 0u;
        }
    }
    int turn = 0, n_ge;
    unsigned top;
    const unsigned lo = row_bound<TPW, W>(key, n / 16, T, top, &share, turn, wave, lane);
    const unsigned t = row_threshold<E, W>(key, T, lo, top, &share, turn, wave, lane, n_ge);
    if (!PACK) {                                              // of the keys equal to t, the ones at the smallest indices are taken
        // (the same in all waves: counts are the workgroup's)
        const bool tie = n_ge > T + kSpare;
        if (__ballot(tie) != 0) {
            int above = 0;
#pragma unroll
            for (int i = 0; i < E; i++) above += (key[i] > t) ? 1 : 0;
            above = rows_sum<W>(above, &share, turn, wave, lane);
            int a0 = -1, a1 = n - 1;                          // count(equal, index <= a0) < T - above <= count(equal, index <= a1)
            while (__ballot(tie && a1 - a0 > 1) != 0) {
                const int mid = a0 + ((a1 - a0) >> 1);
                const unsigned te = compare_again(t, a1);
                int c = 0;
#pragma unroll
                for (int i = 0; i < E; i++) c += (key[i] == te && ((i >> 2) * W + wave) * 16 + 4 * quad + (i & 3) <= mid) ? 1 : 0;
                c = rows_sum<W>(c, &share, turn, wave, lane);
                if (a1 - a0 > 1) {
                    if (c >= T - above) a1 = mid;
                    else a0 = mid;
                }
            }
            if (tie) {
#pragma unroll
                for (int i = 0; i < E; i++) key[i] = (key[i] == t && ((i >> 2) * W + wave) * 16 + 4 * quad + (i & 3) > a1) ? 0u : key[i];
            }
        }
    }
    // winners to LDS, in any order (their keys are unique)
    int mine = 0;
#pragma unroll
    for (int i = 0; i < E; i++) mine += key[i] >= t ? 1 : 0;
    __syncthreads();                                          // (n_win is cleared)
    int slot = mine > 0 ? atomicAdd(&n_win[r], mine) : 0;
    const unsigned t2 = compare_again(t, slot);
#pragma unroll
    for (int i = 0; i < E; i++) {
        const bool on = key[i] >= t2;
        win[r][on ? min(slot, kWin) : kWin] = wide_key(PACK ? key[i] & 0xFFFF0000u : key[i], ((i >> 2) * W + wave) * 16 + 4 * quad + (i & 3));
        slot += on ? 1 : 0;
    }
    __syncthreads();
    write_winners<W>(win, n_win, T, out + ((int64_t)bh * n + q0) * T, T, tid, wide_index);
}

// Dense selection for n <= 64, scores rounded to bf16, in small grids: a wave per row ranks all its keys.  Sixteen rows a wave (topk_dense_kernel<4, 1>) take
// fewer instructions over all rows, but a longer chain, which grows with T where the winners are ranked.
__global__ __launch_bounds__(256) void topk_rank_kernel(const bf16* __restrict__ pq, const bf16* __restrict__ pk, int* __restrict__ out, int n, int T,
                                                        int tiled) {
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int64_t row = (int64_t)blockIdx.y * n + blockIdx.x * 4 + wave;      // (n is a multiple of 16)
    const KeyPieces pieces(tiled, lane);
    const RankedKeys<1> ranked = rank_keys<1>(pq + row * kD, pk + (int64_t)blockIdx.y * n * kD, pieces.first, pieces.second, n, lane);
    const int idx = ranked.index(0, lane);
    if (ranked.rank[0] < T && idx < n) out[row * T + ranked.rank[0]] = idx;
}

// Dense selection for longer rows: two looks at all scores, and between them a bound of every row's T-th best.
//  * First look: the largest score of each of G groups of a row's keys.  The T-th largest of those is a bound: at least T keys reach
//    it, and few more do if the groups are many and neighbours, which score alike, fall into different ones.  So a group is a
//    position among the sixteen keys of a tile, by wave (a tile in four) and, for T > 16, by a further one or two bits of the tile: 64
//    consecutive keys, which are a patch of 8 x 8 on image-like data, are in 64 groups.
//  * Second look: the keys that reach the bound go to their row's buffer in LDS, and the T best of those are ranked.
// A workgroup is 16 RT rows, and its four waves take every fourth key tile of the row each, four tiles on their way to registers while four are worked
// on.  What bounds it is the rate at which key tiles arrive -- each is read once per workgroup and look, hence many
// rows a workgroup where the grid is large -- and the chain through LDS for the tiles that hold a key that passes.
// Where a row's bound lets more than kBuf keys through (ties; a period of the image that puts the best keys into few groups), the second look ends and the workgroup
// looks a third time with a running bound: four tiles a round, and rows whose buffers could not hold another round are cut back to little more than
// their T best, whose least is the new bound.  No two keys of a row are equal, so behind a cut no equal score further on passes.  All scores equal, us, by a
// bisection of the bound with a look a step / this (spread scores): 8 x 4096 rows, T = 8, 708 / 136 (95);  4 x 4096, T = 16, 384 / 80 (65);  6 x 2048, T = 8, 202 /
// 54 (35.6);  4 x 2048, T = 32, 115 / 43 (32.7);  16 x 4096 in 64 bits, T = 32, 3770 / 312 (240).  The best keys in T - 1 of 64 groups: 4 x 4096, T = 16, 176 / 134.
// Key: the 32-bit packed key (scores rounded to bf16, n <= kMaxPackedKeys) or the 64-bit wide key.
// (8 x 4096 rows of 4096 keys out of tiles: 49 us, T = 32 68; out of rows 72 and 84.  Out of rows, a T-step arg-max over chunks of 512 keys per row took
// 1480; a running threshold per row, raised whenever a buffer was full, by a wave for itself 128 and 142, with key tiles shared through LDS
// behind barriers 157.  5 x 3072, T = 16: 69 / 38, tiles 30;  1 x 4096, T = 32: 57 / 43, tiles 28;  1 x 1088, T = 8: 21 / 17, tiles 11.)
constexpr int kStreamWaves = 4;
constexpr int kAhead = 4;                         // key tiles on their way to a wave while as many are worked on

template <typename Key>
struct StreamKey;
template <>
struct StreamKey<unsigned> {
    static __device__ __forceinline__ unsigned make(float s, int idx, bool) { return packed_key(s, idx); }
    static __device__ __forceinline__ unsigned long long wide(unsigned k) { return wide_key(k & 0xFFFF0000u, 0xFFFF - (int)(k & 0xFFFFu)); }
    // the smallest key a score (given as ordered key of the score before rounding) can make
    static __device__ __forceinline__ unsigned least(unsigned score, bool) { return ordered_key(rn_bf16(key_score(score))) & 0xFFFF0000u; }
    // a score below this cannot make a key of at least t: one bf16 step below t's score
    static __device__ __forceinline__ unsigned score_bits(unsigned t) { return t & 0xFFFF0000u; }
};
template <>
struct StreamKey<unsigned long long> {
    static __device__ __forceinline__ unsigned long long make(float s, int idx, bool round) {
        return wide_key(ordered_key(round ? rn_bf16(s) : s), idx);
    }
    static __device__ __forceinline__ unsigned long long wide(unsigned long long k) { return k; }
    static __device__ __forceinline__ unsigned long long least(unsigned score, bool round) {
        return (unsigned long long)(round ? ordered_key(rn_bf16(key_score(score))) : score) << 32;
    }
    static __device__ __forceinline__ unsigned score_bits(unsigned long long t) { return (unsigned)(t >> 32) & 0xFFFF0000u; }
};
// The largest float that is certainly below (or rounds below) the score of key bits `k` (its low 16 bits are zero).
__device__ __forceinline__ float score_floor(unsigned k) {
    if (k < 0x00020000u) return -INFINITY;
    k -= 0x00010000u;                                         // one bf16 step down
    const unsigned b = (k & 0x80000000u) ? (k ^ 0x80000000u) : ~k;
    const float f = __uint_as_float(b);
    return (f != f) ? -INFINITY : f;
}
__device__ __forceinline__ float largest(const f32x4& s) { return fmaxf(fmaxf(s[0], s[1]), fmaxf(s[2], s[3])); }

// RT: sixteens of rows per workgroup (n is a multiple of 16 RT); SETS: groups per row / 64
template <typename Key, int RT, int SETS>
__global__ __launch_bounds__(64 * kStreamWaves) void topk_stream_kernel(const bf16* __restrict__ pq, const bf16* __restrict__ pk,
                                                                        int* __restrict__ out, int n, int T, int round_scores, int tiled) {
    static_assert(RT == 1 || RT == 2 || RT == 4, "the waves are dealt to the row tiles");
    static_assert(kAhead % SETS == 0, "a tile's set of groups is known at compile time");
    constexpr int W = kStreamWaves, kPer = W / RT;            // waves per row tile where the rows are finished
    constexpr int kRows = 16 * RT, kGroups = 64 * SETS;
    constexpr bool kWide = sizeof(Key) == 8;                  // (the buffers in 64 KB of LDS)
    constexpr int kBuf = RT == 4 ? (kWide ? 96 : 128) : SETS < 4 ? 128 : (kWide && RT == 2) ? 224 : 256;
    // where the bound is a running one: the largest T (see topk_dense), a row's keys behind a cut, key tiles a round, and a row's keys in front of a cut
    constexpr int kMostT = SETS == 1 ? 16 : RT == 4 ? 32 : kMaxT, kKept = kMostT + kSpare;
    constexpr int kRound = (kBuf - kKept) / 16 < W ? (kBuf - kKept) / 16 : W, kSlack = 40;
    constexpr int kFull = kKept + 16 * kRound + kSlack < kBuf ? kKept + 16 * kRound + kSlack : kBuf;
    static_assert(kRound >= 1 && kFull >= kKept + 16 * kRound, "the buffers hold a cut row and a round's keys");
    // one piece of LDS, for the groups' largest scores, then the rows' buffers, then what is ranked
    constexpr int kBytesGroups = kRows * (kGroups + 1) * 4, kBytesBuf = kRows * (kBuf + 1) * (int)sizeof(Key), kBytesWin = kRows * kWinStride * 8;
    constexpr int kBytes = kBytesGroups > kBytesBuf ? (kBytesGroups > kBytesWin ? kBytesGroups : kBytesWin)
                                                    : (kBytesBuf > kBytesWin ? kBytesBuf : kBytesWin);
    __shared__ unsigned long long space[(kBytes + 7) / 8];
    __shared__ Key bound[kRows];
    __shared__ int cnt[kRows], n_win[RT][16];
    unsigned (*const groups)[kGroups + 1] = reinterpret_cast<unsigned (*)[kGroups + 1]>(space);
    Key (*const buf)[kBuf + 1] = reinterpret_cast<Key (*)[kBuf + 1]>(space);
    unsigned long long (*const win)[16][kWinStride] = reinterpret_cast<unsigned long long (*)[16][kWinStride]>(space);
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), quad = lane >> 4, r = lane & 15;
    const int lid = xcd_logical_id();                         // (a (b,h)'s keys on one XCD)
    const int bh = lid / (int)gridDim.x, q0 = lid % (int)gridDim.x * kRows;
    const bf16* pqb = pq + ((int64_t)bh * n + q0) * kD;
    const bf16* pkb = pk + (int64_t)bh * n * kD;
    const KeyPieces pieces(tiled, lane);
    const int tiles = n / 16;
    const bool round = round_scores != 0;
    bf16x8 bq[RT][2];
#pragma unroll
    for (int rt = 0; rt < RT; rt++) {
        bq[rt][0] = ld16(pqb + (rt * 16 + r) * kD + quad * 8);
        bq[rt][1] = ld16(pqb + (rt * 16 + r) * kD + quad * 8 + 32);
    }
    auto scores = [&](f32x4 (&s)[RT], const bf16x8 (&k)[2]) __attribute__((always_inline)) {
#pragma unroll
        for (int rt = 0; rt < RT; rt++) {
            f32x4 z = {0.f, 0.f, 0.f, 0.f};
            s[rt] = mfma_bf16(k[1], bq[rt][1], mfma_bf16(k[0], bq[rt][0], z));
        }
    };
    auto settle = [&]() __attribute__((always_inline)) {      // LDS of this wave: what was read and written is, before what follows
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
    };
    // A look at all scores: see(s, i, tile) gets the scores of all row tiles against a key tile of this wave's, i (known at compile
    // time) = its place among the wave's tiles modulo kAhead
    auto look = [&](auto&& see, auto&& more) __attribute__((always_inline)) {
        struct Tiles { bf16x8 k[kAhead][2]; } ta, tb;
        auto load = [&](Tiles& o, int t) __attribute__((always_inline)) {
#pragma unroll
            for (int i = 0; i < kAhead; i++) {
                const bf16* p = pkb + (int64_t)min(t + i * W, tiles - 1) * 16 * kD;
                o.k[i][0] = ld16(p + pieces.first);
                o.k[i][1] = ld16(p + pieces.second);
            }
        };
        auto work = [&](const Tiles& o, int t) __attribute__((always_inline)) {
#pragma unroll
            for (int i = 0; i < kAhead; i++) {
                if (t + i * W < tiles) {
                    f32x4 s[RT];
                    scores(s, o.k[i]);
                    see(s, i, t + i * W);
                }
            }
        };
        constexpr int kStep = kAhead * W;
        load(ta, wave);
        for (int t = wave; t < tiles && more(); t += 2 * kStep) {
            load(tb, t + kStep);
            work(ta, t);
            load(ta, t + 2 * kStep);
            work(tb, t + kStep);
        }
    };

    // ---- the groups' largest scores
    f32x4 most[RT][SETS];
#pragma unroll
    for (int rt = 0; rt < RT; rt++)
#pragma unroll
        for (int g = 0; g < SETS; g++) most[rt][g] = f32x4{-INFINITY, -INFINITY, -INFINITY, -INFINITY};
    look([&](const f32x4 (&s)[RT], int i, int) __attribute__((always_inline)) {
#pragma unroll
        for (int rt = 0; rt < RT; rt++)
#pragma unroll
            for (int e = 0; e < 4; e++) most[rt][i % SETS][e] = fmaxf(most[rt][i % SETS][e], s[rt][e]);
    }, []() { return true; });
    if (tid < kRows) cnt[tid] = 0;
    if (tid < 16 * RT) n_win[tid / 16][tid % 16] = 0;
#pragma unroll
    for (int rt = 0; rt < RT; rt++)
#pragma unroll
        for (int g = 0; g < SETS; g++)
#pragma unroll
            for (int e = 0; e < 4; e++) groups[rt * 16 + r][((wave * SETS + g) * 4 + e) * 4 + quad] = ordered_key(most[rt][g][e]);
    __syncthreads();
    const int own_rt = wave / kPer;                           // the row tile this wave finishes, if it is the first of that tile's waves
    const bool finishes = wave % kPer == 0;
    if (finishes) {
        unsigned key[kGroups / 4], top;
#pragma unroll
        for (int i = 0; i < kGroups / 4; i++) key[i] = groups[own_rt * 16 + r][i * 4 + quad];
        int turn = 0, n_ge;
        const unsigned lo = row_bound<kGroups / 16, 1>(key, kGroups / 16, T, top, (RowShare<1>*)nullptr, turn, 0, lane);
        const unsigned t = row_threshold<kGroups / 4, 1>(key, T, lo, top, (RowShare<1>*)nullptr, turn, 0, lane, n_ge);
        // (a group without a number has the score -infinity, and below that there are keys yet: those of NaNs)
        if (quad == 0) bound[own_rt * 16 + r] = t <= ordered_key(-INFINITY) ? (Key)1 : StreamKey<Key>::least(t, round);
    }
    __syncthreads();

    // ---- the keys that reach the bound
    Key tau[RT];                                              // keys below it are not among the row's T best
    float low[RT];                                            // scores below it do not make such a key
    auto set_bounds = [&](int rt, Key t) __attribute__((always_inline)) {
        tau[rt] = t;
        low[rt] = score_floor(StreamKey<Key>::score_bits(t));
    };
    auto take = [&](const f32x4 (&s)[RT], int tile) __attribute__((always_inline)) {
        bool pass[RT], any = false;
#pragma unroll
        for (int rt = 0; rt < RT; rt++) {
            pass[rt] = !(largest(s[rt]) < low[rt]);           // (a NaN passes: it has to be able to fill a row that has nothing better)
            any |= pass[rt];
        }
        if (__ballot(any) == 0) return;
#pragma unroll
        for (int rt = 0; rt < RT; rt++) {
            if (!pass[rt]) continue;
            Key k[4];
            int mine = 0;
#pragma unroll
            for (int e = 0; e < 4; e++) {
                k[e] = StreamKey<Key>::make(s[rt][e], tile * 16 + 4 * quad + e, round);
                mine += k[e] >= tau[rt] ? 1 : 0;
            }
            if (mine > 0) {
                int slot = atomicAdd(&cnt[rt * 16 + r], mine);
#pragma unroll
                for (int e = 0; e < 4; e++)
                    if (k[e] >= tau[rt]) buf[rt * 16 + r][min(slot++, kBuf)] = k[e];
            }
        }
    };
#pragma unroll
    for (int rt = 0; rt < RT; rt++) set_bounds(rt, bound[rt * 16 + r]);
    int counted = 0;
    look([&](const f32x4 (&s)[RT], int, int tile) __attribute__((always_inline)) { take(s, tile); },
         [&]() __attribute__((always_inline)) {               // (a row with more keys than its buffer holds: the rest is no help)
             const bool none = __ballot(counted > kBuf) == 0;
             counted = __atomic_load_n(&cnt[lane % kRows], __ATOMIC_RELAXED);      // (looked at eight tiles later)
             return none;
         });
    __syncthreads();
    bool over = false;
#pragma unroll
    for (int rt = 0; rt < RT; rt++) over |= cnt[rt * 16 + r] > kBuf;
    if (__ballot(over) != 0) {                                // (the same in all waves)
        __syncthreads();                                      // (the counts have been read)
        if (tid < kRows) cnt[tid] = 0;
        __syncthreads();
        bf16x8 k[2];
        auto load = [&](int t) __attribute__((always_inline)) {
            const bf16* p = pkb + (int64_t)min(t, tiles - 1) * 16 * kD;
            k[0] = ld16(p + pieces.first);
            k[1] = ld16(p + pieces.second);
        };
        load(wave);
        for (int t0 = 0; t0 < tiles; t0 += kRound) {
            if (wave < kRound && t0 + wave < tiles) {
                f32x4 s[RT];
                scores(s, k);
                load(t0 + kRound + wave);
                take(s, t0 + wave);
            }
            __syncthreads();
            bool full = false;
#pragma unroll
            for (int rt = 0; rt < RT; rt++) full |= cnt[rt * 16 + r] > kFull - 16 * kRound;
            if (__ballot(full) != 0) {                        // (the same in all waves)
                __syncthreads();                              // (every wave has decided)
                if (finishes) {
                    const int row = own_rt * 16 + r, have = cnt[row];
                    Key key[(kFull + 3) / 4], top = 0;
#pragma unroll
                    for (int i = 0; i < (kFull + 3) / 4; i++) {
                        const int at = i * 4 + quad;
                        key[i] = at < have ? buf[row][at] : (Key)0;
                        top = key[i] > top ? key[i] : top;
                    }
                    top = quad_max_u(top);
                    int turn = 0, n_ge, mine = 0;
                    const Key t = row_threshold<(kFull + 3) / 4, 1, Key>(key, min(T, have), bound[row], top, (RowShare<1>*)nullptr, turn, 0, lane, n_ge);
#pragma unroll
                    for (int i = 0; i < (kFull + 3) / 4; i++) mine += key[i] >= t ? 1 : 0;
                    settle();
                    if (quad == 0) {
                        cnt[row] = 0;
                        bound[row] = t;
                    }
                    settle();
                    int slot = mine > 0 ? atomicAdd(&cnt[row], mine) : 0;
                    const Key t2 = compare_again(t, slot);
#pragma unroll
                    for (int i = 0; i < (kFull + 3) / 4; i++)
                        if (key[i] >= t2) buf[row][min(slot++, kBuf)] = key[i];
                }
                __syncthreads();
#pragma unroll
                for (int rt = 0; rt < RT; rt++) set_bounds(rt, bound[rt * 16 + r]);
            }
            __syncthreads();                                  // (the counts have been read)
        }
    }

    // ---- little more than the T best of a row's buffer, and those ranked
    Key key[kBuf / 4], t = 1;
    if (finishes) {
        const int have = min(cnt[own_rt * 16 + r], kBuf);
        Key top = 0, least = 0;
#pragma unroll
        for (int i = 0; i < kBuf / 4; i++) {
            const int at = i * 4 + quad;
            key[i] = at < have ? buf[own_rt * 16 + r][at] : (Key)0;
            top = key[i] > top ? key[i] : top;
        }
#pragma unroll
        for (int rt = 0; rt < RT; rt++) least = rt == own_rt ? tau[rt] : least;
        t = least;                                            // (all of them, where they are few enough to be ranked)
        if (__ballot(have > kWin) != 0) {
            top = quad_max_u(top);
            int turn = 0, n_ge;
            t = row_threshold<kBuf / 4, 1, Key>(key, T, least, top, (RowShare<1>*)nullptr, turn, 0, lane, n_ge);
        }
    }
    __syncthreads();                                          // (the buffers have been read: what is ranked takes their place)
    if (finishes) {
        int mine = 0;
#pragma unroll
        for (int i = 0; i < kBuf / 4; i++) mine += key[i] >= t ? 1 : 0;
        int slot = mine > 0 ? atomicAdd(&n_win[own_rt][r], mine) : 0;
        const Key t2 = compare_again(t, slot);
#pragma unroll
        for (int i = 0; i < kBuf / 4; i++)
            if (key[i] >= t2) win[own_rt][r][min(slot++, kWin)] = StreamKey<Key>::wide(key[i]);
    }
    __syncthreads();
    write_winners<kPer>(win[own_rt], n_win[own_rt], T, out + ((int64_t)bh * n + q0 + own_rt * 16) * T, T, tid % (64 * kPer), wide_index);
}

// Parent-guided selection: 16 sibling rows per workgroup against the 16 * T2 tokens under their parent's T2 blocks, W waves
// (1 up to T2 = 16, 2 beyond: 64 keys a lane).  The parents are sorted by index first, so that of equal scores the one at the
// smaller position wins, as it must.
// P > 0: the parents are selected here first -- row G of the level above (N1/16 tokens, at most 16 P W) against all of its
// keys, scores rounded to bf16, top T2 as topk_dense_kernel does it -- and written to par_out; otherwise they are read from pidx.
// RANK: at most 64 parents, and every wave ranks them all (rank_keys).
// (One row per wave and 512 threads a workgroup took 25 us for 768 groups of 16 rows, T = T2 = 16, and 123 us for 6144.)
constexpr int kCascadeMaxParents = 256;           // P * W <= 16
template <int TPW, int W, int P, bool RANK>
__global__ __launch_bounds__(64 * W) void topk_sparse_kernel(const bf16* __restrict__ pq, const bf16* __restrict__ pk,
                                                             const int* __restrict__ pidx, int* __restrict__ out, int N1, int T, int T2,
                                                             const bf16* __restrict__ pq_par, const bf16* __restrict__ pk_par,
                                                             int* __restrict__ par_out, int tiled) {
    constexpr int E = 4 * TPW;
    __shared__ RowShare<W> share;
    __shared__ unsigned long long win[16][kWinStride];
    __shared__ int n_win[16];
    __shared__ int par[kMaxCand / 16], par_sorted[W][kMaxCand / 16], n_par;
    const int tid = threadIdx.x, lane = tid & 63, wave = W == 1 ? 0 : __builtin_amdgcn_readfirstlane(tid >> 6), quad = lane >> 4, r = lane & 15;
    const int lid = xcd_logical_id();                         // (neighbouring groups have parents in common: one L2)
    const int bh = lid / (int)gridDim.x, G = lid % (int)gridDim.x;
    const int N2 = N1 / kBlk;
    const bf16* pqb = pq + ((int64_t)bh * N1 + G * kBlk) * kD;
    const bf16* pkb = pk + (int64_t)bh * N1 * kD;
    const KeyPieces pieces(tiled, lane);
    bf16x8 bq[2];
    bq[0] = ld16(pqb + r * kD + quad * 8);
    bq[1] = ld16(pqb + r * kD + quad * 8 + 32);
    if (tid < 16) n_win[tid] = 0;
    if (tid == 16) n_par = 0;

    if constexpr (RANK) {
        static_assert(P * W == 4, "64 keys");
        const RankedKeys<1> ranked = rank_keys<1>(pq_par + ((int64_t)bh * N2 + G) * kD, pk_par + (int64_t)bh * N2 * kD, pieces.first, pieces.second, N2, lane);
        if (wave == 0 && ranked.rank[0] < T2) {
            const int idx = ranked.index(0, lane);
            par[ranked.rank[0]] = idx;
            par_out[((int64_t)bh * N2 + G) * T2 + ranked.rank[0]] = idx;
        }
    } else if constexpr (P > 0) {
        // every column of the score tiles is the parent row G, so all sixteen "rows" decide alike; row 0's lanes write
        const bf16* qt = pq_par + ((int64_t)bh * N2 + G) * kD;
        bf16x8 bp[2];
        bp[0] = ld16(qt + quad * 8);
        bp[1] = ld16(qt + quad * 8 + 32);
        unsigned key[4 * P], top;
        f32x4 sp[P];
        int turn = 0, n_ge;
        score_tiles<P>(sp, pk_par + (int64_t)bh * N2 * kD, [=](int a) { return min(a * W + wave, N2 / 16 - 1) * 16; }, bp, pieces);
#pragma unroll
        for (int a = 0; a < P; a++)
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const int tile = a * W + wave;
                key[4 * a + e] = tile * 16 < N2 ? packed_key(sp[a][e], tile * 16 + 4 * quad + e) : 0u;
            }
        const unsigned lo = row_bound<P, W>(key, N2 / 16, T2, top, &share, turn, wave, lane);
        const unsigned t = row_threshold<4 * P, W>(key, T2, lo, top, &share, turn, wave, lane, n_ge);
        int mine = 0;
#pragma unroll
        for (int i = 0; i < 4 * P; i++) mine += key[i] >= t ? 1 : 0;
        __syncthreads();                                      // (n_par is cleared)
        int slot = (r == 0 && mine > 0) ? atomicAdd(&n_par, mine) : 0;
        const unsigned t2 = compare_again(t, slot);
        if (r == 0) {
#pragma unroll
            for (int i = 0; i < 4 * P; i++) {
                const bool on = key[i] >= t2;
                win[0][on ? min(slot, kWin) : kWin] = key[i];
                slot += on ? 1 : 0;
            }
        }
        __syncthreads();
        const unsigned own = (unsigned)win[0][lane];          // (at most 32 + kSpare keys, one a lane, handed round with readlane)
        const int m = __builtin_amdgcn_readfirstlane(n_ge);
        int rank = 0;
        for (int j = 0; j < m; j++) rank += (unsigned)__builtin_amdgcn_readlane((int)own, j) > own ? 1 : 0;
        const int idx = 0xFFFF - (int)(own & 0xFFFFu);
        if (wave == 0 && lane < m && rank < T2) {
            par[rank] = idx;
            par_out[((int64_t)bh * N2 + G) * T2 + rank] = idx;
        }
    } else {
        if (tid < T2) par[tid] = clampi(pidx[((int64_t)bh * N2 + G) * T2 + tid], 0, N2 - 1);
    }
    __syncthreads();
    {   // by index, every wave for itself; the clamp keeps what a lane without a parent reads out of use
        const int own = par[min(lane, T2 - 1)];
        int rank = 0;
        for (int j = 0; j < T2; j++) {
            const int o = __builtin_amdgcn_readlane(own, j);
            rank += (o < own || (o == own && j < lane)) ? 1 : 0;
        }
        if (lane < T2) par_sorted[wave][rank] = own;
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    const int mine_par = par_sorted[wave][min(lane, T2 - 1)];

    // position of key i of this lane: tile (i / 4) * W + wave, token 4 * quad + i % 4 of it
    unsigned key[E];
    int blk[TPW];                                             // (wave-uniform: scalar registers)
#pragma unroll
    for (int a = 0; a < TPW; a++) blk[a] = __builtin_amdgcn_readlane(mine_par, min(a * W + wave, T2 - 1)) * kBlk;
    f32x4 s[TPW];
    score_tiles<TPW>(s, pkb, [&](int a) { return blk[a]; }, bq, pieces);
#pragma unroll
    for (int a = 0; a < TPW; a++)
#pragma unroll
        for (int e = 0; e < 4; e++) key[4 * a + e] = a * W + wave < T2 ? ordered_key(s[a][e]) : 0u;
    int turn = 0, n_ge;
    unsigned top;
    const unsigned lo = row_bound<TPW, W>(key, T2, T, top, &share, turn, wave, lane);
    const unsigned t = row_threshold<E, W>(key, T, lo, top, &share, turn, wave, lane, n_ge);
    const bool tie = n_ge > T + kSpare;
    if (__ballot(tie) != 0) {                                 // of the keys equal to t, the ones at the smallest positions are taken
        int above = 0;
#pragma unroll
        for (int i = 0; i < E; i++) above += (key[i] > t) ? 1 : 0;
        above = rows_sum<W>(above, &share, turn, wave, lane);
        int a0 = -1, a1 = T2 * kBlk - 1;
        while (__ballot(tie && a1 - a0 > 1) != 0) {
            const int mid = a0 + ((a1 - a0) >> 1);
            const unsigned te = compare_again(t, a1);
            int c = 0;
#pragma unroll
            for (int i = 0; i < E; i++) c += (key[i] == te && ((i >> 2) * W + wave) * 16 + 4 * quad + (i & 3) <= mid) ? 1 : 0;
            c = rows_sum<W>(c, &share, turn, wave, lane);
            if (a1 - a0 > 1) {
                if (c >= T - above) a1 = mid;
                else a0 = mid;
            }
        }
        if (tie) {
#pragma unroll
            for (int i = 0; i < E; i++) key[i] = (key[i] == t && ((i >> 2) * W + wave) * 16 + 4 * quad + (i & 3) > a1) ? 0u : key[i];
        }
    }
    int mine = 0;
#pragma unroll
    for (int i = 0; i < E; i++) mine += key[i] >= t ? 1 : 0;
    int slot = mine > 0 ? atomicAdd(&n_win[r], mine) : 0;
    const unsigned t2 = compare_again(t, slot);
#pragma unroll
    for (int a = 0; a < TPW; a++) {
        const int base = (a * W + wave) * kBlk + 4 * quad;   // position: unique also where a caller's list names a parent twice
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const bool on = key[4 * a + e] >= t2;
            win[r][on ? min(slot, kWin) : kWin] = wide_key(key[4 * a + e], base + e);
            slot += on ? 1 : 0;
        }
    }
    __syncthreads();
    write_winners<W>(win, n_win, T, out + ((int64_t)bh * N1 + G * kBlk) * T, T, tid, [&](unsigned low) {
        const int pos = wide_index(low);
        return par_sorted[wave][pos / kBlk] * kBlk + pos % kBlk;
    });
}

}  // namespace llsa

using namespace llsa;

static int topk_dense(const void* pq, const void* pk, int32_t* out_idx, int B, int H, int n, int T, int round_scores, int tiled, void* stream) {
    LLSA_REQUIRE(pq && pk && out_idx, "topk_dense: null argument");
    LLSA_REQUIRE(B > 0 && H > 0 && n > 0 && n % 16 == 0, "topk_dense: n=%d must be a positive multiple of 16", n);
    LLSA_REQUIRE(T >= 1 && T <= kMaxT && T <= n, "topk_dense: need 1 <= T <= min(%d, n=%d), got %d", kMaxT, n, T);
    LLSA_REQUIRE(aligned16(pq) && aligned16(pk), "topk_dense: inputs must be 16-byte aligned");
    const hipStream_t st = (hipStream_t)stream;
    const bf16 *q = (const bf16*)pq, *k = (const bf16*)pk;
    // By rows over all heads, us, sixteen a wave / one a wave, 64 keys out of tiles:  T = 4: 384 4.2 / 3.3, 1536 4.2 / 3.9, 6144 4.5 / 6.5;  T = 8: 384 5.1 / 3.3, 1536
    // 5.2 / 3.9, 6144 5.4 / 6.4;  T = 16: 6144 7.1 / 6.5, 24576 8.5 / 17.2;  T = 32: 384 9.4 / 3.3, 6144 10.1 / 6.5, 24576 12.2 / 17.6;  T = 64: 384 11.6 / 3.4,
    // 6144 12.7 / 6.6, 24576 16.8 / 17.9.  Out of rows:  T = 8: 1536 5.4 / 5.1, 3072 5.6 / 6.3;  T = 16: 6144 7.4 / 9.3;  T = 32: 6144 10.3 / 9.3
    if (round_scores && n <= 64 && (int64_t)B * H * n <= std::min((tiled ? 384 : 192) * T, 16384)) {
        hipLaunchKernelGGL(topk_rank_kernel, dim3(n / 4, B * H), dim3(256), 0, st, q, k, out_idx, n, T, tiled);
    } else if (n <= kRegMaxN) {
        const dim3 grid(n / 16, B * H);
#define LLSA_DENSE(TPW, W)                                                                                                               \
    do {                                                                                                                                 \
        if (round_scores)                                                                                                                \
            hipLaunchKernelGGL(HIP_KERNEL_NAME(topk_dense_kernel<TPW, W, true>), grid, dim3(64 * W), 0, st, q, k, out_idx, n, T, tiled); \
        else hipLaunchKernelGGL(HIP_KERNEL_NAME(topk_dense_kernel<TPW, W, false>), grid, dim3(64 * W), 0, st, q, k, out_idx, n, T, tiled); \
    } while (0)
        if (n <= 64) LLSA_DENSE(4, 1);
        else if (n <= 128) LLSA_DENSE(2, 4);
        else if (n <= 256) LLSA_DENSE(4, 4);
        else if (n <= 512) LLSA_DENSE(8, 4);
        else LLSA_DENSE(16, 4);
#undef LLSA_DENSE
    } else {
        // Rows per workgroup.  A workgroup reads the row of keys twice however many rows it has, so 64 on large grids (32 beyond T = 32,
        // whose groups and buffers are larger), and 16 while those workgroups find room beside one another.  Tiles, us with 16 / 32 / 64, by sixteens of rows
        // (keys per row):
        //   T = 8: 256 (4096) 20.1 / 22.9 / 33.9;  400 (1280) 14.3 / 14.0 / 19.7;  448 (3584) 24.2 / 22.0 / 32.1;  512 (2048) 18.1 / 16.6 / 23.6
        //     544 (1088) 17.2 / 15.8 / 18.6;  1024 (2048) 27.9 / 21.7 / 24.8;  1536 (4096) 63.9 / 42.5 / 47.9;  1792 (2048) 42.5 / 35.9 / 31.1
        //     1920 (1536) 39.2 / 30.8 / 26.9;  2048 (4096) 82.3 / 56.3 / 48.8
        //   T = 16: 448 (3584) 25.0 / 24.1 / 35.0;  480 (1536) 16.4 / 17.1 / 23.6;  512 (2048) 18.7 / 19.4 / 26.7;  576 (3072) 29.3 / 28.1 / 35.1
        //     1536 (4096) 64.5 / 45.6 / 52.6;  1792 (2048) 44.7 / 38.5 / 35.2
        //   T = 32: 512 (2048) 27.8 / 29.3 / 42.5;  544 (1088) 24.6 / 27.2 / 34.8;  576 (3072) 35.4 / 36.3 / 46.0;  1024 (2048) 34.6 / 33.7 / 41.5
        //     1536 (4096) 74.0 / 55.5 / 66.8;  2048 (4096) 92.4 / 77.3 / 67.7
        // Rows, whose loads are what takes the time, T = 8: 128 (2048) 21 / 23 / 26;  256 (4096) 36 / 37 / 40;  400 (1280) 30 / 20 / 23;  512 (4096) 66 /
        //   38 / 40;  544 (1088) 43 / 30 / 22;  576 (3072) 73 / 52 / 33;  2048 (4096) 243 / 127 / 71
        const int64_t tiles = (int64_t)n / 16 * B * H;        // sixteens of rows
        const int64_t line1 = !tiled ? 256 : T <= 8 ? 400 : 560, line2 = !tiled ? 512 : 1536;
        const int rt = tiles <= line1 || n % 32 != 0 ? 1 : tiles <= line2 || n % 64 != 0 || T > 32 ? 2 : 4;
#define LLSA_STREAM(KEY, RT, SETS)                                                                                                              \
    hipLaunchKernelGGL(HIP_KERNEL_NAME(topk_stream_kernel<KEY, RT, SETS>), dim3(n / (16 * RT), B * H), dim3(64 * kStreamWaves), 0, st, q, k, out_idx, n, T, \
                       round_scores, tiled)
        const bool wide = !round_scores || n > kMaxPackedKeys;
        if (wide && rt == 1) LLSA_STREAM(unsigned long long, 1, 4);
        else if (wide && rt == 2) LLSA_STREAM(unsigned long long, 2, 4);
        else if (wide) LLSA_STREAM(unsigned long long, 4, 2);
        else if (rt == 1 && T <= 16) LLSA_STREAM(unsigned, 1, 1);
        else if (rt == 1) LLSA_STREAM(unsigned, 1, 4);
        else if (rt == 2 && T <= 16) LLSA_STREAM(unsigned, 2, 1);
        else if (rt == 2) LLSA_STREAM(unsigned, 2, 4);
        else if (T <= 16) LLSA_STREAM(unsigned, 4, 1);
        else LLSA_STREAM(unsigned, 4, 2);
#undef LLSA_STREAM
    }
    return launch_status("topk_dense");
}
extern "C" int llsa_topk_dense(const void* pq, const void* pk, int32_t* out_idx, int B, int H, int n, int T, int round_scores, void* stream) {
    return topk_dense(pq, pk, out_idx, B, H, n, T, round_scores, 0, stream);
}
extern "C" int llsa_topk_dense_tiles(const void* pq, const void* pk_tiles, int32_t* out_idx, int B, int H, int n, int T, int round_scores, void* stream) {
    return topk_dense(pq, pk_tiles, out_idx, B, H, n, T, round_scores, 1, stream);
}

static void launch_sparse(const bf16* pq, const bf16* pk, const int* pidx, int* out, int B, int H, int N1, int T, int T2, const bf16* pq_par,
                          const bf16* pk_par, int* par_out, int tiled, hipStream_t st) {
    const dim3 grid(N1 / 16, B * H);
#define LLSA_SPARSE_P(TPW, W, P, RANK) \
    hipLaunchKernelGGL(HIP_KERNEL_NAME(topk_sparse_kernel<TPW, W, P, RANK>), grid, dim3(64 * W), 0, st, pq, pk, pidx, out, N1, T, T2, pq_par, pk_par, par_out, tiled)
    // Up to 64 parents: ranked by every wave, the shorter chain, which out of rows costs four waves four times as many accesses as their quarters of the
    // keys.  By groups of 16 rows, us, with quarters / ranked, rows:  topk 8/8: 64 8.9 / 8.6;  512 10.2 / 10.3;  768 11.1 / 12.2;  1152 14.1 / 16.8;  1536 15.9 /
    // 19.0;  16/16: 64 11.8 / 10.8;  512 13.3 / 13.3;  768 14.9 / 15.3;  1536 21.0 / 24.7;  8/32: 64 15.4 / 13.5;  512 17.8 / 17.1;  768 20.7 / 20.2;  1536 28.1 / 32.0;
    // one wave each:  8/8: 3072 20.9 / 18.2;  16/16: 35.0 / 32.2.  Tiles:  8/8: 64 8.5 / 7.6;  384 9.5 / 8.7;  1152 13.2 / 13.8;  1536 15.1 / 15.6;  3072 16.7 / 14.5;
    // 16/16: 768 13.5 / 12.7;  1536 20.2 / 20.0;  3072 26.9 / 24.4;  8/32: 1536 26.0 / 26.0;  3072 50.6 / 43.5
    const int64_t groups = (int64_t)N1 / 16 * B * H;
#define LLSA_SPARSE(TPW, W)                                                                               \
    do {                                                                                                  \
        if (pq_par == nullptr) LLSA_SPARSE_P(TPW, W, 0, false);                                           \
        else if (N1 / 16 <= 64 && (tiled || W < 4 || groups <= 512)) LLSA_SPARSE_P(TPW, W, 4 / W, true);  \
        else if (N1 / 16 <= 64) LLSA_SPARSE_P(TPW, W, 4 / W, false);                                      \
        else LLSA_SPARSE_P(TPW, W, 16 / W, false);                                                        \
    } while (0)
    // few groups: four waves each, for the shorter chain of steps; many (2 waves per SIMD): as few as hold the keys, for fewer instructions
    const bool few = groups < 2048;
    if (T2 <= 4) LLSA_SPARSE(4, 1);
    else if (T2 <= 8 && few) LLSA_SPARSE(2, 4);
    else if (T2 <= 8) LLSA_SPARSE(8, 1);
    else if (T2 <= 16 && few) LLSA_SPARSE(4, 4);
    else if (T2 <= 16) LLSA_SPARSE(16, 1);
    else if (few) LLSA_SPARSE(8, 4);
    else LLSA_SPARSE(16, 2);
#undef LLSA_SPARSE
#undef LLSA_SPARSE_P
}

static int topk_sparse(const void* pq, const void* pk, const int32_t* parent_idx, int32_t* out_idx, int B, int H, int N1, int T, int T2, int tiled,
                       void* stream) {
    LLSA_REQUIRE(pq && pk && parent_idx && out_idx, "topk_sparse: null argument");
    LLSA_REQUIRE(B > 0 && H > 0 && N1 > 0 && N1 % 16 == 0, "topk_sparse: N1=%d must be a positive multiple of 16", N1);
    LLSA_REQUIRE(T2 >= 1 && T2 * 16 <= kMaxCand && T2 <= N1 / 16, "topk_sparse: need 1 <= T2 <= min(%d, N1/16), got %d", kMaxCand / 16, T2);
    LLSA_REQUIRE(T >= 1 && T <= kMaxT && T <= T2 * 16, "topk_sparse: need 1 <= T <= min(%d, 16*T2), got %d", kMaxT, T);
    LLSA_REQUIRE(aligned16(pq) && aligned16(pk), "topk_sparse: inputs must be 16-byte aligned");
    launch_sparse((const bf16*)pq, (const bf16*)pk, parent_idx, out_idx, B, H, N1, T, T2, nullptr, nullptr, nullptr, tiled, (hipStream_t)stream);
    return launch_status("topk_sparse");
}
extern "C" int llsa_topk_sparse(const void* pq, const void* pk, const int32_t* parent_idx, int32_t* out_idx, int B, int H, int N1, int T, int T2,
                                void* stream) {
    return topk_sparse(pq, pk, parent_idx, out_idx, B, H, N1, T, T2, 0, stream);
}
extern "C" int llsa_topk_sparse_tiles(const void* pq, const void* pk_tiles, const int32_t* parent_idx, int32_t* out_idx, int B, int H, int N1, int T,
                                      int T2, void* stream) {
    return topk_sparse(pq, pk_tiles, parent_idx, out_idx, B, H, N1, T, T2, 1, stream);
}

// (a wave selects its parent row sixteen times over: beyond a few hundred parent tokens the separate dense kernel is faster)
extern "C" int llsa_topk_cascade_max_parents(void) { return kCascadeMaxParents; }

static int topk_cascade(const void* pq_parent, const void* pk_parent, int32_t* parent_out, const void* pq, const void* pk, int32_t* out_idx, int B, int H,
                        int N1, int T, int T2, int tiled, void* stream) {
    LLSA_REQUIRE(pq_parent && pk_parent && parent_out && pq && pk && out_idx, "topk_cascade: null argument");
    LLSA_REQUIRE(B > 0 && H > 0 && N1 > 0 && N1 % 256 == 0, "topk_cascade: N1=%d must be a positive multiple of 256", N1);
    LLSA_REQUIRE(N1 / 16 <= kCascadeMaxParents, "topk_cascade: at most %d parent tokens (got %d): use llsa_topk_dense and llsa_topk_sparse",
                 kCascadeMaxParents, N1 / 16);
    LLSA_REQUIRE(T2 >= 1 && T2 * 16 <= kMaxCand && T2 <= N1 / 16, "topk_cascade: need 1 <= T2 <= min(%d, N1/16), got %d", kMaxCand / 16, T2);
    LLSA_REQUIRE(T >= 1 && T <= kMaxT && T <= T2 * 16, "topk_cascade: need 1 <= T <= min(%d, 16*T2), got %d", kMaxT, T);
    LLSA_REQUIRE(aligned16(pq) && aligned16(pk) && aligned16(pq_parent) && aligned16(pk_parent), "topk_cascade: inputs must be 16-byte aligned");
    launch_sparse((const bf16*)pq, (const bf16*)pk, nullptr, out_idx, B, H, N1, T, T2, (const bf16*)pq_parent, (const bf16*)pk_parent, parent_out,
                  tiled, (hipStream_t)stream);
    return launch_status("topk_cascade");
}
extern "C" int llsa_topk_cascade(const void* pq_parent, const void* pk_parent, int32_t* parent_out, const void* pq, const void* pk, int32_t* out_idx,
                                 int B, int H, int N1, int T, int T2, void* stream) {
    return topk_cascade(pq_parent, pk_parent, parent_out, pq, pk, out_idx, B, H, N1, T, T2, 0, stream);
}
extern "C" int llsa_topk_cascade_tiles(const void* pq_parent, const void* pk_parent_tiles, int32_t* parent_out, const void* pq, const void* pk_tiles,
                                       int32_t* out_idx, int B, int H, int N1, int T, int T2, void* stream) {
    return topk_cascade(pq_parent, pk_parent_tiles, parent_out, pq, pk_tiles, out_idx, B, H, N1, T, T2, 1, stream);
}
