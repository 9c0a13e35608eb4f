// The one-launch index transpose as a device function: a kernel of its own (transpose.hip), and workgroups of the forward attention
// kernel's launch (attn_fwd.hip).
#pragma once
#include "llsa_device.h"
#include "../../include/llsa_hip.h"

namespace llsa {

__device__ __forceinline__ int wave_incl_scan(int v, int lane) {
#pragma unroll
    for (int d = 1; d < kWave; d <<= 1) {
        const int o = __shfl_up(v, d);
        if (lane >= d) v += o;
    }
    return v;
}

// The middle step of every form of the transpose: counts per key block -> offsets, segment starts and the work list.
// count_of(i): entries of key block i; set_start(i, start): where the caller wants the start of segment i (its cursor);
// wave_tot: 5 * NT / 64 ints of LDS.  Called by all NT threads of the workgroup; `work` already points at the
// (b,h)'s list (or is nullptr).  E: the sum of all counts.
template <int NT, typename CountFn, typename StartFn>
__device__ __forceinline__ void offsets_and_work_list(CountFn count_of, StartFn set_start, int* wave_tot, int* __restrict__ offsets,
                                                       int* __restrict__ work, int Kb, int E, int chunk) {
    constexpr int NW = NT / kWave;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    // exclusive scan over the counts: each thread owns `per` consecutive counters
    const int per = (Kb + NT - 1) / NT;
    const int c0 = min(tid * per, Kb), c1 = min(c0 + per, Kb);
    // l_items: short items, l_long: long items (more than chunk/2 entries)
    const int long_min = chunk / 2 + 1;
    int local = 0, l_items = 0, l_slots = 0, l_multi = 0, l_long = 0;
    for (int i = c0; i < c1; i++) {
        const int c = count_of(i);
        const int nch = max(1, (c + chunk - 1) / chunk);
        const int n_long = (nch - 1) + ((c - (nch - 1) * chunk >= long_min) ? 1 : 0);   // all chunks but the last are full
        local += c;
        l_long += n_long;
        l_items += nch - n_long;
        l_slots += (nch > 1) ? nch : 0;
        l_multi += (nch > 1) ? 1 : 0;
    }
    const int incl = wave_incl_scan(local, lane);
    const int incl_i = wave_incl_scan(l_items, lane);
    const int incl_s = wave_incl_scan(l_slots, lane);
    const int incl_m = wave_incl_scan(l_multi, lane);
    const int incl_l = wave_incl_scan(l_long, lane);
    if (lane == kWave - 1) {
        wave_tot[wave] = incl;
        wave_tot[NW + wave] = incl_i;
        wave_tot[2 * NW + wave] = incl_s;
        wave_tot[3 * NW + wave] = incl_m;
        wave_tot[4 * NW + wave] = incl_l;
    }
    __syncthreads();
    int run = incl - local, run_i = incl_i - l_items, run_s = incl_s - l_slots, run_m = incl_m - l_multi, run_l = incl_l - l_long;
    // (five LDS reads in flight together; the sums over the waves go by readlane)
    int total_long = 0, tot[5];
#pragma unroll
    for (int k = 0; k < 5; k++) tot[k] = wave_tot[k * NW + (lane & (NW - 1))];
#pragma unroll
    for (int w = 0; w < NW; w++) {
        int o[5];
#pragma unroll
        for (int k = 0; k < 5; k++) o[k] = __builtin_amdgcn_readlane(tot[k], w);
        total_long += o[4];
        if (w < wave) {                                       // (uniform)
            run += o[0];
            run_i += o[1];
            run_s += o[2];
            run_m += o[3];
            run_l += o[4];
        }
    }
    run_i += total_long;                                      // short items follow the long ones
    const int max_items = E / chunk + Kb;
    for (int i = c0; i < c1; i++) {
        const int c = count_of(i);
        offsets[i] = run;
        set_start(i, run);
        run += c;
        if (work != nullptr) {
            const int nch = max(1, (c + chunk - 1) / chunk);
            for (int ci = 0; ci < nch; ci++) {
                const int n_ent = min(chunk, c - ci * chunk);
                int* it = work + 4 + 4 * ((n_ent >= long_min) ? run_l++ : run_i++);
                it[0] = i;
                it[1] = run - c + ci * chunk;                  // (run already points past this segment)
                it[2] = n_ent;
                it[3] = (nch > 1) ? run_s + ci : -1;
            }
            if (nch > 1) {
                int* m = work + 4 + 4 * max_items + 4 * run_m++;
                m[0] = i;
                m[1] = run_s;
                m[2] = nch;
                m[3] = 0;
            }
            run_s += (nch > 1) ? nch : 0;
        }
    }
    if (tid == NT - 1) offsets[Kb] = run;        // (the last thread's running sum is the total)
    if (work != nullptr && tid == NT - 1) {
        work[0] = run_i;                                      // (the last thread's short items end the list)
        work[1] = run_s;
        work[2] = run_m;
        work[3] = total_long;
    }
}

// The transpose of all levels of one operator call in one launch, sorted as it is built.  A workgroup owns a range of key
// blocks of one (b,h): it reads all entries, keeps one bitmap over the query blocks per key block of its range in LDS (one
// word of padding per row keeps the rows off each other's banks), and counts the entries below its range -- which is
// where its first segment starts, so that no word passes between workgroups.  A key block's segment is written by reading its
// row's bits back in order -- ascending query blocks with no scatter through atomic cursors and no sorting pass
// afterwards; the inverse position of an entry is its segment's start plus the bits below its own.  One more workgroup per (b,h)
// makes a histogram over all key blocks and from it offsets and work list.
// All counts are of entries.  A query block that names a key block twice (a top-k does not, a caller's own indices may) is one
// bit but two entries, and its segment is longer than its row has bits: such a segment is written again with as many copies of
// every query block as it has entries (write_repeats), and so are those entries' places in the inverse.
// Reading every entry once per range is cheap (4 a lane and load, from the L2), clearing and filling the bitmaps of
// the whole matrix in every workgroup was not (two levels of 12 x 16384 tokens 15.9 us), and a range fits LDS where the
// matrix does not.
struct TrJob {
    const int* idx; int* offsets; int* flat; int* work; int* inv;
    int Mb, Kb, T, chunk, work_stride;
    int parts, rows;                                          // ranges per (b,h), key blocks per range
    unsigned row_magic;                                       // entry i (of four, if `quads`) belongs to query block i * row_magic >> 32
    int sums;                                                 // see tr_stride
    int quads;                                                // T is a multiple of 4 and idx 16-byte aligned: entries are read four at a time
};
constexpr int kTrSums = 4;                                    // words to a sum where one for every word would cost ranges (tr_ranges)
struct TrJobs {
    TrJob job[LLSA_MAX_LEVELS];
    int n_jobs, wgs;                                          // workgroups per (b,h): job[i].parts + 1 for each job, one after the other
};
// ints of LDS per key block: its row of bits, its count and then its start, and for an inverse the bits in front of every `sums`-th word (0: no inverse)
__host__ __device__ inline int tr_stride(int Mb, int sums) {
    const int words = (Mb + 31) / 32;
    return words + 1 + (sums > 0 ? (words + sums - 1) / sums : 0);
}

// calls fn(key block, query block) for every entry of the (b,h), each in one thread
template <int NT, typename Fn>
__device__ __forceinline__ void tr_entries(const TrJob& jb, const int* __restrict__ idx, Fn fn) {
    const int tid = threadIdx.x, n = jb.quads ? jb.Mb * jb.T / 4 : jb.Mb * jb.T;
    constexpr int kBatch = 8;
    auto query = [&](int i) { return jb.row_magic == 0 ? i : (int)(((unsigned long long)(unsigned)i * jb.row_magic) >> 32); };
    if (jb.quads) {
        for (int i0 = 0; i0 < n; i0 += kBatch * NT) {     // eight loads in flight per thread
            i32x4 v[kBatch];
#pragma unroll
            for (int k = 0; k < kBatch; k++) v[k] = reinterpret_cast<const i32x4*>(idx)[min(i0 + k * NT + tid, n - 1)];
#pragma unroll
            for (int k = 0; k < kBatch; k++) {
                const int i = i0 + k * NT + tid;
                if (i < n) {
                    const int q = query(i);
#pragma unroll
                    for (int e = 0; e < 4; e++) fn(clampi(v[k][e], 0, jb.Kb - 1), q, 4 * i + e);
                }
            }
        }
    } else {
        for (int i = tid; i < n; i += NT) fn(clampi(idx[i], 0, jb.Kb - 1), query(i), i);
    }
}

// The segment of key block n (places `start` .. of flat) from words w_lo .. w_hi of its row of bits and from idx, one wave: every query
// block as often as it names n, and with `inv` the places of those entries.  Rare: only for a segment that is longer than its row has
// bits, after the bits alone have been written to it.
__device__ __forceinline__ void write_repeats(const int* __restrict__ idx, const unsigned* row, int w_lo, int w_hi, int n, int T, int Kb,
                                              int* flat, int* inv, int start, int lane) {
    for (int w = w_lo; w < w_hi; w++)
        for (unsigned wd = (unsigned)__builtin_amdgcn_readfirstlane((int)row[w]); wd != 0u; wd &= wd - 1u) {
            const int q = w * 32 + __ffs((int)wd) - 1;
            for (int t0 = 0; t0 < T; t0 += kWave) {
                const int64_t e = (int64_t)q * T + min(t0 + lane, T - 1);
                const bool names = t0 + lane < T && clampi(idx[e], 0, Kb - 1) == n;
                const unsigned long long all = __ballot(names);
                const int at = start + __popcll(all & ((1ull << lane) - 1ull));
                if (names) {
                    flat[at] = q;
                    if (inv != nullptr) inv[e] = at;
                }
                start += __popcll(all);
            }
        }
}

// Workgroup `block` of B * H * jobs.wgs, NT threads.  smem: what the plan asks for; wave_tot: tr_scratch_ints(NT) ints of LDS.
__host__ __device__ constexpr int tr_scratch_ints(int threads) { return 5 * threads / kWave + 2; }
template <int NT>
__device__ __forceinline__ void transpose_block(const TrJobs& jobs, int block, int* smem, int* wave_tot) {
    constexpr int NW = NT / kWave;
    int& range_end = wave_tot[5 * NW];                        // where the range's last segment ends
    int& repeats = wave_tot[5 * NW + 1];                      // whether a row of it has fewer bits than entries
    const int bh = block / jobs.wgs;
    int part = block % jobs.wgs, ji = 0;
    while (ji < jobs.n_jobs - 1 && part > jobs.job[ji].parts) part -= jobs.job[ji++].parts + 1;
    const TrJob& jb = jobs.job[ji];
    const int Mb = jb.Mb, Kb = jb.Kb, T = jb.T, E = Mb * T;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int* idx = jb.idx + (int64_t)bh * E;

    if (part == jb.parts) {                                   // offsets and work list
        for (int i = tid; i < Kb; i += NT) smem[i] = 0;
        __syncthreads();
        tr_entries<NT>(jb, idx, [&](int n, int, int) { atomicAdd(&smem[n], 1); });
        __syncthreads();
        offsets_and_work_list<NT>([&](int i) { return smem[i]; }, [](int, int) {}, wave_tot, jb.offsets + (int64_t)bh * (Kb + 1),
                              jb.work ? jb.work + (int64_t)bh * jb.work_stride : nullptr, Kb, E, jb.chunk);
        return;
    }

    const int words = (Mb + 31) / 32, stride = tr_stride(Mb, jb.sums);
    const int lo = part * jb.rows, nr = min(jb.rows, Kb - lo);       // > 0: the host leaves no range empty
    unsigned* bm = reinterpret_cast<unsigned*>(smem);         // [nr][stride]
    for (int i = tid; i < nr * stride; i += NT) bm[i] = 0u;
    if (tid == 0) repeats = 0;
    __syncthreads();
    int below = 0;
    tr_entries<NT>(jb, idx, [&](int n, int q, int) {
        const int r = n - lo;
        below += r < 0 ? 1 : 0;
        if ((unsigned)r < (unsigned)nr) {
            atomicOr(&bm[r * stride + (q >> 5)], 1u << (q & 31));
            atomicAdd(&bm[r * stride + words], 1u);           // the row's count, in its padding word
        }
    });
    below = wave_incl_scan(below, lane);
    if (lane == kWave - 1) wave_tot[wave] = below;
    __syncthreads();
    int start = 0, tot = wave_tot[lane & (NW - 1)];     // (one LDS read; the sums over the waves go by readlane)
#pragma unroll
    for (int w = 0; w < NW; w++) start += __builtin_amdgcn_readlane(tot, w);
    {   // the rows' starts take the place of the counts (a range has at most 256 rows)
        const int c = tid < nr ? (int)bm[tid * stride + words] : 0;
        const int incl = wave_incl_scan(c, lane);
        if (lane == kWave - 1) wave_tot[NW + wave] = incl;
        __syncthreads();
        tot = wave_tot[NW + (lane & (NW - 1))];
#pragma unroll
        for (int w = 0; w < NW; w++) {
            const int o = __builtin_amdgcn_readlane(tot, w);
            start += w < wave ? o : 0;
        }
        if (tid < nr) bm[tid * stride + words] = (unsigned)(start + incl - c);
        if (tid == nr - 1) range_end = start + incl;
    }
    __syncthreads();
    if (jb.inv != nullptr) {
        for (int r = tid; r < nr; r += NT) {
            unsigned* row = bm + r * stride;
            int before = 0;
            if (jb.sums == 1) {
#pragma unroll 4
                for (int w = 0; w < words; w++) {
                    row[words + 1 + w] = (unsigned)before;
                    before += __popc(row[w]);
                }
            } else {
#pragma unroll 4
                for (int w = 0; w < words; w++) {
                    if (w % kTrSums == 0) row[words + 1 + w / kTrSums] = (unsigned)before;
                    before += __popc(row[w]);
                }
            }
        }
        __syncthreads();
        int* inv = jb.inv + (int64_t)bh * E;
        tr_entries<NT>(jb, idx, [&](int n, int q, int e) {
            const int r = n - lo;
            if ((unsigned)r >= (unsigned)nr) return;
            const unsigned* row = bm + r * stride;
            const int w = q >> 5;
            int pos = (int)row[words] + __popc(row[w] & ((1u << (q & 31)) - 1u));
            if (jb.sums == 1) {
                pos += (int)row[words + 1 + w];
            } else {
                const int w0 = w / kTrSums * kTrSums;
                pos += (int)row[words + 1 + w / kTrSums];
#pragma unroll
                for (int i = 0; i < kTrSums - 1; i++) pos += __popc(w0 + i < w ? row[min(w0 + i, w)] : 0u);
            }
            inv[e] = pos;
        });
    }
    // The segments, ascending.  Eight neighbouring lanes share a row, each with an eighth of its words: the lanes count their
    // bits, a scan over the eight gives each its place in the segment, and each writes the query blocks of its own words.
    // (Stores of 4 bytes, every lane into a line of its own: with one lane per row a wave walked as many rounds as its longest
    // segment has entries.)
    const int sub = tid & 7, wps = (words + 7) / 8, w_lo = min(words, sub * wps), w_hi = min(words, w_lo + wps);
    int* flat = jb.flat + (int64_t)bh * E;
    for (int r0 = 0; r0 < nr; r0 += NT / 8) {
        const int r = r0 + (tid >> 3);
        const unsigned* row = bm + min(r, nr - 1) * stride;
        int mine = 0;
        if (r < nr)
            for (int w = w_lo; w < w_hi; w++) mine += __popc(row[w]);
        int incl = mine;                                      // (all lanes take part in the shuffles)
#pragma unroll
        for (int d = 1; d < 8; d <<= 1) {
            const int o = __shfl_up(incl, d, 8);
            if (sub >= d) incl += o;
        }
        if (r < nr) {
            int out = (int)row[words] + incl - mine;
            for (int w = w_lo; w < w_hi; w++) {
                unsigned wd = row[w];
                while (wd) {
                    flat[out++] = w * 32 + __ffs((int)wd) - 1;
                    wd &= wd - 1u;
                }
            }
        }
        if (r < nr && sub == 7 && (int)row[words] + incl != (r + 1 < nr ? (int)row[stride + words] : range_end)) repeats = 1;
    }
    __syncthreads();
    if (repeats == 0) return;                                 // (uniform)
    for (int r = wave; r < nr; r += NW) {
        const unsigned* row = bm + r * stride;
        const int start_r = __builtin_amdgcn_readfirstlane((int)row[words]);
        const int end = __builtin_amdgcn_readfirstlane(r + 1 < nr ? (int)row[stride + words] : range_end);
        int bits = 0;
        for (int w = 0; w < words; w++) bits += __popc((unsigned)__builtin_amdgcn_readfirstlane((int)row[w]));
        if (bits != end - start_r) write_repeats(idx, row, 0, words, lo + r, T, Kb, flat, jb.inv ? jb.inv + (int64_t)bh * E : nullptr, start_r, lane);
    }
}

// Plans all jobs for workgroups with `lds_ints` ints of LDS (at least one of 8160, see kTrLdsFwd); false if one of them does not fit
// the form or its arguments are wrong (which the caller finds out from the general entry point).
bool plan_transpose(const llsa_transpose_job* jobs, int n_jobs, int B, int H, int lds_ints, TrJobs& plan);

}  // namespace llsa
