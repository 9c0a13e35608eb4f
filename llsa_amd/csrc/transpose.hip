// Index transpose: query-major top-k lists -> key-major CSR (offsets + flat list), used by the dK/dV passes.  Up to 65536
// entries per (b,h) one launch makes the lists of all levels from bitmaps in LDS (transpose_bitmap_kernel).  Larger lists are
// a counting sort -- histogram, exclusive scan, scatter with a cursor -- after which every segment is put in ascending
// query-block order with a per-wave bitmap (set one bit per entry, then read the bits back in order).  Either way the result,
// and therefore the accumulation order of dK/dV, does not depend on the timing of atomics.  An entry that its row repeats
// counts as often as it is there.
#include "llsa_device.h"
#include "llsa_host.h"
#include "../../include/llsa_hip.h"
#include <algorithm>

namespace llsa {

// Threads per workgroup: 1024 where the kernel has the chip to itself.  Beside the forward attention kernel on another stream
// 256: a CU that kernel fills leaves room for one more wave of few registers per SIMD, and a workgroup of sixteen waves
// waits until the CU has drained.
constexpr int kTrThreads = 1024, kTrThreadsBeside = 256;

__device__ __forceinline__ int wave_incl_scan(int v, int lane) {
#pragma unroll
    for (int d = 1; d < kWave; d <<= 1) {
        const int o = __shfl_up(v, d);
        if (lane >= d) v += o;
    }
    return v;
}

constexpr int kTrPart = 16 * kTrThreadsBeside; // entries per workgroup of the split path
constexpr int kTrSplitMin = 65536;             // entries from which the split path is taken

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

// Work list (optional): the K-side kernels walk each key block's segment in chunks of at most
// `chunk` entries so that a popular key block does not serialise on one wave.  Per (b,h), all
// records 4 ints (16-byte aligned when the list is, so that one load fetches a record):
//   work[0] = number of items, work[1] = number of partial-sum slots, work[2] = number of key
//   blocks with more than one chunk, work[3] = number of items with more than chunk/2 entries (they come first),
//   work[4 + 4i ..]             item i = {key block n, first entry in flat, entries, partial-sum slot
//                               or -1 when n has one chunk}      (items of one key block are adjacent),
//   work[4 + 4 max_items + 4j ..] j-th key block with more than one chunk = {n, first slot, chunks, 0}.
// Every key block has at least one item (an unselected block's item has no entries and only
// writes zeros), and max_items = Mb*T/chunk + Kb.  Items with more than chunk/2 entries come first
// in the list: a wave walks its item serially, so the long ones have to start early or the kernel
// ends with a few waves still working.
// SPLIT = false: the whole job of one (b,h).  SPLIT = true (many entries): the middle step of three --
// tr_count_kernel has left the histogram in the tail of the work list, this kernel scans it, writes
// offsets and work list and leaves every segment's start in the same place as the cursor that
// tr_scatter_kernel advances.
template <bool SPLIT>
__global__ __launch_bounds__(SPLIT ? kTrThreadsBeside : kTrThreads) void transpose_indices_kernel(const int* __restrict__ idx, int* __restrict__ offsets,
                                                                      int* __restrict__ flat, int* __restrict__ work,
                                                                      int Mb, int Kb, int T, int chunk, int work_stride) {
    // These kernels run beside the forward attention kernel on a second stream and are on the
    // critical path of nothing until the backward starts, but one slow workgroup per (b,h) is all
    // there is of them: let their waves go first when they share a CU.
    __builtin_amdgcn_s_setprio(3);
    constexpr int NT = SPLIT ? kTrThreadsBeside : kTrThreads;
    HIP_DYNAMIC_SHARED(int, smem)
    int* pos = smem;                               // Kb
    int* wave_tot = smem + (SPLIT ? 0 : Kb);       // 5 ints per wave (the split form keeps no counters in LDS)

    const int tid = threadIdx.x;
    const int bh = blockIdx.x;
    const int E = Mb * T;
    idx += (int64_t)bh * E;
    flat += (int64_t)bh * E;
    offsets += (int64_t)bh * (Kb + 1);

    constexpr int kBatch = 16;
    int* tail = SPLIT ? work + (int64_t)bh * work_stride + (work_stride - work_tail_len(Kb)) : nullptr;
    if (!SPLIT) {
        for (int i = tid; i < Kb; i += NT) pos[i] = 0;
    }
    __syncthreads();
    // entries are taken 16 per thread at a time, all 16 loads issued before the first is used
    for (int e0 = 0; e0 < (SPLIT ? 0 : E); e0 += kBatch * NT) {
        int v[kBatch];
#pragma unroll
        for (int k = 0; k < kBatch; k++) {
            const int e = e0 + k * NT + tid;
            v[k] = (e < E) ? idx[e] : -1;
        }
#pragma unroll
        for (int k = 0; k < kBatch; k++)
            if (e0 + k * NT + tid < E) atomicAdd(&pos[clampi(v[k], 0, Kb - 1)], 1);
    }
    __syncthreads();

    if (work != nullptr) work += (int64_t)bh * work_stride;
    offsets_and_work_list<NT>([&](int i) { return SPLIT ? tail[i] : pos[i]; },
                          [&](int i, int start) {
                              if (SPLIT) tail[i] = start;
                              else pos[i] = start;
                          },
                          wave_tot, offsets, work, Kb, E, chunk);
    __syncthreads();

    for (int e0 = 0; e0 < (SPLIT ? 0 : E); e0 += kBatch * NT) {
        int v[kBatch];
#pragma unroll
        for (int k = 0; k < kBatch; k++) {
            const int e = e0 + k * NT + tid;
            v[k] = (e < E) ? idx[e] : -1;
        }
#pragma unroll
        for (int k = 0; k < kBatch; k++) {
            const int e = e0 + k * NT + tid;
            if (e < E) flat[atomicAdd(&pos[clampi(v[k], 0, Kb - 1)], 1)] = e / T;
        }
    }
    // pos[n] is now the END of segment n; the segments are sorted by sort_segments_kernel
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
    int quads;                                                // T is a multiple of 4 and idx 16-byte aligned: entries are read four at a time
};
struct TrJobs {
    TrJob job[LLSA_MAX_LEVELS];
    int n_jobs, wgs;                                          // workgroups per (b,h): job[i].parts + 1 for each job, one after the other
};
__host__ __device__ inline int tr_stride(int Mb) { return (Mb + 31) / 32 + 1; }

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

template <int NT>
__global__ __launch_bounds__(NT) void transpose_bitmap_kernel(TrJobs jobs) {
    constexpr int NW = NT / kWave;
    HIP_DYNAMIC_SHARED(int, smem)
    __shared__ int wave_tot[5 * NW];
    __shared__ int range_end, repeats;                        // where the range's last segment ends; whether a row of it has fewer bits than entries
    const int bh = blockIdx.x / jobs.wgs;
    int part = blockIdx.x % jobs.wgs, ji = 0;
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

    const int words = (Mb + 31) / 32, stride = words + 1;
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
        int* inv = jb.inv + (int64_t)bh * E;
        tr_entries<NT>(jb, idx, [&](int n, int q, int e) {
            const int r = n - lo;
            if ((unsigned)r >= (unsigned)nr) return;
            const unsigned* row = bm + r * stride;
            int pos = (int)row[words];
            for (int w = 0; w < (q >> 5); w++) pos += __popc(row[w]);
            inv[e] = pos + __popc(row[q >> 5] & ((1u << (q & 31)) - 1u));
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

// Split path, first and last step: one workgroup per kTrPart entries.
__global__ __launch_bounds__(kTrThreadsBeside) void tr_zero_kernel(int* __restrict__ work, int Kb, int work_stride) {
    int* tail = work + (int64_t)blockIdx.x * work_stride + (work_stride - work_tail_len(Kb));
    for (int i = threadIdx.x; i < Kb; i += kTrThreadsBeside) tail[i] = 0;
}
__global__ __launch_bounds__(kTrThreadsBeside) void tr_count_kernel(const int* __restrict__ idx, int* __restrict__ work, int E, int Kb,
                                                             int work_stride) {
    // (global atomics, no LDS histogram: this kernel runs beside the forward attention kernel, whose
    // workgroups leave no room for 64 KB of LDS, and its workgroups would wait for that kernel to end)
    __builtin_amdgcn_s_setprio(3);
    const int tid = threadIdx.x, bh = blockIdx.y;
    int* tail = work + (int64_t)bh * work_stride + (work_stride - work_tail_len(Kb));
    idx += (int64_t)bh * E;
    int v[16];
#pragma unroll
    for (int k = 0; k < 16; k++) {
        const int e = blockIdx.x * kTrPart + k * kTrThreadsBeside + tid;
        v[k] = (e < E) ? idx[e] : -1;
    }
#pragma unroll
    for (int k = 0; k < 16; k++)
        if (blockIdx.x * kTrPart + k * kTrThreadsBeside + tid < E) atomicAdd(&tail[clampi(v[k], 0, Kb - 1)], 1);
}
__global__ __launch_bounds__(kTrThreadsBeside) void tr_scatter_kernel(const int* __restrict__ idx, int* __restrict__ flat,
                                                               int* __restrict__ work, int E, int Kb, int T, int work_stride) {
    __builtin_amdgcn_s_setprio(3);
    const int tid = threadIdx.x, bh = blockIdx.y;
    int* cursor = work + (int64_t)bh * work_stride + (work_stride - work_tail_len(Kb));
    idx += (int64_t)bh * E;
    flat += (int64_t)bh * E;
    int v[16];
#pragma unroll
    for (int k = 0; k < 16; k++) {
        const int e = blockIdx.x * kTrPart + k * kTrThreadsBeside + tid;
        v[k] = (e < E) ? idx[e] : -1;
    }
#pragma unroll
    for (int k = 0; k < 16; k++) {
        const int e = blockIdx.x * kTrPart + k * kTrThreadsBeside + tid;
        if (e < E) flat[atomicAdd(&cursor[clampi(v[k], 0, Kb - 1)], 1)] = e / T;      // order inside a segment: sorted afterwards
    }
}

// Puts every segment of `flat` in ascending order: one wave per key block sets one bit per
// entry in a private LDS bitmap over the query blocks and reads the bits back in order.  Only the
// words between the smallest and the largest query block of the segment are cleared and read.  A segment with more entries than
// bits (a query block that names the key block twice) is written again (write_repeats).
__global__ __launch_bounds__(256) void sort_segments_kernel(const int* __restrict__ idx, const int* __restrict__ offsets,
                                                            int* __restrict__ flat, int Mb, int Kb, int T) {
    __builtin_amdgcn_s_setprio(3);
    HIP_DYNAMIC_SHARED(unsigned, bitmaps)                     // waves x words
    const int words = (Mb + 31) / 32;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int bh = blockIdx.y, n = blockIdx.x * (int)(blockDim.x >> 6) + wave;
    if (n >= Kb) return;                                      // no workgroup barrier below
    idx += (int64_t)bh * Mb * T;
    flat += (int64_t)bh * Mb * T;
    const int* o = offsets + (int64_t)bh * (Kb + 1) + n;
    const int s = o[0], e = o[1];
    if (e - s <= 1) return;
    int qlo = Mb - 1, qhi = 0;
    for (int i = s + lane; i < e; i += kWave) {
        const int q = clampi(flat[i], 0, Mb - 1);
        qlo = q < qlo ? q : qlo;
        qhi = q > qhi ? q : qhi;
    }
    for (int d = 1; d < kWave; d <<= 1) {
        const int a = __shfl_xor(qlo, d), b = __shfl_xor(qhi, d);
        qlo = a < qlo ? a : qlo;
        qhi = b > qhi ? b : qhi;
    }
    const int w_lo = qlo >> 5, w_hi = (qhi >> 5) + 1;         // the same in every lane
    unsigned* bm = bitmaps + wave * words;
    for (int w = w_lo + lane; w < w_hi; w += kWave) bm[w] = 0u;
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    for (int i = s + lane; i < e; i += kWave) {
        const int q = clampi(flat[i], 0, Mb - 1);
        atomicOr(&bm[q >> 5], 1u << (q & 31));
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    int out = s;
    for (int wb = w_lo; wb < w_hi; wb += kWave) {
        unsigned wd = (wb + lane < w_hi) ? bm[wb + lane] : 0u;
        const int cnt = __popc(wd);
        const int incl2 = wave_incl_scan(cnt, lane);
        int oo = out + incl2 - cnt;
        while (wd) {
            const int bit = __ffs((int)wd) - 1;
            flat[oo++] = (wb + lane) * 32 + bit;
            wd &= wd - 1;
        }
        out += __shfl(incl2, kWave - 1);
    }
    if (out == e) return;                                     // (the same in every lane)
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    write_repeats(idx, bm, w_lo, w_hi, n, T, Kb, flat, nullptr, s, lane);
}

// The inverse of the sorted lists: entry (query block q, slot t) of idx names key block n, and q sits somewhere in
// n's ascending segment of flat -- one thread per entry finds where by bisection.  (The copies of a query block that names the key
// block several times are neighbours there and belong to its slots in order.)
__global__ __launch_bounds__(256) void inverse_positions_kernel(const int* __restrict__ idx, const int* __restrict__ offsets,
                                                                const int* __restrict__ flat, int* __restrict__ inv, int Mb, int Kb,
                                                                int T) {
    const int e = blockIdx.x * 256 + threadIdx.x, bh = blockIdx.y;
    const int E = Mb * T;
    if (e >= E) return;
    const int q = e / T;
    const int n = clampi(idx[(int64_t)bh * E + e], 0, Kb - 1);
    const int* o = offsets + (int64_t)bh * (Kb + 1) + n;
    const int* f = flat + (int64_t)bh * E;
    int lo = o[0], hi = o[1] - 1;                             // the segment holds q: it is never empty
    while (lo < hi) {
        const int mid = (lo + hi) >> 1;
        if (f[mid] < q) lo = mid + 1;
        else hi = mid;
    }
    if (lo + 1 < o[1] && f[lo + 1] == q)
        for (int t = 0; t < e - q * T; t++) lo += clampi(idx[(int64_t)bh * E + q * T + t], 0, Kb - 1) == n ? 1 : 0;
    inv[(int64_t)bh * E + e] = clampi(lo, 0, E - 1);
}

}  // namespace llsa

using namespace llsa;

extern "C" int llsa_fine_chunk(int N) { return fine_chunk(N); }
extern "C" int llsa_fine_chunk_for(int B, int H, int N, int T) { return fine_chunk_for((int64_t)B * H, N, T); }

extern "C" int64_t llsa_work_list_len(int Mb, int Kb, int T, int chunk) {
    if (Mb <= 0 || Kb <= 0 || T <= 0 || chunk <= 0) return -1;
    const int64_t e = (int64_t)Mb * T;
    return 4 + 4 * (e / chunk + Kb) + 4 * (e / chunk + 1) + work_tail_len(Kb);
}

static int check_transpose_job(const int32_t* idx, const int32_t* offsets, const int32_t* flat, const int32_t* work, int B, int H, int Mb, int Kb,
                               int T, int chunk) {
    LLSA_REQUIRE(idx && offsets && flat, "transpose_indices: null argument");
    LLSA_REQUIRE(B > 0 && H > 0 && Mb > 0 && Kb > 0 && T > 0, "transpose_indices: bad shape");
    LLSA_REQUIRE(work == nullptr || chunk >= 1, "transpose_indices: work list needs chunk >= 1");
    return 0;
}

// Ranges of key blocks a job is cut into for transpose_bitmap_kernel, 0: too large for it.  At least so many that a range's bitmaps take
// at most 64 KB of LDS, and towards half the CUs over all (b,h): every range reads all entries, which is what a range's workgroup
// spends its time on beyond about four of them (with a workgroup for every CU two levels of 12 x 16384 tokens 15.3 us, so 12).
// More than 65536 entries (65536 tokens at topk 16) take as long here as the several kernels for large jobs take
// beside the attention kernel on another stream (131072 entries: step 928 against 923 us, 196608: 672 against 664).
constexpr int kTrLdsInts = 16 * 1024;
static int tr_parts(int Mb, int Kb, int T, int BH) {
    const int64_t stride = tr_stride(Mb), E = (int64_t)Mb * T;
    if (stride > kTrLdsInts || Kb > 2 * kTrLdsInts) return 0;
    const int most_rows = (int)std::min<int64_t>(kTrLdsInts / stride, kTrThreadsBeside);
    const int least = (Kb + most_rows - 1) / most_rows;
    if (E > 1 << 16) return 0;
    const int parts = std::max({least, std::min(std::max(128 / BH - 1, 4), Kb / 32), 1});
    const int rows = (Kb + parts - 1) / parts;
    return (Kb + rows - 1) / rows;                            // no empty range
}

// the jobs that are small enough, all in one launch
static int launch_bitmap_jobs(TrJobs& jobs, int n_jobs, int B, int H, bool beside, hipStream_t st) {
    int64_t ints = 0;
    jobs.wgs = 0;
    jobs.n_jobs = n_jobs;
    for (int i = 0; i < n_jobs; i++) {
        const TrJob& j = jobs.job[i];
        ints = std::max<int64_t>(ints, std::max<int64_t>((int64_t)j.rows * tr_stride(j.Mb), j.Kb));
        jobs.wgs += j.parts + 1;
    }
    const size_t lds = sizeof(int) * (size_t)ints;
    const void* kernel = beside ? (const void*)transpose_bitmap_kernel<kTrThreadsBeside> : (const void*)transpose_bitmap_kernel<kTrThreads>;
    if (lds > 60 * 1024) {
        hipError_t e = hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess) return fail(-101, "transpose_indices: cannot raise dynamic LDS to %zu bytes: %s", lds, hipGetErrorString(e));
    }
    if (beside)
        hipLaunchKernelGGL(HIP_KERNEL_NAME(transpose_bitmap_kernel<kTrThreadsBeside>), dim3(B * H * jobs.wgs), dim3(kTrThreadsBeside), lds, st, jobs);
    else
        hipLaunchKernelGGL(HIP_KERNEL_NAME(transpose_bitmap_kernel<kTrThreads>), dim3(B * H * jobs.wgs), dim3(kTrThreads), lds, st, jobs);
    return launch_status("transpose_indices");
}

static int transpose_general(const int32_t* idx, int32_t* offsets, int32_t* flat, int32_t* work, int32_t* inv, int B, int H, int Mb, int Kb,
                             int T, int chunk, void* stream) {
    const size_t lds = sizeof(int) * ((size_t)Kb + 128);
    static_assert(5 * kTrThreads / kWave <= 128, "wave totals must fit their LDS slot");
    LLSA_REQUIRE(lds <= 160 * 1024 || (work != nullptr && (int64_t)Mb * T >= kTrSplitMin),
                 "transpose_indices: Kb=%d needs %zu bytes of LDS (limit 163840)", Kb, lds);
    // the segment sort keeps one bitmap over the query blocks per wave: four waves a workgroup while they fit, then two, then one
    const size_t bitmap = sizeof(unsigned) * ((size_t)(Mb + 31) / 32);
    const int sort_waves = 4 * bitmap <= 160 * 1024 ? 4 : 2 * bitmap <= 160 * 1024 ? 2 : 1;
    const size_t lds_sort = bitmap * sort_waves;
    LLSA_REQUIRE(lds_sort <= 160 * 1024, "transpose_indices: Mb=%d needs %zu bytes of LDS for the segment sort (limit 163840)", Mb, lds_sort);
    const int64_t E = (int64_t)Mb * T;
    const bool split = work != nullptr && E >= kTrSplitMin;
    if (!split && lds > 64 * 1024) {
        hipError_t e = hipFuncSetAttribute((const void*)transpose_indices_kernel<false>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess) return fail(-101, "transpose_indices: cannot raise dynamic LDS to %zu bytes: %s", lds, hipGetErrorString(e));
    }
    const int wl = (int)llsa_work_list_len(Mb, Kb, T, chunk);
    hipStream_t st = (hipStream_t)stream;
    if (split) {
        // many entries: histogram and scatter spread over E / kTrPart workgroups per (b,h)
        const int parts = (int)((E + kTrPart - 1) / kTrPart);
        hipLaunchKernelGGL(tr_zero_kernel, dim3(B * H), dim3(kTrThreadsBeside), 0, st, work, Kb, wl);
        hipLaunchKernelGGL(tr_count_kernel, dim3(parts, B * H), dim3(kTrThreadsBeside), 0, st, idx, work, (int)E, Kb, wl);
        hipLaunchKernelGGL(HIP_KERNEL_NAME(transpose_indices_kernel<true>), dim3(B * H), dim3(kTrThreadsBeside), sizeof(int) * 128, st, idx,
                           offsets, flat, work, Mb, Kb, T, chunk, wl);
        hipLaunchKernelGGL(tr_scatter_kernel, dim3(parts, B * H), dim3(kTrThreadsBeside), 0, st, idx, flat, work, (int)E, Kb, T, wl);
    } else {
        hipLaunchKernelGGL(HIP_KERNEL_NAME(transpose_indices_kernel<false>), dim3(B * H), dim3(kTrThreads), lds, st, idx, offsets, flat,
                           work, Mb, Kb, T, chunk, wl);
    }
    if (lds_sort > 64 * 1024) {
        hipError_t e = hipFuncSetAttribute((const void*)sort_segments_kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_sort);
        if (e != hipSuccess) return fail(-101, "transpose_indices: cannot raise dynamic LDS to %zu bytes: %s", lds_sort, hipGetErrorString(e));
    }
    hipLaunchKernelGGL(sort_segments_kernel, dim3((Kb + sort_waves - 1) / sort_waves, B * H), dim3(64 * sort_waves), lds_sort,
                       (hipStream_t)stream, idx, (const int*)offsets, flat, Mb, Kb, T);
    if (inv != nullptr)
        hipLaunchKernelGGL(inverse_positions_kernel, dim3((unsigned)((E + 255) / 256), B * H), dim3(256), 0, (hipStream_t)stream, idx,
                           (const int*)offsets, (const int*)flat, inv, Mb, Kb, T);
    return launch_status("transpose_indices");
}

extern "C" int llsa_transpose_one_launch(int Mb, int Kb, int T, int B, int H) {
    return Mb > 0 && Kb > 0 && T > 0 && B > 0 && H > 0 && tr_parts(Mb, Kb, T, B * H) > 0;
}

extern "C" int llsa_transpose_indices_multi(const llsa_transpose_job* jobs, int n_jobs, int B, int H, void* stream) {
    LLSA_REQUIRE(jobs != nullptr && n_jobs >= 1 && n_jobs <= LLSA_MAX_LEVELS, "transpose_indices: 1..%d jobs, got %d", LLSA_MAX_LEVELS, n_jobs);
    TrJobs small;
    int n_small = 0;
    for (int i = 0; i < n_jobs; i++) {
        const llsa_transpose_job& j = jobs[i];
        const int rc = check_transpose_job(j.idx, j.offsets, j.flat, j.work, B, H, j.Mb, j.Kb, j.T, j.chunk);
        if (rc != 0) return rc;
    }
    for (int i = 0; i < n_jobs; i++) {
        const llsa_transpose_job& j = jobs[i];
        const int chunk = j.chunk < 1 ? 1 : j.chunk, parts = tr_parts(j.Mb, j.Kb, j.T, B * H);
        if (parts > 0) {
            TrJob& t = small.job[n_small++];
            t.idx = j.idx; t.offsets = j.offsets; t.flat = j.flat; t.work = j.work; t.inv = j.inv;
            t.Mb = j.Mb; t.Kb = j.Kb; t.T = j.T; t.chunk = chunk;
            t.work_stride = j.work ? (int)llsa_work_list_len(j.Mb, j.Kb, j.T, chunk) : 0;
            t.parts = parts;
            t.rows = (j.Kb + parts - 1) / parts;
            t.quads = j.T % 4 == 0 && aligned16(j.idx);
            const unsigned per = t.quads ? j.T / 4 : j.T;     // (i * ceil(2^32 / per) >> 32 is i / per while i * per < 2^32)
            t.row_magic = per == 1 ? 0u : (unsigned)((((uint64_t)1 << 32) + per - 1) / per);
        } else {
            const int rc = transpose_general(j.idx, j.offsets, j.flat, j.work, j.inv, B, H, j.Mb, j.Kb, j.T, chunk, stream);
            if (rc != 0) return rc;
        }
    }
    if (n_small > 0) return launch_bitmap_jobs(small, n_small, B, H, n_small < n_jobs, (hipStream_t)stream);
    return 0;
}

extern "C" int llsa_transpose_indices(const int32_t* idx, int32_t* offsets, int32_t* flat, int32_t* work, int32_t* inv, int B, int H,
                                      int Mb, int Kb, int T, int chunk, void* stream) {
    llsa_transpose_job j;
    j.idx = idx; j.offsets = offsets; j.flat = flat; j.work = work; j.inv = inv;
    j.Mb = Mb; j.Kb = Kb; j.T = T; j.chunk = chunk;
    return llsa_transpose_indices_multi(&j, 1, B, H, stream);
}
