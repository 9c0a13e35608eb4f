// Index transpose: query-major top-k lists -> key-major CSR (offsets + flat list), used by the dK/dV passes.  Up to 65536
// entries per (b,h) one launch makes the lists of all levels from bitmaps in LDS (transpose_bitmap_kernel).  Larger lists of a
// selection that is nested in the level above's are made from that one's (nested_*_kernel).  Any other larger list is a counting
// sort -- histogram, exclusive scan, scatter with a cursor -- after which every segment is put in ascending query-block order with
// a per-wave bitmap (set one bit per entry, then read the bits back in order).  Every way the result, and therefore the
// accumulation order of dK/dV, does not depend on the timing of atomics.  An entry that its row repeats counts as often as it is
// there (a nested selection has none).
#include "llsa_device.h"
#include "llsa_host.h"
#include "transpose_device.h"
#include "../../include/llsa_hip.h"
#include <algorithm>

namespace llsa {

// Threads per workgroup: 1024 where the kernel has the chip to itself.  Beside the forward attention kernel on another stream
// 256: a CU that kernel fills leaves room for one more wave of few registers per SIMD, and a workgroup of sixteen waves
// waits until the CU has drained.
constexpr int kTrThreads = 1024, kTrThreadsBeside = 256;

constexpr int kTrPart = 16 * kTrThreadsBeside; // entries per workgroup of the split path
constexpr int kTrSplitMin = 65536;             // entries from which the split path is taken

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

template <int NT>
__global__ __launch_bounds__(NT) void transpose_bitmap_kernel(TrJobs jobs) {
    HIP_DYNAMIC_SHARED(int, smem)
    __shared__ int wave_tot[tr_scratch_ints(NT)];
    transpose_block<NT>(jobs, blockIdx.x, smem, wave_tot);
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

// The lists of a level whose selection is nested (llsa_transpose_job.nested): the key blocks a query block names are children of those
// its parent, one of the next job's query blocks, names, each once.  So the sixteen segments under a parent key block are made of
// the query blocks under that parent's own segment, in its order, and no entry has to be looked for or sorted: a cell of sixteen by sixteen
// bits per entry of the parents' lists says which of the sixteen query blocks names which of the sixteen key blocks, and the cells of
// a parent key block lie side by side in its segment's order (the parents' inverse positions).  Four kernels: the cells, out of every
// entry once; the counts under every parent key block; their sums in front of each; the segments, offsets and work list.  They run beside the forward attention
// kernel, in waves of at most 32 registers, which fit beside that kernel's; so do the kernels for any list, whose atomics and sorting pass they replace.  The
// four alone / those kernels beside the forward, us: 6 x 16384 lists of 16 37 / 417, the forward with them 920 -> 850 (790 alone), 676 -> 600 with three
// levels (546 alone); 3 x 3072 lists of 64 35 / 153, 168 -> 148 (144 alone).  Training steps 4055 -> 3890, 3070 -> 2925, 676 -> 645.  (On the
// forward's own stream 3884, 2929 and 672.)
struct NestedJob {
    const int* idx; int* offsets; int* flat; int* work;       // the level itself
    const int* p_sel; const int* p_inv; const int* p_off; const int* p_flat;      // the parents' selection and its transpose
    unsigned* cells;                                          // (BH, owners * p_T, 8): bit 16 (j % 2) + i of word j / 2: query block i names key block j
    int* sums;                                                // (BH, parents, kNestedSums): see there
    int Mb, Kb, T, chunk, work_stride;
    int owners, parents, p_T;                                 // Mb / 16, Kb / 16
};
constexpr int kNestedMaxParents = kWave;                      // a parent's list lives in one lane per entry
// What is known of the sixteen key blocks under a parent key block: 0..4 their entries, items, slots, cut blocks and long items, then (after
// nested_scan_kernel) those of everything in front, 8..23 the entries of each.
constexpr int kNestedSums = 8 + kBlk;

__global__ __launch_bounds__(256) void nested_cells_kernel(NestedJob p) {
    __builtin_amdgcn_s_setprio(3);
    __shared__ unsigned rows[4][kNestedMaxParents * kBlk];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int G = blockIdx.x * 4 + wave, bh = blockIdx.y;
    if (G >= p.owners) return;                                // no workgroup barrier below
    unsigned* const mine = rows[wave];
    const int64_t list = ((int64_t)bh * p.owners + G) * p.p_T;
    const int parent = lane < p.p_T ? clampi(p.p_sel[list + lane], 0, p.parents - 1) : -1;
    const int pos = lane < p.p_T ? clampi(p.p_inv[list + lane], 0, p.owners * p.p_T - 1) : 0;
    for (int i = lane; i < p.p_T * kBlk; i += kWave) mine[i] = 0u;
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    const int per = p.T / 4, n = kBlk * per;                  // (T is a multiple of 4, rows are 16-byte aligned)
    const i32x4* e = reinterpret_cast<const i32x4*>(p.idx + ((int64_t)bh * p.Mb + (int64_t)G * kBlk) * p.T);
    for (int i0 = 0; i0 < n; i0 += kWave) {
        const int i = min(i0 + lane, n - 1), row = i / per;
        const i32x4 v = e[i];
        int at[4] = {-1, -1, -1, -1};
        for (int s = 0; s < p.p_T; s++) {
            const int o = __builtin_amdgcn_readlane(parent, s);
#pragma unroll
            for (int k = 0; k < 4; k++) at[k] = (clampi(v[k], 0, p.Kb - 1) >> 4) == o ? s : at[k];
        }
        if (i0 + lane < n)
#pragma unroll
            for (int k = 0; k < 4; k++)
                if (at[k] >= 0) atomicOr(&mine[at[k] * kBlk + (clampi(v[k], 0, p.Kb - 1) & (kBlk - 1))], 1u << row);
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    unsigned* const out = p.cells + (int64_t)bh * p.owners * p.p_T * 8;
    for (int i0 = 0; i0 < p.p_T * 8; i0 += kWave) {           // (every lane takes part in the shuffle)
        const int i = min(i0 + lane, p.p_T * 8 - 1);
        const int at = __shfl(pos, i >> 3);
        if (i0 + lane < p.p_T * 8) out[(int64_t)at * 8 + (i & 7)] = mine[2 * i] | mine[2 * i + 1] << 16;
    }
}

struct NestedItems { int entries, items, slots, multi, longs; };     // of a key block (offsets_and_work_list's counts), or sums of those
__device__ __forceinline__ NestedItems nested_items(int c, int chunk) {
    const int nch = max(1, (c + chunk - 1) / chunk);
    NestedItems t;
    t.entries = c;
    t.longs = (nch - 1) + ((c - (nch - 1) * chunk >= chunk / 2 + 1) ? 1 : 0);
    t.items = nch - t.longs;
    t.slots = nch > 1 ? nch : 0;
    t.multi = nch > 1 ? 1 : 0;
    return t;
}
template <typename Fn>
__device__ __forceinline__ NestedItems nested_each(const NestedItems& a, Fn fn) {
    return NestedItems{fn(a.entries), fn(a.items), fn(a.slots), fn(a.multi), fn(a.longs)};
}
__device__ __forceinline__ NestedItems operator+(const NestedItems& a, const NestedItems& b) {
    return NestedItems{a.entries + b.entries, a.items + b.items, a.slots + b.slots, a.multi + b.multi, a.longs + b.longs};
}
__device__ __forceinline__ NestedItems nested_load(const int* t) {
    const i32x4 v = *reinterpret_cast<const i32x4*>(t);
    return NestedItems{v[0], v[1], v[2], v[3], t[4]};
}
__device__ __forceinline__ void nested_store(int* t, const NestedItems& v) {
    *reinterpret_cast<i32x4*>(t) = i32x4{v.entries, v.items, v.slots, v.multi};
    t[4] = v.longs;
}
__device__ __forceinline__ void nested_range(const NestedJob& p, int bh, int c, int& p0, int& p1) {
    const int* o = p.p_off + (int64_t)bh * (p.parents + 1) + c;
    p0 = clampi(o[0], 0, p.owners * p.p_T);
    p1 = clampi(o[1], p0, p.owners * p.p_T);
}

__global__ __launch_bounds__(256) void nested_totals_kernel(NestedJob p) {
    __builtin_amdgcn_s_setprio(3);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int c = blockIdx.x * 4 + wave, bh = blockIdx.y;
    if (c >= p.parents) return;
    int p0, p1;
    nested_range(p, bh, c, p0, p1);
    const unsigned short* cells = reinterpret_cast<const unsigned short*>(p.cells + (int64_t)bh * p.owners * p.p_T * 8);
    int n = 0;                                                // entries of key block 16 c + j: a quarter of the cells a lane
#pragma unroll 4
    for (int q = p0 + (lane >> 4); q < p1; q += 4) n += __popc(cells[(int64_t)q * kBlk + (lane & 15)]);
    n += __shfl_xor(n, 16);
    n += __shfl_xor(n, 32);
    int* o = p.sums + ((int64_t)bh * p.parents + c) * kNestedSums;
    if (lane < kBlk) o[8 + lane] = n;
    NestedItems t = nested_items(n, p.chunk);
#pragma unroll
    for (int d = 1; d < kBlk; d <<= 1) t = t + nested_each(t, [&](int v) { return __shfl_xor(v, d); });
    if (lane == 0) nested_store(o, t);
}

// One workgroup per (b,h): the sums become those of everything in front of a parent key block, short items counted from the last long one on.
__global__ __launch_bounds__(256) void nested_scan_kernel(NestedJob p) {
    __builtin_amdgcn_s_setprio(3);
    __shared__ NestedItems wave_sum[4];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, bh = blockIdx.x;
    int* const sums = p.sums + (int64_t)bh * p.parents * kNestedSums;
    const int per = (p.parents + 255) / 256, c0 = min(tid * per, p.parents), c1 = min(c0 + per, p.parents);
    NestedItems own{0, 0, 0, 0, 0};
    for (int c = c0; c < c1; c++) own = own + nested_load(sums + (int64_t)c * kNestedSums);
    NestedItems incl = own;
#pragma unroll
    for (int d = 1; d < kWave; d <<= 1) {
        const NestedItems o = nested_each(incl, [&](int v) { return __shfl_up(v, d); });
        if (lane >= d) incl = incl + o;
    }
    if (lane == kWave - 1) wave_sum[wave] = incl;
    __syncthreads();
    NestedItems run = incl + nested_each(own, [](int v) { return -v; }), all{0, 0, 0, 0, 0};
#pragma unroll
    for (int w = 0; w < 4; w++) {
        const NestedItems o = wave_sum[w];
        all = all + o;
        if (w < wave) run = run + o;
    }
    run.items += all.longs;
    for (int c = c0; c < c1; c++) {
        const NestedItems t = nested_load(sums + (int64_t)c * kNestedSums);
        nested_store(sums + (int64_t)c * kNestedSums, run);
        run = run + t;
    }
    if (tid == 0) {
        p.offsets[(int64_t)bh * (p.Kb + 1) + p.Kb] = all.entries;
        if (p.work != nullptr)
            *reinterpret_cast<i32x4*>(p.work + (int64_t)bh * p.work_stride) = i32x4{all.longs + all.items, all.slots, all.multi, all.longs};
    }
}

// A wave per parent key block: offsets, work list and segments of its sixteen key blocks.
__global__ __launch_bounds__(256) void nested_lists_kernel(NestedJob p) {
    __builtin_amdgcn_s_setprio(3);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, j = lane & 15, part = lane >> 4;
    const int c = blockIdx.x * 4 + wave, bh = blockIdx.y;
    if (c >= p.parents) return;                               // no workgroup barrier below
    int p0, p1;
    nested_range(p, bh, c, p0, p1);
    const int* sums = p.sums + ((int64_t)bh * p.parents + c) * kNestedSums;
    const int count = sums[8 + j], E = p.Mb * p.T;
    const NestedItems own = nested_items(count, p.chunk);
    NestedItems incl = own;                                   // over the sixteen key blocks
#pragma unroll
    for (int d = 1; d < kBlk; d <<= 1) {
        const NestedItems o = nested_each(incl, [&](int v) { return __shfl_up(v, d, kBlk); });
        if (j >= d) incl = incl + o;
    }
    const NestedItems at = nested_load(sums) + nested_each(own, [](int v) { return -v; }) + incl;
    if (part == 0) {
        const int n = c * kBlk + j;
        p.offsets[(int64_t)bh * (p.Kb + 1) + n] = at.entries;
        if (p.work != nullptr) {
            int* const work = p.work + (int64_t)bh * p.work_stride;
            const int nch = max(1, (count + p.chunk - 1) / p.chunk), max_items = E / p.chunk + p.Kb;
            int i_long = at.longs, i_short = at.items;
            for (int ci = 0; ci < nch; ci++) {
                const int n_ent = min(p.chunk, count - ci * p.chunk);
                int* it = work + 4 + 4 * ((n_ent >= p.chunk / 2 + 1) ? i_long++ : i_short++);
                *reinterpret_cast<i32x4*>(it) = i32x4{n, at.entries + ci * p.chunk, n_ent, nch > 1 ? at.slots + ci : -1};
            }
            if (nch > 1) *reinterpret_cast<i32x4*>(work + 4 + 4 * max_items + 4 * at.multi) = i32x4{n, at.slots, nch, 0};
        }
    }
    // the segments: four cells of the parent's segment at a time, in order; the loads of two such steps go out together (of more: more registers than the forward's waves leave)
    const unsigned short* cells = reinterpret_cast<const unsigned short*>(p.cells + (int64_t)bh * p.owners * p.p_T * 8);
    const int* owner = p.p_flat + (int64_t)bh * p.owners * p.p_T;
    int* const flat = p.flat + (int64_t)bh * E;
    int base = at.entries;
    constexpr int kBatch = 2;
    for (int q0 = p0; q0 < p1; q0 += 4 * kBatch) {
        unsigned bits[kBatch];
        int first[kBatch];
#pragma unroll
        for (int k = 0; k < kBatch; k++) {
            const int q = q0 + 4 * k + part, in = min(q, p1 - 1);
            bits[k] = cells[(int64_t)in * kBlk + j];
            first[k] = owner[in] * kBlk;
            if (q >= p1) bits[k] = 0u;
        }
#pragma unroll
        for (int k = 0; k < kBatch; k++) {
            const int n = __popc(bits[k]), n0 = __shfl(n, j), n1 = __shfl(n, 16 + j), n2 = __shfl(n, 32 + j), n3 = __shfl(n, 48 + j);
            int out = base + (part > 0 ? n0 : 0) + (part > 1 ? n1 : 0) + (part > 2 ? n2 : 0);
            while (bits[k]) {
                flat[out++] = first[k] + __ffs((int)bits[k]) - 1;
                bits[k] &= bits[k] - 1u;
            }
            base += (n0 + n1) + (n2 + n3);
        }
    }
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
// More than 65536 entries take longer here than lists made from those of the level above take beside the attention kernel on another stream where there are
// many key blocks, up to 65536 the nested form takes longer or as long.  Training steps of two levels, topk 16/16, us, here / nested: 12 x 16384 tokens (16384 entries)
// 289 / 306;  6 x 32768 313 / 359;  2 x 65536 (65536) 272 / 316;  6 x 65536 642 / 644;  16 x 65536 1697 / 1686;  32 x 65536 3329 / 3298;  2 x 131072 (131072) 564 / 534;  6 x
// 131072 1526 / 1462;  3 x 196608 1363 / 1268.  (With few key blocks and long lists this form is the faster one beyond that line too: 3 x 65536 at 32/16, 131072
// entries, 462 / 476;  3 x 49152 at 64/32, 196608, 617 / 626;  one level, 6 x 65536 at 32, against the counting sort 2196 / 2205.)
constexpr int kTrLdsInts = 16 * 1024;
static int tr_parts(int Mb, int Kb, int T, int BH, int sums, int lds_ints = kTrLdsInts, int histogram_ints = 2 * kTrLdsInts) {
    const int64_t stride = tr_stride(Mb, sums), E = (int64_t)Mb * T;
    if (stride > lds_ints || Kb > histogram_ints) return 0;
    const int most_rows = (int)std::min<int64_t>(lds_ints / stride, kTrThreadsBeside);
    const int least = (Kb + most_rows - 1) / most_rows;
    if (E > 1 << 16) return 0;
    const int parts = std::max({least, std::min(std::max(128 / BH - 1, 4), Kb / 32), 1});
    const int rows = (Kb + parts - 1) / parts;
    return (Kb + rows - 1) / rows;                            // no empty range
}

// The ranges of a job and, for an inverse, after how many words of a row there is a sum (tr_stride).  An entry that adds up the words in front of its own
// itself waits for as many LDS reads; a sum for every word doubles a key block's LDS and, where LDS decides, the ranges, each of which reads all
// entries.  us, no sums / every word / every fourth:  1 x 1024 key blocks, lists of 16, 14.0 / 10.5 / 11.0;  6 x 1024 16.0 / 11.3 / 12.1;  6 x 2048 25.4 / 17.3 /
// 17.3;  and where every word's would take more ranges 48 x 1024 19.5 / 26.4 / 15.9;  96 x 1024 36.2 / 41.2 / 31.0;  6 x 4096 48.0 / 46.0 / 26.0;
// 6 x 8192, lists of 8, 117 / 186 / 92;  1 x 16384, lists of 4, 100 / 188 / 85 (every eighth 6 x 4096 28.1, 6 x 8192 92.6, 1 x 16384 81).
struct TrRanges { int parts, sums; };
static TrRanges tr_ranges(const llsa_transpose_job& j, int BH, int lds_ints = kTrLdsInts, int histogram_ints = 2 * kTrLdsInts) {
    const int least = tr_parts(j.Mb, j.Kb, j.T, BH, 0, lds_ints, histogram_ints);
    if (j.inv == nullptr) return {least, 0};
    if (tr_parts(j.Mb, j.Kb, j.T, BH, 1, lds_ints, histogram_ints) == least) return {least, 1};
    return {tr_parts(j.Mb, j.Kb, j.T, BH, kTrSums, lds_ints, histogram_ints), kTrSums};
}

static void add_to_plan(TrJobs& plan, const llsa_transpose_job& j, const TrRanges& ranges) {
    const int parts = ranges.parts;
    TrJob& t = plan.job[plan.n_jobs++];
    t.idx = j.idx; t.offsets = j.offsets; t.flat = j.flat; t.work = j.work; t.inv = j.inv;
    t.Mb = j.Mb; t.Kb = j.Kb; t.T = j.T; t.chunk = j.chunk < 1 ? 1 : j.chunk;
    t.work_stride = j.work ? (int)llsa_work_list_len(j.Mb, j.Kb, j.T, t.chunk) : 0;
    t.parts = parts;
    t.sums = ranges.sums;
    t.rows = (j.Kb + parts - 1) / parts;
    t.quads = j.T % 4 == 0 && aligned16(j.idx);
    const unsigned per = t.quads ? j.T / 4 : j.T;             // (i * ceil(2^32 / per) >> 32 is i / per while i * per < 2^32)
    t.row_magic = per == 1 ? 0u : (unsigned)((((uint64_t)1 << 32) + per - 1) / per);
    plan.wgs += parts + 1;
}

bool llsa::plan_transpose(const llsa_transpose_job* jobs, int n_jobs, int B, int H, int lds_ints, TrJobs& plan) {
    plan = TrJobs{};
    for (int i = 0; i < n_jobs; i++) {
        const llsa_transpose_job& j = jobs[i];
        if (check_transpose_job(j.idx, j.offsets, j.flat, j.work, B, H, j.Mb, j.Kb, j.T, j.chunk) != 0) return false;
        const TrRanges ranges = tr_ranges(j, B * H, lds_ints, lds_ints);
        if (ranges.parts == 0) return false;
        add_to_plan(plan, j, ranges);
    }
    return true;
}

// the jobs that are small enough, all in one launch
static int launch_bitmap_jobs(const TrJobs& jobs, int B, int H, bool beside, hipStream_t st) {
    int64_t ints = 0;
    for (int i = 0; i < jobs.n_jobs; i++) {
        const TrJob& j = jobs.job[i];
        ints = std::max<int64_t>(ints, std::max<int64_t>((int64_t)j.rows * tr_stride(j.Mb, j.sums), j.Kb));
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
    return Mb > 0 && Kb > 0 && T > 0 && B > 0 && H > 0 && tr_parts(Mb, Kb, T, B * H, 0) > 0;
}

extern "C" int64_t llsa_transpose_nested_bytes(int Mb, int Kb, int T_parent, int B, int H) {
    if (Mb <= 0 || Kb <= 0 || Mb % kBlk != 0 || Kb % kBlk != 0 || T_parent <= 0 || T_parent > kNestedMaxParents || B <= 0 || H <= 0) return -1;
    return (int64_t)B * H * ((int64_t)(Mb / kBlk) * T_parent * 32 + (int64_t)(Kb / kBlk) * kNestedSums * (int64_t)sizeof(int));
}

static int check_nested_job(const llsa_transpose_job& j, const llsa_transpose_job& above, int B, int H) {
    LLSA_REQUIRE(j.inv == nullptr && above.inv != nullptr && above.Mb * kBlk == j.Mb && above.Kb * kBlk == j.Kb && above.T <= kNestedMaxParents,
                 "transpose_indices: a nested job needs no inverse, and the job above its parents' lists with theirs");
    LLSA_REQUIRE(j.T % 4 == 0 && aligned16(j.idx) && aligned16(j.work) && aligned16(j.nested) && (int64_t)j.Mb * j.T < (int64_t)1 << 31 && B * H <= 65535,
                 "transpose_indices: a nested job's entries are read four at a time");
    return 0;
}
// job: its lists are made from those of `above`, which are there
static int transpose_nested(const llsa_transpose_job& j, const llsa_transpose_job& above, int B, int H, hipStream_t st) {
    NestedJob p;
    p.idx = j.idx; p.offsets = j.offsets; p.flat = j.flat; p.work = j.work;
    p.p_sel = above.idx; p.p_inv = above.inv; p.p_off = above.offsets; p.p_flat = above.flat;
    p.Mb = j.Mb; p.Kb = j.Kb; p.T = j.T; p.chunk = j.chunk < 1 ? 1 : j.chunk;
    p.work_stride = j.work ? (int)llsa_work_list_len(j.Mb, j.Kb, j.T, p.chunk) : 0;
    p.owners = above.Mb; p.parents = above.Kb; p.p_T = above.T;
    p.cells = (unsigned*)j.nested;
    p.sums = (int*)j.nested + (int64_t)B * H * p.owners * p.p_T * 8;
    const int BH = B * H;
    hipLaunchKernelGGL(nested_cells_kernel, dim3((p.owners + 3) / 4, BH), dim3(256), 0, st, p);
    hipLaunchKernelGGL(nested_totals_kernel, dim3((p.parents + 3) / 4, BH), dim3(256), 0, st, p);
    hipLaunchKernelGGL(nested_scan_kernel, dim3(BH), dim3(256), 0, st, p);
    hipLaunchKernelGGL(nested_lists_kernel, dim3((p.parents + 3) / 4, BH), dim3(256), 0, st, p);
    return launch_status("transpose_indices");
}

extern "C" int llsa_transpose_indices_multi(const llsa_transpose_job* jobs, int n_jobs, int B, int H, void* stream) {
    LLSA_REQUIRE(jobs != nullptr && n_jobs >= 1 && n_jobs <= LLSA_MAX_LEVELS, "transpose_indices: 1..%d jobs, got %d", LLSA_MAX_LEVELS, n_jobs);
    TrJobs small{};
    for (int i = 0; i < n_jobs; i++) {
        const llsa_transpose_job& j = jobs[i];
        const int rc = check_transpose_job(j.idx, j.offsets, j.flat, j.work, B, H, j.Mb, j.Kb, j.T, j.chunk);
        if (rc != 0) return rc;
        if (j.nested == nullptr) continue;
        LLSA_REQUIRE(i + 1 < n_jobs, "transpose_indices: no job above a nested one");
        const int rc2 = check_nested_job(j, jobs[i + 1], B, H);
        if (rc2 != 0) return rc2;
    }
    bool several = false;                                     // kernels of small workgroups beside the forward
    for (int i = 0; i < n_jobs; i++) {
        const llsa_transpose_job& j = jobs[i];
        if (j.nested != nullptr) {
            several = true;
            continue;
        }
        const int chunk = j.chunk < 1 ? 1 : j.chunk;
        const TrRanges ranges = tr_ranges(j, B * H);
        if (ranges.parts > 0) {
            add_to_plan(small, j, ranges);
        } else {
            const int rc = transpose_general(j.idx, j.offsets, j.flat, j.work, j.inv, B, H, j.Mb, j.Kb, j.T, chunk, stream);
            if (rc != 0) return rc;
            several = true;
        }
    }
    if (small.n_jobs > 0) {
        const int rc = launch_bitmap_jobs(small, B, H, several, (hipStream_t)stream);
        if (rc != 0) return rc;
    }
    for (int i = n_jobs - 2; i >= 0; i--) {                   // from the coarsest down: every one's parents are done
        if (jobs[i].nested == nullptr) continue;
        const int rc = transpose_nested(jobs[i], jobs[i + 1], B, H, (hipStream_t)stream);
        if (rc != 0) return rc;
    }
    return 0;
}

extern "C" int llsa_transpose_indices(const int32_t* idx, int32_t* offsets, int32_t* flat, int32_t* work, int32_t* inv, int B, int H,
                                      int Mb, int Kb, int T, int chunk, void* stream) {
    llsa_transpose_job j{};
    j.idx = idx; j.offsets = offsets; j.flat = flat; j.work = work; j.inv = inv;
    j.Mb = Mb; j.Kb = Kb; j.T = T; j.chunk = chunk;
    return llsa_transpose_indices_multi(&j, 1, B, H, stream);
}
