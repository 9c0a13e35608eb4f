// Index transpose: query-major top-k lists -> key-major CSR (offsets + flat list), used by the dK/dV passes.  Up to 65536
// entries per (b,h) one launch makes the lists of all levels from bitmaps in LDS (transpose_bitmap_kernel).  Larger lists are
// a counting sort -- histogram, exclusive scan, scatter with a cursor -- after which every segment is put in ascending
// query-block order with a per-wave bitmap (set one bit per entry, then read the bits back in order).  Either way the result,
// and therefore the accumulation order of dK/dV, does not depend on the timing of atomics.  An entry that its row repeats
// counts as often as it is there.
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
static int tr_parts(int Mb, int Kb, int T, int BH, int lds_ints = kTrLdsInts, int histogram_ints = 2 * kTrLdsInts) {
    const int64_t stride = tr_stride(Mb), E = (int64_t)Mb * T;
    if (stride > lds_ints || Kb > histogram_ints) return 0;
    const int most_rows = (int)std::min<int64_t>(lds_ints / stride, kTrThreadsBeside);
    const int least = (Kb + most_rows - 1) / most_rows;
    if (E > 1 << 16) return 0;
    const int parts = std::max({least, std::min(std::max(128 / BH - 1, 4), Kb / 32), 1});
    const int rows = (Kb + parts - 1) / parts;
    return (Kb + rows - 1) / rows;                            // no empty range
}

static void add_to_plan(TrJobs& plan, const llsa_transpose_job& j, int parts) {
    TrJob& t = plan.job[plan.n_jobs++];
    t.idx = j.idx; t.offsets = j.offsets; t.flat = j.flat; t.work = j.work; t.inv = j.inv;
    t.Mb = j.Mb; t.Kb = j.Kb; t.T = j.T; t.chunk = j.chunk < 1 ? 1 : j.chunk;
    t.work_stride = j.work ? (int)llsa_work_list_len(j.Mb, j.Kb, j.T, t.chunk) : 0;
    t.parts = parts;
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
        const int parts = tr_parts(j.Mb, j.Kb, j.T, B * H, lds_ints, lds_ints);
        if (parts == 0) return false;
        add_to_plan(plan, j, parts);
    }
    return true;
}

// the jobs that are small enough, all in one launch
static int launch_bitmap_jobs(const TrJobs& jobs, int B, int H, bool beside, hipStream_t st) {
    int64_t ints = 0;
    for (int i = 0; i < jobs.n_jobs; i++) {
        const TrJob& j = jobs.job[i];
        ints = std::max<int64_t>(ints, std::max<int64_t>((int64_t)j.rows * tr_stride(j.Mb), j.Kb));
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
    TrJobs small{};
    for (int i = 0; i < n_jobs; i++) {
        const llsa_transpose_job& j = jobs[i];
        const int rc = check_transpose_job(j.idx, j.offsets, j.flat, j.work, B, H, j.Mb, j.Kb, j.T, j.chunk);
        if (rc != 0) return rc;
    }
    for (int i = 0; i < n_jobs; i++) {
        const llsa_transpose_job& j = jobs[i];
        const int chunk = j.chunk < 1 ? 1 : j.chunk, parts = tr_parts(j.Mb, j.Kb, j.T, B * H);
        if (parts > 0) {
            add_to_plan(small, j, parts);
        } else {
            const int rc = transpose_general(j.idx, j.offsets, j.flat, j.work, j.inv, B, H, j.Mb, j.Kb, j.T, chunk, stream);
            if (rc != 0) return rc;
        }
    }
    if (small.n_jobs > 0) return launch_bitmap_jobs(small, B, H, small.n_jobs < n_jobs, (hipStream_t)stream);
    return 0;
}

extern "C" int llsa_transpose_indices(const int32_t* idx, int32_t* offsets, int32_t* flat, int32_t* work, int32_t* inv, int B, int H,
                                      int Mb, int Kb, int T, int chunk, void* stream) {
    llsa_transpose_job j;
    j.idx = idx; j.offsets = offsets; j.flat = flat; j.work = work; j.inv = inv;
    j.Mb = Mb; j.Kb = Kb; j.T = T; j.chunk = chunk;
    return llsa_transpose_indices_multi(&j, 1, B, H, stream);
}
