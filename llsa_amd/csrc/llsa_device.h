// Device-side building blocks shared by the gfx950 kernels: vector types, the bf16
// 16x16x32 MFMA wrapper with its register layout, 64-lane reductions, bf16 rounding.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <utility>
#include "../../include/llsa_hip.h"

namespace llsa {

typedef __bf16 bf16;
typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2;
typedef __attribute__((ext_vector_type(4))) __bf16 bf16x4;
typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(2))) float f32x2;
typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((ext_vector_type(4))) unsigned u32x4;
typedef __attribute__((ext_vector_type(4))) int i32x4;

constexpr int kWave = 64;        // CDNA wavefront
constexpr int kBlk = 16;         // tokens per block (block_size of the operator)
constexpr int kD = 64;           // head dimension the MFMA kernels are specialised for
constexpr float kLog2e = 1.4426950408889634f;
constexpr float kLn2 = 0.6931471805599453f;
constexpr float kScale = 0.125f;                          // 1/sqrt(kD)
constexpr float kScaleLog2e = 0.125f * 1.4426950408889634f;

// v_mfma_f32_16x16x32_bf16:  D(16x16) = A(16x32) * B(32x16) + C.
//   lane l supplies  A[row = l%16][k = 8*(l/16) + e]   e = 0..7
//                    B[k = 8*(l/16) + e][col = l%16]
//   and owns         D[row = 4*(l/16) + e][col = l%16] e = 0..3
// Both operands are "8 consecutive k for one row/column", i.e. a 16-byte load from a
// row-major matrix whose fast axis is the contraction axis.
__device__ __forceinline__ f32x4 mfma_bf16(bf16x8 a, bf16x8 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ bf16x8 ld16(const bf16* p) { return *reinterpret_cast<const bf16x8*>(p); }
__device__ __forceinline__ bf16x4 ld8(const bf16* p) { return *reinterpret_cast<const bf16x4*>(p); }
__device__ __forceinline__ void st16(bf16* p, bf16x8 v) { *reinterpret_cast<bf16x8*>(p) = v; }
// the same without a claim to the caches: for data that is not read again before much else has passed through them
__device__ __forceinline__ bf16x8 ld16_stream(const bf16* p) { return __builtin_nontemporal_load(reinterpret_cast<const bf16x8*>(p)); }
__device__ __forceinline__ void st8(bf16* p, bf16x4 v) { *reinterpret_cast<bf16x4*>(p) = v; }

__device__ __forceinline__ bf16x8 cat(bf16x4 lo, bf16x4 hi) {
    return __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
}
__device__ __forceinline__ bf16x8 zero8() {
    bf16x8 z;
#pragma unroll
    for (int i = 0; i < 8; i++) z[i] = (bf16)0.0f;
    return z;
}
__device__ __forceinline__ bf16x4 zero4() {
    bf16x4 z;
#pragma unroll
    for (int i = 0; i < 4; i++) z[i] = (bf16)0.0f;
    return z;
}
__device__ __forceinline__ bf16x4 cvt4(f32x4 v) {
    bf16x4 r;
#pragma unroll
    for (int i = 0; i < 4; i++) r[i] = (bf16)v[i];
    return r;
}

// The value has to exist in vector registers here: what computes it cannot be moved to its use.  (The register class is the
// GPU's; the CPU build of these sources has no such constraint and nothing to hold back.)
__device__ __forceinline__ void pin_in_registers(bf16x8& v) {
#ifndef LLSA_CPU_EMU_BUILD
    asm volatile("" : "+v"(v));
#endif
}

// round-to-nearest-even through bf16, value kept in fp32
__device__ __forceinline__ float rn_bf16(float x) { return (float)(bf16)x; }

__device__ __forceinline__ float exp2_fast(float x) { return __builtin_amdgcn_exp2f(x); }

// Reductions over the four lanes {l, l^16, l^32, l^48} that share one MFMA column, with the lane
// swaps of gfx950 (v_permlane16_swap, v_permlane32_swap: vector-ALU instructions, where a shuffle
// goes through the LDS unit and makes the wave wait for it).  swap16(v, v) leaves in its two
// results v of this lane and v of lane l^16 (which is which depends on the row), swap32 the same
// for l^32; both reductions are symmetric, so every lane of the four ends with the same bits.
typedef __attribute__((ext_vector_type(2))) unsigned u32x2;
__device__ __forceinline__ float quad_max(float v) {
    u32x2 a = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1]));
    u32x2 b = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return fmaxf(__uint_as_float(b[0]), __uint_as_float(b[1]));
}
__device__ __forceinline__ float quad_sum(float v) {
    u32x2 a = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = __uint_as_float(a[0]) + __uint_as_float(a[1]);
    u32x2 b = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return __uint_as_float(b[0]) + __uint_as_float(b[1]);
}

// The value of lane l ^ XOR, for what a move inside a vector instruction can reach (rows of 16 lanes turned by 8, halves of 8 mirrored, quads permuted): a
// shuffle goes through the LDS unit.
template <int XOR>
__device__ __forceinline__ float across(float v) {
    static_assert(XOR == 8 || XOR == 7 || XOR == 2 || XOR == 1, "no such move");
#ifndef LLSA_CPU_EMU_BUILD
    constexpr int kMove = XOR == 8 ? 0x128 : XOR == 7 ? 0x141 : XOR == 2 ? 0x4E : 0xB1;       // row_ror:8, row_half_mirror, quad_perm
    return __uint_as_float((unsigned)__builtin_amdgcn_update_dpp(0, (int)__float_as_uint(v), kMove, 0xf, 0xf, true));
#else
    return __shfl_xor(v, XOR);
#endif
}
// Sum over lanes l ^ 0 .. 7, the same bits in all eight
__device__ __forceinline__ float octet_sum(float v) {
    v += across<1>(v);
    v += across<2>(v);
    return v + across<7>(v);                                  // (all lanes of a quad have the same sum)
}

// Sixteen token rows out of the accumulator layout: this lane's o[dt] are channels 16 dt + 4 (l/16) .. +3 of token l%16, whose row starts at `row`.
// In pieces of 8 bytes of sixteen rows at a time every piece is an access of its own in the L1, and a work item of the K side had as many of
// those in its stores as in the tiles of eight list entries.  Swapped between neighbouring sixteens of lanes the pieces are 16 bytes and the half
// rows of a store 64.  48 x 16384 tokens, forward 237 -> 230 us, K side 319 -> 306.5; 24 x 4096, topk 16, 29.9 -> 28.6 and 39.8 -> 38.3; 6 x 262144, K
// side 702 -> 665.  (Through 2 KB of LDS, whole rows a store: 654 there, but 311 and 67.3 against 66.0 at 12 x 16384, and the step the same.)
// wide: rows 16-byte aligned (uniform); stored as they are otherwise.
__device__ __forceinline__ void store_rows(bf16* row, const bf16x4 (&o)[4], int quad, bool wide) {
    if (wide) {
#pragma unroll
        for (int p = 0; p < 2; p++) {
            const u32x2 a = __builtin_bit_cast(u32x2, o[2 * p]), b = __builtin_bit_cast(u32x2, o[2 * p + 1]);
            const u32x2 lo = __builtin_amdgcn_permlane16_swap(a[0], b[0], false, false), hi = __builtin_amdgcn_permlane16_swap(a[1], b[1], false, false);
            st16(row + 32 * p + 16 * (quad & 1) + 8 * (quad >> 1), __builtin_bit_cast(bf16x8, u32x4{lo[0], hi[0], lo[1], hi[1]}));
        }
    } else {
#pragma unroll
        for (int dt = 0; dt < 4; dt++) st8(row + 16 * dt + 4 * quad, o[dt]);
    }
}
// The other way round: x[dt] = channels 16 dt + 4 (l/16) .. +3 of the row at `row` (16-byte aligned), requested and, once it is there, put in order
__device__ __forceinline__ void request_rows(bf16x8 (&raw)[2], const bf16* row, int quad) {
#pragma unroll
    for (int p = 0; p < 2; p++) raw[p] = ld16(row + 32 * p + 16 * (quad & 1) + 8 * (quad >> 1));
}
__device__ __forceinline__ void arrange_rows(bf16x4 (&x)[4], const bf16x8 (&raw)[2]) {
#pragma unroll
    for (int p = 0; p < 2; p++) {
        const u32x4 v = __builtin_bit_cast(u32x4, raw[p]);
        const u32x2 lo = __builtin_amdgcn_permlane16_swap(v[0], v[2], false, false), hi = __builtin_amdgcn_permlane16_swap(v[1], v[3], false, false);
        x[2 * p] = __builtin_bit_cast(bf16x4, u32x2{lo[0], hi[0]});
        x[2 * p + 1] = __builtin_bit_cast(bf16x4, u32x2{lo[1], hi[1]});
    }
}
__device__ __forceinline__ void load_rows(bf16x4 (&x)[4], const bf16* row, int quad) {
    bf16x8 raw[2];
    request_rows(raw, row, quad);
    arrange_rows(x, raw);
}
__device__ __forceinline__ bool rows_wide(const void* p, int64_t sb, int64_t sh, int64_t sn) {
    return ((reinterpret_cast<uintptr_t>(p) & 15u) | ((sb | sh | sn) & 7)) == 0;
}

// Unsigned integers that sort like the floats; 0 is kept for empty slots (a NaN becomes 1, below every number).
__device__ __forceinline__ unsigned ordered_key(float f) {
    const unsigned b = __float_as_uint(f);
    const unsigned k = (b & 0x80000000u) ? ~b : (b | 0x80000000u);
    return (f != f || k == 0u) ? 1u : k;
}
// Score rounded to bf16 and key index in one integer: the larger is the better key, equal scores by smaller index, and no
// two keys of a row are equal.  For indices below 2^16 - 1 (a NaN sorts below every number, by index as well).
constexpr int kMaxPackedKeys = 65535;
__device__ __forceinline__ unsigned packed_key(float f, int idx) {
    return (ordered_key(rn_bf16(f)) & 0xFFFF0000u) | (unsigned)(0xFFFF - idx);
}

// Up to 64 KEYS keys ranked against one query by one wave: the products topk_dense_kernel makes, scores rounded to bf16, equal ones by index.  Every
// column of the score tiles is the query, so that lane l holds key 16 (l%16 / 4) + 4 (l/16) + l%4 of every 64 and counts the larger ones, handed
// round with readlane: 0.4 us for 64 keys, where bisection and the exchange of its counts take several.  keys: sixteen at a time in kTile elements, a lane's pieces
// at `first` and `second`; n (a multiple of 16) of them there are, the others rank last.
template <int KEYS>
struct RankedKeys {
    int rank[KEYS];
    __device__ __forceinline__ int index(int m, int lane) const { return m * 64 + 16 * ((lane & 15) >> 2) + 4 * (lane >> 4) + (lane & 3); }
};
template <int KEYS>
__device__ __forceinline__ RankedKeys<KEYS> rank_keys(const bf16* q_row, const bf16* keys, int first, int second, int n, int lane) {
    const int quad = lane >> 4, r = lane & 15;
    const bf16x8 q0 = ld16(q_row + quad * 8), q1 = ld16(q_row + quad * 8 + 32);
    bf16x8 k[KEYS][4][2];                                     // (all loads in flight together)
#pragma unroll
    for (int m = 0; m < KEYS; m++)
#pragma unroll
        for (int a = 0; a < 4; a++) {
            const bf16* p = keys + min(m * 4 + a, n / 16 - 1) * (16 * kD);
            k[m][a][0] = ld16(p + first);
            k[m][a][1] = ld16(p + second);
        }
    RankedKeys<KEYS> ranked;
    unsigned key[KEYS];
#pragma unroll
    for (int m = 0; m < KEYS; m++) {
        float own = 0.f;
#pragma unroll
        for (int a = 0; a < 4; a++) {
            f32x4 z = {0.f, 0.f, 0.f, 0.f};
            const f32x4 s = mfma_bf16(k[m][a][1], q1, mfma_bf16(k[m][a][0], q0, z));
#pragma unroll
            for (int e = 0; e < 4; e++) own = r == 4 * a + e ? s[e] : own;
        }
        const int idx = ranked.index(m, lane);
        key[m] = idx < n ? packed_key(own, idx) : 0u;
        ranked.rank[m] = 0;
    }
#pragma unroll
    for (int m = 0; m < KEYS; m++) {
#pragma unroll 8
        for (int j = 0; j < kWave; j++) {
            const unsigned o = (unsigned)__builtin_amdgcn_readlane((int)key[m], j);
#pragma unroll
            for (int i = 0; i < KEYS; i++) ranked.rank[i] += o > key[i] ? 1 : 0;
        }
    }
    return ranked;
}

// Operand tiles.  The attention kernels never read K/V/Q/dO row-major: a 16-row x 64-channel
// block (1024 bf16 = 2 KB) is stored twice, each time in exactly the order the 64 lanes of a
// wave consume it as an MFMA operand, so that every operand load is one fully coalesced
// instruction (lane l reads bytes [16 l, 16 l + 16) or [8 l, 8 l + 8) of a contiguous piece)
// instead of 64 scattered 16-byte accesses, which would saturate the L1's access rate.
//   R tile ("rows", contraction over channels):  element (row i, channel c) at
//        ((c >> 3) * 16 + i) * 8 + (c & 7)
//     lane l, step s (channels 32 s ..) loads 8 elements at  s * 512 + l * 8
//   T tile ("tokens", contraction over the 16 rows): element (row t, channel c) at
//        (((c >> 4) * 4 + (t >> 2)) * 16 + (c & 15)) * 4 + (t & 3)
//     lane l, channel tile dt (channels 16 dt ..) loads 4 elements at  dt * 256 + l * 4
constexpr int kTile = kBlk * kD;     // elements per block tile
__device__ __forceinline__ int r_tile_off(int i, int c) { return ((c >> 3) * 16 + i) * 8 + (c & 7); }
__device__ __forceinline__ int t_tile_off(int t, int c) { return (((c >> 4) * 4 + (t >> 2)) * 16 + (c & 15)) * 4 + (t & 3); }

// A T operand out of an R tile that sits in LDS, with the transposing LDS read of gfx950
// (ds_read_b64_tr_b16).  Within each group of 16 lanes, lane j supplies the address of four
// consecutive 16-bit elements and lane i receives element i%4 of the chunks supplied by lanes
// i/4, 4 + i/4, 8 + i/4, 12 + i/4.  Pointing lane j at (token 4*(l/16) + j/4, channels
// 16*dt + 4*(j%4) ..+3) therefore hands lane i tokens 4*(l/16)..+3 of channel 16*dt + i: the T
// operand.  So K/Q/dO are fetched from HBM once, as R tiles, and the second orientation is
// made on chip instead of being read from a second copy.
//
// In LDS such a tile is kept with the rows of every odd 8-channel chunk permuted (row ^ 12).  In the layout of memory the transposing
// read's groups of 16 lanes take 64 bytes of chunk 2 dt and 64 bytes of chunk 2 dt + 1, which lie 256 bytes further and so in the
// same banks, and every one of these reads takes two cycles more: a quarter to a third of all LDS cycles of the backward kernels.
// The permutation costs nothing: the lane that copies a 16-byte unit into LDS fetches another one of the same kilobyte
// (r_unit), and plain reads use the same lane-dependent offset.
typedef __attribute__((ext_vector_type(4))) short s16x4;
__device__ __forceinline__ int r_unit(int lane) { return (lane ^ ((lane >> 4) & 1) * 12) * 8; }    // element offset of a lane's unit in half a tile
__device__ __forceinline__ bf16x4 lds_t_operand(const bf16* r_tile_in_lds, int dt, int lane) {
    const int j = lane & 15, q = lane >> 4;
    const bf16* p = r_tile_in_lds + r_tile_off((4 * q + (j >> 2)) ^ ((j >> 1) & 1) * 12, 16 * dt + 4 * (j & 3));
    const s16x4 v = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)p);
    return __builtin_bit_cast(bf16x4, v);
}

// Asynchronous 16-byte-per-lane copy from global memory straight into LDS (no registers):
// lane l's 16 bytes land at lds_wave_base + 16*l, so a wave moves 1 KB that is contiguous in
// LDS.  lds_wave_base must be the same in every lane.  The copy is tracked by the vector-memory
// counter: wait_vm0() before the data (or a barrier that publishes it) is relied on.
// OFF: elements, added on both sides by the instruction itself, where a second pair of addresses costs registers and vector adds.
template <int OFF = 0>
__device__ __forceinline__ void copy16_global_to_lds(const bf16* g_lane, bf16* lds_wave_base) {
    __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)g_lane,
                                     (__attribute__((address_space(3))) void*)lds_wave_base, 16, OFF * (int)sizeof(bf16), 0);
}
__device__ __forceinline__ void wait_vm0() { __builtin_amdgcn_s_waitcnt(0x0F70); }   // vmcnt(0), other counters untouched
// A workgroup barrier of which waves may stand at different places in the code: the hardware's barrier counts arrivals, one per wave,
// whatever instruction they come from.  __syncthreads() is the same instructions, but promises this only where all waves meet at
// the same one.  Every wave must arrive equally often, and the branch between the places must be wave-uniform.
__device__ __forceinline__ void counted_barrier() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
}
// vmcnt(0) and lgkmcnt(0).  The compiler books a copy into LDS against both counters; until it has seen
// both drained it takes the vector-memory queue for out of order and turns every later wait into vmcnt(0).
__device__ __forceinline__ void wait_all_mem() { __builtin_amdgcn_s_waitcnt(0x0070); }

// ---------------------------------------------------------------------------------------
// rotation of one 8-channel chunk (4 interleaved pairs) with bf16 rounding after every
// multiply and add, the arithmetic the reference performs in the tensor dtype
// ---------------------------------------------------------------------------------------
//
// Contraction must stay off here: with it the compiler narrows the fp32 expression to bf16
// arithmetic and then fuses multiply and add into one bf16 FMA, i.e. one rounding fewer.
__device__ __forceinline__ bf16x8 rope_chunk_fwd(bf16x8 x, bf16x8 f) {
#pragma clang fp contract(off)
    bf16x8 y;
#pragma unroll
    for (int j = 0; j < 4; j++) {
        float s = (float)f[2 * j], c = (float)f[2 * j + 1];
        float xe = (float)x[2 * j], xo = (float)x[2 * j + 1];
        y[2 * j] = (bf16)(rn_bf16(c * xe) - rn_bf16(s * xo));
        y[2 * j + 1] = (bf16)(rn_bf16(s * xe) + rn_bf16(c * xo));
    }
    return y;
}

// Rotates a gradient back through the 2-D RoPE: 4 consecutive channels = two (even, odd) pairs, f
// holds their [sin, cos] entries.  Every product and sum is rounded to bf16 like the forward rotation.
__device__ __forceinline__ bf16x4 rope_bwd4(bf16x4 o, bf16x4 f) {
#pragma clang fp contract(off)
    bf16x4 y;
#pragma unroll
    for (int j = 0; j < 2; j++) {
        const float s = (float)f[2 * j], c = (float)f[2 * j + 1];
        const float ge = (float)o[2 * j], go = (float)o[2 * j + 1];
        y[2 * j] = (bf16)(rn_bf16(c * ge) + rn_bf16(s * go));
        y[2 * j + 1] = (bf16)(rn_bf16(-s * ge) + rn_bf16(c * go));
    }
    return y;
}

// ints at the end of a (b,h)'s work list (see transpose.hip) that the transpose of many entries uses as
// histogram, then as cursors
__host__ __device__ inline int work_tail_len(int Kb) { return (Kb + 3) & ~3; }
__host__ __device__ inline int fine_chunk(int N) { return N > 16384 ? 256 : 64; }      // llsa_fine_chunk
// llsa_fine_chunk_for.  Short pieces trade the length of the longest item, which is what a pass over few entries takes, for fp32
// partial sums (8 KB a piece) and their reduction, which is what it takes over many.  So the lines are drawn on the entries of
// all heads, up to 2048 tokens, where they were measured: K-side pass + reduction in us with pieces of 16 / 32 / 64, smooth
// inputs, N = 1024 unless given --
//     6 heads, topk 8    (3 Ki entries)    15 / 18 / 25          96 heads, topk 8  (48 Ki)     44 / 37 / 38
//     24 heads, topk 8   (12 Ki)           20 / 21 / 26          24 heads, topk 32 (48 Ki)     34 / 34 / 36
//     24 heads, topk 16  (24 Ki)           25 / 24 / 27          24 x 2048, topk 16 (48 Ki)    37 / 31 / 35
//     6 x 2048, topk 32  (24 Ki)           25 / 25 / 31          24 heads, topk 64 (96 Ki)     43 / 42 / 39
//     96 heads, topk 64  (384 Ki)         163 / 138 / 97         384 heads, topk 64           748 / 599 / 367
inline int fine_chunk_for(int64_t BH, int N, int T) {
    const int64_t entries = BH * (N / kBlk) * T;
    if (N > 2048 || entries > (1 << 16)) return fine_chunk(N);
    return entries > (1 << 14) ? 32 : 16;
}

constexpr int kGroup = 4;      // pooled blocks per LDS buffer in the query-side attention kernels (one per wave)

__device__ __forceinline__ int clampi(int v, int lo, int hi) { return v < lo ? lo : (v > hi ? hi : v); }

// The blocks of the pooled levels a group of query blocks reads, as the forward and the dQ kernel walk them:
// level 1's selected blocks, level 2's, ..., then every block of the coarsest level.  `Level` is llsa_fwd_level
// or llsa_bwd_level (fields sel, T).  Blocks of level l per (b,h): N / 16^(l+1).
// What a wave looks up per block stays in registers.  With a loop over the levels in the kernel's arguments every block waited for a chain of scalar loads,
// and with them for its LDS reads (they share a counter): 6 x 262144 tokens of two levels, forward 853 -> 811 us, dQ 996 -> 961; forward of 8 x 65536 of one
// level 651 -> 627, which is less than its cycles say (these kernels run at 1.9 to 2.1 GHz of 2.4).
struct SharedTiles { const bf16 *k, *v; };                    // tiles of a block
struct SharedList {
    int mine;                  // lane i: the i-th selected entry over all levels below the coarsest
    int n_first, n_listed;     // how many of those there are in level 1, in all
    int n_blocks;              // n_listed + blocks of the coarsest level
    int n0;                    // blocks of level 1 per (b,h)
    SharedTiles first, coarse; // tiles of block 0 of level 1 and of the coarsest
};
__host__ __device__ inline int64_t coarsest_multiple(int levels) {       // N must be a multiple of 64 * 16^levels
    int64_t m = 64;
    for (int l = 0; l < levels; l++) m *= 16;
    return m;
}
__device__ __forceinline__ const void* value_tiles(const llsa_fwd_level& l) { return l.vt; }
__device__ __forceinline__ const void* value_tiles(const llsa_bwd_level& l) { return l.vr; }
template <typename Level>
__device__ __forceinline__ SharedTiles level_tiles(const Level& l, int64_t block) {
    return {(const bf16*)l.kr + block * kTile, (const bf16*)value_tiles(l) + block * kTile};
}
template <typename Level>
__device__ __forceinline__ SharedList shared_list(const Level* lvl, int levels, int N, int bh, int g, int lane) {
    SharedList sl;
    sl.mine = 0;
    int base = 0, nb = N / (kBlk * kBlk);                     // blocks of level 1 per (b,h) = owners of its selection
    int owner = g / kBlk;
    sl.n0 = nb;
    sl.n_first = levels > 1 ? lvl[0].T : 0;
    sl.first = level_tiles(lvl[0], (int64_t)bh * nb);
    for (int l = 1; l < levels; l++) {
        const int T = lvl[l - 1].T;
        if (lane >= base && lane < base + T) sl.mine = lvl[l - 1].sel[((int64_t)bh * nb + owner) * T + (lane - base)];
        base += T;
        nb /= kBlk;
        owner /= kBlk;
    }
    sl.n_listed = base;
    sl.n_blocks = base + nb;                                  // nb is now the block count of the coarsest level
    sl.coarse = level_tiles(lvl[levels - 1], (int64_t)bh * nb);
    return sl;
}
// the i-th block of the walk (i is wave-uniform)
template <typename Level>
__device__ __forceinline__ SharedTiles shared_tiles(const SharedList& sl, const Level* lvl, int bh, int i) {
    if (i >= sl.n_listed) {
        const int64_t at = (int64_t)(i - sl.n_listed) * kTile;
        return {sl.coarse.k + at, sl.coarse.v + at};
    }
    const int entry = __builtin_amdgcn_readlane(sl.mine, i);  // (i < 64 here)
    if (i < sl.n_first) {
        const int64_t at = (int64_t)clampi(entry, 0, sl.n0 - 1) * kTile;
        return {sl.first.k + at, sl.first.v + at};
    }
    int base = sl.n_first, nb = sl.n0 / kBlk, l = 1;
    while (i >= base + lvl[l].T) {
        base += lvl[l++].T;
        nb /= kBlk;
    }
    return level_tiles(lvl[l], (int64_t)bh * nb + clampi(entry, 0, nb - 1));
}
// The weight of the walk's groups of kGroup blocks, which changes from level to level (every level's count is a multiple of kGroup)
struct SharedWeight {
    float w;
    int level, next;           // index into lvl[]; the group it ends in front of
};
template <typename Level>
__device__ __forceinline__ void next_weight(SharedWeight& sw, const Level* lvl, int levels) {
    sw.level++;
    sw.w = lvl[sw.level].w;
    sw.next = sw.level + 1 < levels ? sw.next + lvl[sw.level].T / kGroup : 0x7fffffff;
}
template <typename Level>
__device__ __forceinline__ SharedWeight first_weight(const Level* lvl, int levels) {
    SharedWeight sw{0.f, -1, 0};
    next_weight(sw, lvl, levels);
    return sw;
}

// The fine lists of Q sibling query blocks (ip: Q rows of T entries one after the other, Q * T <= 64 R), merged: the
// distinct blocks, each with the set of rows that name it (bit u: row u), ordered by that set.  A row that names a block twice
// keeps all lists as they are (every entry on its own).  Entry i of the result sits in lane i % 64 of register i / 64.
// `scratch`: 64 R ints of LDS private to the wave.
constexpr int kSetShift = 28;     // an entry is block | set << 28: a sequence of fewer than 2^31 tokens has fewer than 2^27 blocks
template <int Q, int R>
struct MergedLists {
    static_assert(Q <= 32 - kSetShift, "a set has one bit per row");
    int packed[R];
    int n;
    __device__ __forceinline__ int at(int i) const {          // i is wave-uniform
        const int v = __builtin_amdgcn_readlane(packed[0], i & (kWave - 1));
        if (R == 1) return v;
        const int o = __builtin_amdgcn_readlane(packed[R - 1], i & (kWave - 1));
        return i < kWave ? v : o;
    }
    __device__ __forceinline__ int block(int i) const { return at(i) & ((1 << kSetShift) - 1); }
    __device__ __forceinline__ unsigned rows(int i) const { return (unsigned)at(i) >> kSetShift; }
};
// The values of a row of sixteen lanes turned by TURN places
template <int TURN>
__device__ __forceinline__ unsigned row_turn(unsigned v) {
    if constexpr (TURN == 0) return v;
#ifndef LLSA_CPU_EMU_BUILD
    return (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0x120 + (TURN == 0 ? 1 : TURN), 0xf, 0xf, true);      // row_ror
#else
    const int lane = (int)(threadIdx.x & (kWave - 1));
    return __shfl(v, (lane & ~15) | ((lane - TURN) & 15));
#endif
}
// Whether one of the sixteen values that the lanes of this row have in `o` is v; FIRST = 1: of the fifteen other lanes
template <int FIRST, int... TURN>
__device__ __forceinline__ bool in_row(unsigned v, unsigned o, std::integer_sequence<int, TURN...>) {
    unsigned least = ~0u;
    ((least = TURN < FIRST ? least : min(least, v ^ row_turn<TURN>(o))), ...);
    return least == 0;
}
template <int FIRST>
__device__ __forceinline__ bool in_row(unsigned v, unsigned o) { return in_row<FIRST>(v, o, std::make_integer_sequence<int, 16>{}); }
// The value of lane l ^ 16, of lane l ^ 32
__device__ __forceinline__ unsigned lane_xor16(unsigned v, int lane) {
    const u32x2 s = __builtin_amdgcn_permlane16_swap(v, v, false, false);
    return (lane & 16) ? s[0] : s[1];
}
__device__ __forceinline__ unsigned lane_xor32(unsigned v, int lane) {
    const u32x2 s = __builtin_amdgcn_permlane32_swap(v, v, false, false);
    return (lane & 32) ? s[0] : s[1];
}
// Merged entries into their places: v, set, lead of every lane and register
template <int Q, int R>
__device__ __forceinline__ MergedLists<Q, R> place_merged(const int (&v)[R], const int (&set)[R], const bool (&lead)[R], int lane, int* scratch) {
    MergedLists<Q, R> ml;
    const unsigned long long below = (1ull << lane) - 1ull;
    int n = 0;
#pragma unroll 1
    for (int c = (1 << Q) - 1; c > 0; c--) {
#pragma unroll
        for (int k = 0; k < R; k++) {
            const unsigned long long m = __ballot(lead[k] && set[k] == c);
            if (lead[k] && set[k] == c) scratch[n + __popcll(m & below)] = v[k] | (int)((unsigned)c << kSetShift);
            n += __popcll(m);
        }
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
    for (int k = 0; k < R; k++) ml.packed[k] = scratch[k * kWave + lane];
    ml.n = n;
    return ml;
}
// Two lists of at most 32 entries, one in either half of the wave: an entry is compared with sixteen of the other list at a time, and with those of its own, by
// turning rows of sixteen lanes inside the comparisons: at most 126 instructions, where a loop over the entries (readlane, ballots) took 32 to 64 rounds of
// about fifteen in front of every wave.  With dQ's lists merged behind its first rows, training steps: 48 x 16384 tokens 1174 -> 1165.5 us, 24 x 16384 at topk
// 32/16 719 -> 706, 6 x 262144 3803 -> 3776, 12 x 16384 291.6 -> 289.3, 24 x 4096 even (in front of them 1 % longer there).
__device__ __forceinline__ MergedLists<2, 1> merge_two(const int* ip, int T, int N1, int lane, int* scratch) {
    const int row = lane >> 5, i = lane & 31;
    const int v[1] = {i < T ? clampi(ip[row * T + i], 0, N1 - 1) : -1 - lane};      // (distinct negative fillers)
    const unsigned own = (unsigned)v[0], other = lane_xor32(own, lane);
    bool both = in_row<0>(own, other), again = in_row<1>(own, own);
    if (T > 16) {
        both |= in_row<0>(own, lane_xor16(other, lane));
        again |= in_row<0>(own, lane_xor16(own, lane));
    }
    const bool twice = __ballot(again) != 0;
    const int set[1] = {both && !twice ? 3 : 1 << row};
    const bool lead[1] = {i < T && (row == 0 || set[0] == 2)};
    return place_merged<2, 1>(v, set, lead, lane, scratch);
}
template <int Q, int R>
__device__ __forceinline__ MergedLists<Q, R> merge_lists(const int* ip, int T, int N1, int lane, int* scratch) {
    if constexpr (Q == 2 && R == 1) return merge_two(ip, T, N1, lane, scratch);
    static_assert(R <= 2, "entries sit in one or two registers");
    MergedLists<Q, R> ml;
    int v[R], row[R];
#pragma unroll
    for (int k = 0; k < R; k++) {
        const int i = k * kWave + lane;
        v[k] = i < Q * T ? clampi(ip[i], 0, N1 - 1) : -1 - i;         // (distinct negative fillers)
        row[k] = 0;
#pragma unroll
        for (int u = 1; u < Q; u++) row[k] += i >= u * T ? 1 : 0;
    }
    if constexpr (Q == 1) {
#pragma unroll
        for (int k = 0; k < R; k++) ml.packed[k] = v[k] | (1 << kSetShift);
        ml.n = T;
        return ml;
    }
    unsigned long long in[Q][R], twice = 0;                   // which lanes' blocks row u names
#pragma unroll
    for (int u = 0; u < Q; u++)
#pragma unroll
        for (int k = 0; k < R; k++) in[u][k] = 0;
#pragma unroll
    for (int u = 0; u < Q; u++)
#pragma unroll 1
        for (int s = 0; s < T; s++) {
            const int j = u * T + s;
            int o = __builtin_amdgcn_readlane(v[0], j & (kWave - 1));
            if (R > 1) {
                const int o1 = __builtin_amdgcn_readlane(v[R - 1], j & (kWave - 1));
                o = j < kWave ? o : o1;
            }
#pragma unroll
            for (int k = 0; k < R; k++) {
                const unsigned long long eq = __ballot(v[k] == o);
                twice |= in[u][k] & eq & __ballot(row[k] == u);       // named by this row before
                in[u][k] |= eq;
            }
        }
    int set[R];
    bool lead[R];
#pragma unroll
    for (int k = 0; k < R; k++) {
        set[k] = 0;
#pragma unroll
        for (int u = 0; u < Q; u++) set[k] |= ((in[u][k] >> lane) & 1ull) ? 1 << u : 0;
        if (twice != 0) set[k] = 1 << row[k];
        lead[k] = k * kWave + lane < Q * T && (set[k] & ((1 << row[k]) - 1)) == 0;
    }
    return place_merged<Q, R>(v, set, lead, lane, scratch);
}
// Two query blocks per wave are possible up to this topk (their lists then fit two registers) ...
constexpr int kPairMaxTopk = 64;
// ... and considered where their workgroups (four waves, a group of eight query blocks) fill the chip.  It holds three of them per CU
// (single query blocks: four of half the work), so a last round that is mostly empty costs a whole one: at most 30 % more places than
// groups.  And below 5/6 of a round the chip has room for all of the waves either way, and a wave of one block has half the
// serial chain.  dQ, one / two, us (topk 16 but for 7168 tokens, where it is 12):
//   groups 384 (6 x 8192) 24.6 / 28.1;  512 (16 x 4096) 23.0 / 23.8;  640 (20 x 4096) 29.0 / 29.1
//   728 (13 x 7168) 34.3 / 33.4;  768 (24 x 4096) 32.2 / 30.5;  784 (14 x 7168) 37.7 / 40.4;  840 (15 x 7168) 38.6 / 41.3
//   1280 (20 x 8192) 62.0 / 57.6;  1536 (24 x 8192) 75.6 / 68.2;  two levels 1536 (12 x 16384) 68.1 / 60.8;  2048 87.3 / 80.5;  3072 140.0 / 120.5
// (The 30 % could be more since two lists are merged in a hundred instructions: 1152 (16 x 9216) 60.6 / 59.0, the step 256.5 / 254.4;  1568 (28 x
// 7168) 68.4 / 65.4, 278.3 / 273.8;  1024 (8 x 16384, two levels) 42.9 / 42.3.)
// The forward's waves are shorter.  In one round of pairs, where the single blocks no longer fit the chip at once, it is two from 513 groups on, which pays
// from about 700: sampling, the whole pass, topk 8:  512 (8 x 8192) 38.2 / 39.4;  576 43.3 / 44.6;  640 44.5 / 45.5;  544 (17 x 4096) 35.4 / 35.8;  640 36.7 /
// 37.2;  768 (24 x 4096, topk 16) 46.1 / 45.2;  beyond a round one:  832 (13 x 8192) 53.0 / 55.9;  960 58.8 / 59.1;  1152 62.1 / 64.6;  1280 67.4 / 67.0
// Where most of the walk is pooled blocks, which a wave of two reads once for both, two win from 512 groups on and with as much as 60 % more
// places than groups.  Sampling, and in brackets the training step with one / two in dQ, topk 8 unless given:
//   512 (2 x 32768, 128 pooled blocks) 73.0 / 71.5 (237.5 / 232.0);  512 (65536, 256) 118.5 / 114.0 (396.9 / 386.4), at topk 16 123.5 / 119.3 (421.0 / 412.9)
//   640 (2 x 40960, 160) 103.0 / 103.4 (328.2 / 321.7);  960 (5 x 24576, 96) 101.7 / 98.2 (325.6 / 316.6);  1024 (2 x 65536) 207.7 / 192.5 (674.5 / 648.9)
//   1024 (8 x 16384, 64) 84.4 / 82.7 (256.2 / 250.4);  1664 (13 x 16384) 123.8 / 121.5 (406.4 / 393.1);  but 512 (4 x 16384) 51.2 / 52.1 (159.7 / 157.5)
//   and 800 (5 x 20480, 80) 80.9 / 84.6 (251.2 / 253.4);  896 (4 x 28672, 112) 104.7 / 106.5 (332.7 / 331.4)
// With a larger topk from a full round on: 1024 (8 x 16384, topk 16) 91.9 / 90.4 (284.0 / 278.6);  960 (5 x 24576, topk 24) 121.3 / 118.2 (390.6 / 382.6)
//   1024 (2 x 65536, topk 64) 280.5 / 276.0 (943.2 / 930.8);  but 512 (4 x 16384, topk 16) 55.5 / 56.3 (174.2 / 173.9);  512 (65536, topk 64) 161.5 / 166.7
constexpr int kPairPlaces = 256 * 3;
inline bool pairs_pay(int64_t groups, int64_t pooled_blocks, int T, bool forward) {
    const int64_t places = (groups + kPairPlaces - 1) / kPairPlaces * kPairPlaces, idle = (places - groups) * 10;
    if (pooled_blocks >= 64 && pooled_blocks >= 4 * T && groups >= (pooled_blocks >= 8 * T ? 512 : kPairPlaces) && idle <= groups * 6) return true;
    if (forward && groups <= kPairPlaces) return groups > 512;
    return groups > 640 && idle <= groups * 3;
}
// Blocks of the pooled levels every query block reads, all levels (topk: of every level, finest first)
inline int64_t pooled_blocks_read(int N, const int32_t* topk, int levels) {
    int64_t blocks = N / 256;
    for (int l = 1; l < levels; l++) blocks /= 16;
    for (int l = 1; l < levels; l++) blocks += topk[l];
    return blocks;
}
// Whether a wave of the forward / dQ kernel takes two query blocks
inline bool two_blocks_per_wave(int64_t BH, int N, const int32_t* topk, int levels, bool forward) {
    const int64_t groups = (int64_t)N / 128 * BH, pooled = pooled_blocks_read(N, topk, levels);
    if (topk[0] > kPairMaxTopk || N % 128 != 0 || !pairs_pay(groups, pooled, topk[0], forward)) return false;
    // Where the fine blocks are most of the walk the forward gains little from two on grids of a few rounds.  Sampling, the whole pass, topk 8, 16 pooled blocks: 28 x
    // 4096 tokens 45.7 / 47.7, 32 x 4096 49.0 / 49.7, 36 x 4096 49.5 / 51.6, 40 x 4096 53.0 / 53.6, 64 x 4096 (2048 groups) 77.2 / 76.8;  two levels 8/8 8 x 16384 50.7 /
    // 51.4;  16/16 12 x 16384 83.1 / 81.4, 16 x 16384 (2048) 104.9 / 101.9, 24 x 16384 149.2 / 142.8.  (At 32/16, where a fine block is named by both rows more often,
    // two would pay from a full round on: 12 x 16384 109.6 / 103.1, its training step 361.8 / 356.9.)
    return !forward || pooled >= 4 * topk[0] || groups >= 2048;
}

// 16- and 8-byte reads that are LDS reads by construction (ds_read_b128 / ds_read_b64)
__device__ __forceinline__ bf16x8 lds_ld16(const bf16* p) {
    return *reinterpret_cast<const __attribute__((address_space(3))) bf16x8*>((const __attribute__((address_space(3))) bf16*)p);
}
__device__ __forceinline__ bf16x4 lds_ld8(const bf16* p) {
    return *reinterpret_cast<const __attribute__((address_space(3))) bf16x4*>((const __attribute__((address_space(3))) bf16*)p);
}
__device__ __forceinline__ void lds_st16(bf16* p, bf16x8 v) {
    *reinterpret_cast<__attribute__((address_space(3))) bf16x8*>((__attribute__((address_space(3))) bf16*)p) = v;
}
__device__ __forceinline__ void lds_st8(bf16* p, bf16x4 v) {
    *reinterpret_cast<__attribute__((address_space(3))) bf16x4*>((__attribute__((address_space(3))) bf16*)p) = v;
}

// Sixteen rows that arrived eight whole rows a load (rows[i]: row 8 i + l/8, channels 8 (l%8) ..+7) as R operand: lane l gets channels
// 8 (l/16) ..+7 of row l%16 and those 32 further on.  place: 2 KB of LDS of the wave.  (In the operand layout straight from memory each of
// a load's 64 pieces is an access of its own in the L1.  A row's eight pieces are in an order of its own: rows start in the same banks.)
__device__ __forceinline__ void rows_to_operand(bf16x8 (&x)[2], const bf16x8 (&rows)[2], bf16* place, int lane) {
    const int r = lane & 15, quad = lane >> 4;
#pragma unroll
    for (int i = 0; i < 2; i++) {
        const int row = 8 * i + (lane >> 3);
        lds_st16(place + row * kD + ((lane & 7) ^ (row & 7)) * 8, rows[i]);
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int i = 0; i < 2; i++) x[i] = lds_ld16(place + r * kD + ((quad + 4 * i) ^ (r & 7)) * 8);
}

// A block's sixteen token rows in LDS as they are in memory, copied eight whole rows at a time, and T operands out of them.  A row's pieces
// change places in pairs (piece ^ (row & 6)): the transposing read's lanes 0..31 and 32..63 take 32 bytes of each of eight rows of 128, whose
// banks are those of every second row.
__device__ __forceinline__ int row_piece(int lane) { return ((lane & 7) ^ ((lane >> 3) & 6)) * 8; }     // the piece of row l/8 (or 8 + l/8) that lane l copies
__device__ __forceinline__ bf16x4 lds_t_operand_rows(const bf16* rows_in_lds, int dt, int lane) {
    const int j = lane & 15, row = 4 * (lane >> 4) + (j >> 2);
    const bf16* p = rows_in_lds + row * kD + ((2 * dt + ((j >> 1) & 1)) ^ (row & 6)) * 8 + 4 * (j & 1);
    const s16x4 v = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)p);
    return __builtin_bit_cast(bf16x4, v);
}

// XCD-aware workgroup order.  The 8 XCDs of the chip each have a private L2 and receive
// workgroups round-robin by linear id (id % 8).  Neighbouring logical work items (query or
// key blocks that are close in Z-order) read overlapping K/V/Q rows, so they should share an
// L2: this maps the hardware id to a logical id such that every XCD walks one contiguous
// range of the (x, y) grid.  Returns the logical linear id in [0, gridDim.x * gridDim.y).
constexpr int kXcds = 8;
// `rows_before`: rows of the grid in front that do other work (their number times gridDim.x is a multiple of 8).
__device__ __forceinline__ int xcd_logical_id(int rows_before = 0) {
    const int total = gridDim.x * (gridDim.y - rows_before);
    const int lin = (blockIdx.y - rows_before) * gridDim.x + blockIdx.x;
    const int xcd = lin % kXcds, slot = lin / kXcds;
    const int q = total / kXcds, rem = total % kXcds;
    return xcd * q + (xcd < rem ? xcd : rem) + slot;
}

}  // namespace llsa
