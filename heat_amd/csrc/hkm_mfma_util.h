// Device helpers shared by the matrix-core kernels (fp32 and split-fp16 products).
#pragma once
#include "hkm_common.h"

namespace hkm {

typedef _Float16 halfx2 __attribute__((ext_vector_type(2)));
typedef float floatx2 __attribute__((ext_vector_type(2)));
typedef _Float16 halfx8 __attribute__((ext_vector_type(8)));
#define MFMA_F16(a, b, c) __builtin_amdgcn_mfma_f32_32x32x16_f16((a), (b), (c), 0, 0, 0)
#define MFMA32(a, b, c) __builtin_amdgcn_mfma_f32_32x32x2f32((a), (b), (c), 0, 0, 0)

__device__ __forceinline__ floatx4 ld4(const float* p) {
    return *reinterpret_cast<const floatx4*>(p);
}

// 16 bytes of row `p` starting at column c; columns >= D read as zero.  VEC: p + c is 16-B aligned
// and D % 4 == 0, so a group is either fully inside or fully outside the row.
template <bool VEC>
__device__ __forceinline__ floatx4 load_row4(const float* row, int c, int D) {
    floatx4 v = {0.f, 0.f, 0.f, 0.f};
    if (VEC) {
        if (c < D) v = ld4(row + c);
    } else {
#pragma unroll
        for (int t = 0; t < 4; ++t)
            if (c + t < D) v[t] = row[c + t];
    }
    return v;
}

// 16 bytes at any 4-byte boundary (global loads of this width need no more)
struct __attribute__((packed, aligned(4))) float4_any { float v[4]; };
__device__ __forceinline__ floatx4 ld4_any(const void* p) {
    return __builtin_bit_cast(floatx4, *static_cast<const float4_any*>(p));
}

// The rows of one tile for a wave: PB blocks of 32 rows starting at row0 (wave-uniform), a lane takes the DP/2 columns
// of its half of row p of each block; columns from D on read as zero.  Tiles that end before the last row (`fast`, lane
// offsets in 32 bits) are fetched with 16-byte loads whatever the rows' width and alignment: what a load reads
// beyond its row are elements of the next one (DP < 2 D), and a select drops them -- the guarded 4-byte loads that
// rows of no whole 16-byte groups took before cost a load instruction per element.  FULL: D == DP.
template <int DP, int PB, bool FULL>
__device__ __forceinline__ void fetch_rows_any(const float* __restrict__ X, int64_t N, int D, int64_t ldx, int64_t row0,
                                               int p, int h, bool fast, unsigned lane_off,
                                               floatx4 (&dst)[PB][DP / 8]) {
    constexpr int NJ = DP / 8;
    constexpr int DMIN = DP == 32 ? 17 : DP == 48 ? 33 : DP == 64 ? 49 : DP == 96 ? 65 : 97;  // least D padded to DP
    if (fast && row0 + PB * 32 + (FULL ? 0 : 1) <= N) {
#pragma unroll
        for (int pb = 0; pb < PB; ++pb) {
            const char* base = reinterpret_cast<const char*>(X + (row0 + pb * 32) * ldx);
#pragma unroll
            for (int j = 0; j < NJ; ++j) {
                floatx4 v = ld4_any(base + lane_off + 16 * j);
                if (!FULL && DP / 2 + 4 * j + 4 > DMIN) {
#pragma unroll
                    for (int t = 0; t < 4; ++t) v[t] = h * (DP / 2) + 4 * j + t < D ? v[t] : 0.f;
                }
                dst[pb][j] = v;
            }
        }
    } else {
#pragma unroll
        for (int pb = 0; pb < PB; ++pb) {
            int64_t r = row0 + pb * 32 + p;
            r = r < N ? r : N - 1;
            const float* xr = X + r * ldx;
#pragma unroll
            for (int j = 0; j < NJ; ++j) dst[pb][j] = load_row4<false>(xr, h * (DP / 2) + 4 * j, D);
        }
    }
}

__device__ __forceinline__ void merge_halves(float& m, int& mi) {
    const float om = __shfl_xor(m, 32);
    const int oi = __shfl_xor(mi, 32);
    if (om < m || (om == m && oi < mi)) {
        m = om;
        mi = oi;
    }
}

// the squared norms of the 16 centroid rows a lane owns in a block (cn16 points at the norm of row
// 4*h of the block; rows 8g + 4h .. 8g + 4h + 3 belong to accumulator elements 4g .. 4g + 3)
__device__ __forceinline__ floatx16 load_cn16(const float* cn16) {
    floatx16 c0;
#pragma unroll
    for (int g = 0; g < 4; ++g) {
        const floatx4 t = ld4(cn16 + 8 * g);
#pragma unroll
        for (int q = 0; q < 4; ++q) c0[4 * g + q] = t[q];
    }
    return c0;
}

// Minimum and first argmin over the 16 distances a lane holds of one centroid block, merged into the
// running (m, mi).  The minimum is a tree of three-input minima (9 instructions, no dependence on
// compare results); only lanes whose block minimum improves the running one look for its position,
// by equality from the last register down so that the first one wins.  Strict '<' keeps the earlier
// block on ties.  NaNs never win.
//
// Both halves are written out as instructions: the compiler's own form of the tree spends more
// instructions on canonicalising operands that are matrix-core results, and it places every compare of
// the lookup directly in front of the select that consumes it, which on this chip costs two idle cycles
// per pair (a vector instruction must not read a scalar register pair written by the instruction before
// it).  Here the compares run two ahead of the selects through three scalar register pairs, so no pair
// is read within two instructions of being written and nothing idles.
__device__ __forceinline__ float block_min16(const floatx16& d) {
    // The first read of the block is left to the compiler (a canonicalisation: one instruction that
    // returns its operand): it knows how many idle cycles a read of fresh matrix-core results needs,
    // which an instruction sequence it cannot see into would not get.
    const float t0 = __builtin_canonicalizef(d[0]);
    float a, b, c, e;
    asm("v_min3_f32 %[a], %[t0], %[d1], %[d2]\n\t"
        "v_min3_f32 %[b], %[d3], %[d4], %[d5]\n\t"
        "v_min3_f32 %[c], %[d6], %[d7], %[d8]\n\t"
        "v_min3_f32 %[e], %[d9], %[d10], %[d11]\n\t"
        "v_min3_f32 %[a], %[a], %[b], %[c]\n\t"
        "v_min3_f32 %[b], %[d12], %[d13], %[d14]\n\t"
        "v_min3_f32 %[a], %[a], %[e], %[b]\n\t"
        "v_min_f32 %[a], %[a], %[d15]"
        : [a] "=&v"(a), [b] "=&v"(b), [c] "=&v"(c), [e] "=&v"(e)
        : [t0] "v"(t0), [d1] "v"(d[1]), [d2] "v"(d[2]), [d3] "v"(d[3]), [d4] "v"(d[4]), [d5] "v"(d[5]), [d6] "v"(d[6]),
          [d7] "v"(d[7]), [d8] "v"(d[8]), [d9] "v"(d[9]), [d10] "v"(d[10]), [d11] "v"(d[11]), [d12] "v"(d[12]),
          [d13] "v"(d[13]), [d14] "v"(d[14]), [d15] "v"(d[15]));
    return a;
}

// position (8 * (v / 4) + v % 4 for register v: the centroid row inside the block, without the
// lane-half term) of the first of the 16 distances that equals bm
__device__ __forceinline__ int block_pos16(const floatx16& d, float bm) {
    int bi;
    unsigned long long s0, s1, s2;
    asm("v_cmp_eq_f32_e64 %[s0], %[d14], %[bm]\n\t"
        "v_cmp_eq_f32_e64 %[s1], %[d13], %[bm]\n\t"
        "v_cmp_eq_f32_e64 %[s2], %[d12], %[bm]\n\t"
        "v_cndmask_b32_e64 %[bi], 27, 26, %[s0]\n\t"
        "v_cmp_eq_f32_e64 %[s0], %[d11], %[bm]\n\t"
        "v_cndmask_b32_e64 %[bi], %[bi], 25, %[s1]\n\t"
        "v_cmp_eq_f32_e64 %[s1], %[d10], %[bm]\n\t"
        "v_cndmask_b32_e64 %[bi], %[bi], 24, %[s2]\n\t"
        "v_cmp_eq_f32_e64 %[s2], %[d9], %[bm]\n\t"
        "v_cndmask_b32_e64 %[bi], %[bi], 19, %[s0]\n\t"
        "v_cmp_eq_f32_e64 %[s0], %[d8], %[bm]\n\t"
        "v_cndmask_b32_e64 %[bi], %[bi], 18, %[s1]\n\t"
        "v_cmp_eq_f32_e64 %[s1], %[d7], %[bm]\n\t"
        "v_cndmask_b32_e64 %[bi], %[bi], 17, %[s2]\n\t"
        "v_cmp_eq_f32_e64 %[s2], %[d6], %[bm]\n\t"
        "v_cndmask_b32_e64 %[bi], %[bi], 16, %[s0]\n\t"
        "v_cmp_eq_f32_e64 %[s0], %[d5], %[bm]\n\t"
        "v_cndmask_b32_e64 %[bi], %[bi], 11, %[s1]\n\t"
        "v_cmp_eq_f32_e64 %[s1], %[d4], %[bm]\n\t"
        "v_cndmask_b32_e64 %[bi], %[bi], 10, %[s2]\n\t"
        "v_cmp_eq_f32_e64 %[s2], %[d3], %[bm]\n\t"
        "v_cndmask_b32_e64 %[bi], %[bi], 9, %[s0]\n\t"
        "v_cmp_eq_f32_e64 %[s0], %[d2], %[bm]\n\t"
        "v_cndmask_b32_e64 %[bi], %[bi], 8, %[s1]\n\t"
        "v_cmp_eq_f32_e64 %[s1], %[d1], %[bm]\n\t"
        "v_cndmask_b32_e64 %[bi], %[bi], 3, %[s2]\n\t"
        "v_cmp_eq_f32_e64 %[s2], %[d0], %[bm]\n\t"
        "v_cndmask_b32_e64 %[bi], %[bi], 2, %[s0]\n\t"
        "v_cndmask_b32_e64 %[bi], %[bi], 1, %[s1]\n\t"
        "v_cndmask_b32_e64 %[bi], %[bi], 0, %[s2]"
        : [bi] "=&v"(bi), [s0] "=&s"(s0), [s1] "=&s"(s1), [s2] "=&s"(s2)
        : [d0] "v"(d[0]), [d1] "v"(d[1]), [d2] "v"(d[2]), [d3] "v"(d[3]), [d4] "v"(d[4]), [d5] "v"(d[5]),
          [d6] "v"(d[6]), [d7] "v"(d[7]), [d8] "v"(d[8]), [d9] "v"(d[9]), [d10] "v"(d[10]), [d11] "v"(d[11]),
          [d12] "v"(d[12]), [d13] "v"(d[13]), [d14] "v"(d[14]), [bm] "v"(bm));
    return bi;
}

__device__ __forceinline__ void block_argmin(const floatx16& d, int kb, float& m, int& mi) {
    const float bm = block_min16(d);
    if (bm < m) {
        mi = kb + block_pos16(d, bm);
        m = bm;
    }
}

// The same running argmin with the lookup deferred: a block whose minimum improves the running one is
// only remembered -- its number and a copy of its 16 distances (eight 64-bit moves) -- and the position
// is looked up once, after the last block, in the copy that survived (kept_argmin).  Same result as
// block_argmin bit for bit: strict '<' keeps the earliest block that reaches the final minimum, the
// lookup its first position.  15 instead of 33 vector instructions per improving block.
__device__ __forceinline__ void block_min_keep(const floatx16& d, int cb, float& m, int& blk, floatx16& keep) {
    const float bm = block_min16(d);
    if (bm < m) {
        // written out so that the two values are updated where they live (the compiler's own form pairs the
        // minima of two point blocks into 64-bit moves and shuffles them into place first)
        asm("v_mov_b32 %0, %2\n\tv_mov_b32 %1, %3" : "+v"(m), "+v"(blk) : "v"(bm), "s"(cb));
        keep = d;
    }
}

// The copy starts out without a value: it is only read after a block improved on +inf (kept_argmin
// ignores it otherwise).  Declaring it written by an empty instruction sequence costs nothing, where
// sixteen zeros would cost sixteen moves per point block.
__device__ __forceinline__ void keep_undefined(floatx16& keep) { asm volatile("" : "=v"(keep)); }

// index (without the lane-half term) of the minimum that block_min_keep tracked; 0 if no block ever
// improved on +inf (all distances +inf or NaN), as block_argmin leaves it
__device__ __forceinline__ int kept_argmin(const floatx16& keep, float m, int blk) {
    const int pos = block_pos16(keep, m);
    return m < HKM_INF ? blk * 32 + pos : 0;
}

}  // namespace hkm
