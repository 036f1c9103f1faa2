// Resident distance + argmin and the one-sweep Lloyd step for rows of 17 to 64 features, with the cross term
// x.c on the fp16 matrix cores from fp32 operands split into two fp16 parts.
//
// What bounds it: the fp32 matrix instruction retires 2 features of a 32 x 32 tile in 64 cycles and shares its
// issue slots with the vector ALU; v_mfma_f32_32x32x16_f16 retires 16 in 32 cycles and runs beside it.  A value v
// is written as v1 + v2 with v1 = fp16(s v), v2 = fp16(s v - v1) for a power of two s: 11 + 11 significand bits
// and a sign, so v1 + v2 misses s v by at most 2^-22 of it (a quarter of all values: by one fp32 ulp, the rest:
// by nothing).  x.c is the sum of the three products x1 c2 + x2 c1 + x1 c1 -- each product of two fp16 values is
// exact in fp32, the matrix core adds in fp32 -- and x2 c2 (below 2^-22 |x c| per feature) is dropped: 3/16 of the
// fp32 path's matrix time.
//
// Precision: an fp32 product chain rounds once per feature, this one three times per 16 features, and the norms,
// which each in one chain were the largest error of a distance, are summed in fp64 (centroids, from their split
// values: what splitting a centroid changes then largely cancels for the rows near it) and in eight chains (rows).
// Measured rms error of min |x - c|^2 against float64 in units of 2^-24 (|x|^2 + |c|^2), fp32 kernel -> this one:
// blobs 0.89 -> 0.72 (20 features), 1.11 -> 0.74 (32), 1.41 -> 0.78 (50), 1.50 -> 0.86 (64); normal rows 0.80 -> 0.74,
// 0.89 -> 0.70, 1.07 -> 0.72, 1.10 -> 0.72; rows that miss the nearest of 256 centroids far from the origin (tied
// to rounding): 678 -> 450 of 100 000.
//
// Time per one-sweep step, fp32 kernel -> this one (with the finishing launches; before rows tied to rounding went to
// split_near_row, which adds 8 to 14 %): 4M x 32, K = 256: 612 -> 294 us;
// x 32, 64: 245 -> 181; x 24, 100: 281 -> 208; x 17, 40: 216 -> 158; 2M x 48, 128: 293 -> 184; x 50, 100: 364 -> 202.
// Assignment alone: 585 -> 230, 177 -> 126, 236 -> 140, 176 -> 113, 234 -> 119, 331 -> 196; 2M x 64, 200: 486 -> 235.
//
// Scaling.  fp16 holds 2^-24 .. 2^15.99, so the operands are scaled by powers of two (exact):
//   * shared: S takes the largest |centroid coordinate| into [2^7, 2^8).  A row whose root mean square is at least
//     1 / S and whose norm is at most 2^14 / S (its parts then hold at least fp32's precision in units of
//     |x|^2 + |c|^2) is scaled by S too: the accumulators start at S^2 |c|^2 (the C operand of the first matrix
//     instruction) and end as S^2 (|c|^2 - 2 x.c), no vector instruction per distance;
//   * any other row is scaled by its own power of two and takes one multiply and one fused multiply-add per distance.
//     That second scan runs for a wave's rows only if one of them needs it, and only that row takes its result, so a
//     row's result does not depend on its neighbours;
//   * centroids whose root mean squares span more than 2^6 below the largest coordinate (or are not finite) are each
//     scaled by a power of two of their own, and every row takes the second scan;
//   * rows whose |x|^2 is inf or NaN take an fp32 scan on the vector ALU.
//
// Everything else is the fp32 resident kernel (hkm_assign_mfma.hip): A = centroids, B = points, a lane owns one
// point and 16 centroid rows of a block; |x|^2 joins the minimum only; lazy clamp at 0; first index wins; the
// fused variant adds the rows, rounded to 28 bits below their exponent, to fp64 accumulators in LDS.
#include <type_traits>

#include "hkm_common.h"
#include "hkm_mfma_util.h"

namespace hkm {

static constexpr int SPLIT_QBITS = 28;

// 16-byte groups of a centroid row are permuted by the low bits of the row index so that the operand reads of
// consecutive rows fall on different banks without padding (the planes then fit wherever the fp32 rows did)
template <int DP>
__device__ __forceinline__ int split_swz(int r) {
    return DP == 32 ? (r >> 2) & 3 : DP == 64 ? (r >> 1) & 7 : 0;
}

// The centroids in LDS: per block of 32 rows first the high, then the low parts, [cb][2][32][DP]; a lane of row p of
// its half h reads 16 bytes per k-step at split_off.
template <int DP>
__device__ __forceinline__ int split_off(int p, int h, int st) {
    return p * DP + 8 * ((h * (DP / 16) + st) ^ split_swz<DP>(p));
}
__device__ __forceinline__ halfx8 ld_half8(const _Float16* p) { return *reinterpret_cast<const halfx8*>(p); }

// Scan of all centroid blocks for the wave's PB point blocks (operand parts xh, xl) that carry their own scales:
// rx = (scale of the results) / (scale of the row), sI holds the same for the centroids.  CLAMP: the full distance
// clamped at 0, as the reference orders it.  m: S^2 (|c|^2 - 2 x.c) resp. with CLAMP the distance.  (Rare rows: kept
// simple, see split_scan for the usual ones.)
template <int DP, int PB, bool CLAMP>
__device__ __forceinline__ void split_scan_own(const _Float16* planes, const float* sCn, const float* sI, int ncb,
                                               int cb0, int p, int h, const halfx8 (&xh)[PB][DP / 16], const halfx8 (&xl)[PB][DP / 16],
                                               const float (&rx)[PB], float inv_s2, const float (&xn)[PB],
                                               float (&m)[PB], int (&blk)[PB], floatx16 (&keep)[PB]) {
    constexpr int NS = DP / 16;
#pragma unroll 1
    for (int cb = 0; cb < ncb; ++cb) {
        const floatx16 c0 = load_cn16(sCn + cb * 32 + 4 * h);
        const floatx16 ci = load_cn16(sI + cb * 32 + 4 * h);
        floatx16 acc[PB];
#pragma unroll
        for (int pb = 0; pb < PB; ++pb)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[pb][v] = 0.f;
#pragma unroll
        for (int st = 0; st < NS; ++st) {
            const _Float16* c = planes + cb * (64 * DP) + split_off<DP>(p, h, st);
            const halfx8 ch = ld_half8(c), cl = ld_half8(c + 32 * DP);
#pragma unroll
            for (int pb = 0; pb < PB; ++pb) {
                acc[pb] = MFMA_F16(cl, xh[pb][st], acc[pb]);
                acc[pb] = MFMA_F16(ch, xl[pb][st], acc[pb]);
                acc[pb] = MFMA_F16(ch, xh[pb][st], acc[pb]);
            }
        }
#pragma unroll
        for (int pb = 0; pb < PB; ++pb) {
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                float d = fmaf(acc[pb][v] * ci[v], rx[pb], c0[v]);
                if (CLAMP) d = fmaxf(fmaf(d, inv_s2, xn[pb]), 0.0f);
                acc[pb][v] = d;
            }
            block_min_keep(acc[pb], cb0 + cb, m[pb], blk[pb], keep[pb]);
        }
    }
}

// The running minimum of a lane, the block it was found in and a copy of that block's 16 distances (block_min_keep's
// state, the copy as eight register pairs).
struct SplitBest {
    float m;
    float m2;  // the smallest minimum of another block
    int blk;
    floatx2 keep[8];
};
__device__ __forceinline__ void split_best_init(SplitBest& b) {
    b.m = HKM_INF;
    b.m2 = HKM_INF;
    b.blk = 0;
#pragma unroll
    for (int i = 0; i < 8; ++i) asm volatile("" : "=v"(b.keep[i]));  // written before it is read: see keep_undefined
}
// block_min_keep in three pieces without a branch the compiler knows of, to be placed between matrix instructions:
// the lanes whose minimum improved copy under an execution mask (12 vector instructions, where selects take 19;
// matrix instructions ignore the mask).  All pieces depend on the minimum, whose first read of the results the
// compiler guards (block_min16).
struct SplitScan {
    float bm;
    unsigned long long lt;
};
template <int PIECE>
__device__ __forceinline__ void split_scan_piece(SplitScan& s, const floatx16& d, int cb, SplitBest& b) {
    unsigned long long save;
    if (PIECE == 0) s.bm = block_min16(d);
    if (PIECE == 1)
        asm("v_cmp_lt_f32_e64 %[lt], %[bm], %[m]\n\t"
            "v_med3_f32 %[m2], %[m], %[m2], %[bm]\n\t"
            "s_and_saveexec_b64 %[save], %[lt]\n\t"
            "v_mov_b32 %[m], %[bm]\n\t"
            "v_mov_b32 %[blk], %[cb]\n\t"
            "v_mov_b64 %[k0], %[d0]\n\t"
            "v_mov_b64 %[k1], %[d1]\n\t"
            "v_mov_b64 %[k2], %[d2]\n\t"
            "s_mov_b64 exec, %[save]"
            : [lt] "=&s"(s.lt), [save] "=&s"(save), [m] "+v"(b.m), [m2] "+v"(b.m2), [blk] "+v"(b.blk), [k0] "+v"(b.keep[0]),
              [k1] "+v"(b.keep[1]), [k2] "+v"(b.keep[2])
            : [bm] "v"(s.bm), [cb] "s"(cb), [d0] "v"(floatx2{d[0], d[1]}), [d1] "v"(floatx2{d[2], d[3]}),
              [d2] "v"(floatx2{d[4], d[5]})
            : "scc");
    if (PIECE == 2)
        asm("s_and_saveexec_b64 %[save], %[lt]\n\t"
            "v_mov_b64 %[k3], %[d3]\n\t"
            "v_mov_b64 %[k4], %[d4]\n\t"
            "v_mov_b64 %[k5], %[d5]\n\t"
            "v_mov_b64 %[k6], %[d6]\n\t"
            "v_mov_b64 %[k7], %[d7]\n\t"
            "s_mov_b64 exec, %[save]"
            : [save] "=&s"(save), [k3] "+v"(b.keep[3]), [k4] "+v"(b.keep[4]), [k5] "+v"(b.keep[5]),
              [k6] "+v"(b.keep[6]), [k7] "+v"(b.keep[7])
            : [lt] "s"(s.lt), [d3] "v"(floatx2{d[6], d[7]}), [d4] "v"(floatx2{d[8], d[9]}),
              [d5] "v"(floatx2{d[10], d[11]}), [d6] "v"(floatx2{d[12], d[13]}), [d7] "v"(floatx2{d[14], d[15]})
            : "scc");
}
__device__ __forceinline__ void split_scan_all(const floatx16& d, int cb, SplitBest& b) {
    SplitScan sc;
    split_scan_piece<0>(sc, d, cb, b);
    split_scan_piece<1>(sc, d, cb, b);
    split_scan_piece<2>(sc, d, cb, b);
}
__device__ __forceinline__ int split_best_index(const SplitBest& b) {
    floatx16 keep;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        keep[2 * i] = b.keep[i][0];
        keep[2 * i + 1] = b.keep[i][1];
    }
    return kept_argmin(keep, b.m, b.blk);
}

// Rows whose two nearest centroids lie closer together than the rounding of the distances: whether another distance is
// within 12 units of 2^-24 (2.5 |x|^2 + 2 d) of the smallest, about 12 units of 2^-24 (|x|^2 + |c|^2).  (What two
// distances of one row err against each other by, fp32 chain and split products taken together, has an rms of 1.9 to 2.4 such
// units.)  xs = S^2 |x|^2.
__device__ __forceinline__ bool split_is_near(const SplitBest& b, float xs) {
    const float m = fminf(b.m, __shfl_xor(b.m, 32));
    const float lim = m + 0x1.8p-21f * (2.5f * xs + 2.0f * fmaxf(m + xs, 0.0f));
    int n = b.m2 <= lim ? 1 : 0;
#pragma unroll
    for (int i = 0; i < 8; ++i) n += (b.keep[i][0] <= lim ? 1 : 0) + (b.keep[i][1] <= lim ? 1 : 0);
    n = b.m <= lim ? n : 0;
    return n + __shfl_xor(n, 32) >= 2;
}

// Such a row is decided by the fp32 product chain (|c|^2 - 2 x_0 c_0 - 2 x_h c_h - 2 x_1 c_1 - ..., h = half the padded
// width: the order of the fp32 matrix kernels), so that the labels of a fit do not depend on which products found
// them: iterations amplify a single tied row that changes sides.  All lanes of the wave work on the row, lane l on the
// centroids l, l + 64, ...  TILED: clamped as the kernel for more centroids than LDS holds does it.
// Out of line: the registers of the caller's tile are put aside for the rare row that needs this.
template <int HALF, bool TILED>
__device__ __noinline__ void split_near_row(const float* __restrict__ x, const float* __restrict__ C, int K, int64_t ldc,
                                            int D, float& m_out, int& i_out) {
    const int lane = threadIdx.x & 63;
    auto load4 = [&](const float* row, int c) { return c + 4 <= D ? ld4_any(row + c) : load_row4<false>(row, c, D); };
    floatx4 xr[HALF / 2];
    float s[2] = {0.f, 0.f};
#pragma unroll
    for (int g = 0; g < HALF / 2; ++g) xr[g] = load4(x, 4 * g);
#pragma unroll
    for (int g = 0; g < HALF / 2; ++g)
#pragma unroll
        for (int t = 0; t < 4; ++t) s[g / (HALF / 4)] = fmaf(xr[g][t], xr[g][t], s[g / (HALF / 4)]);
    const float xn = s[0] + s[1];
    for (int pass = 0; pass < 2; ++pass) {  // the second one: distances clamped at 0 before they are compared
        float m = HKM_INF;
        int mi = 0x7fffffff;
        for (int k = lane; k < K; k += 64) {
            const float* c = C + int64_t(k) * ldc;
            floatx4 cr[HALF / 2];
#pragma unroll
            for (int g = 0; g < HALF / 2; ++g) cr[g] = load4(c, 4 * g);
            float a = 0.f;
#pragma unroll
            for (int g = 0; g < HALF / 2; ++g)
#pragma unroll
                for (int t = 0; t < 4; ++t) a = fmaf(cr[g][t], cr[g][t], a);
#pragma unroll
            for (int g = 0; g < HALF / 4; ++g)
#pragma unroll
                for (int t = 0; t < 4; ++t) {
                    a = fmaf(-2.0f * cr[g][t], xr[g][t], a);
                    a = fmaf(-2.0f * cr[HALF / 4 + g][t], xr[HALF / 4 + g][t], a);
                }
            if (pass == 1) a = fmaxf(a + xn, 0.0f);
            if (a < m) {
                m = a;
                mi = k;
            }
        }
        auto take = [&](float om, int oi) {
            if (om < m || (om == m && oi < mi)) {
                m = om;
                mi = oi;
            }
        };
        // centroids whose index has the bit 4 were the other lane-half's: compared with |x|^2 added
#pragma unroll
        for (int o = 1; o < 64; o <<= 1)
            if (o != 4) take(__shfl_xor(m, o), __shfl_xor(mi, o));
        if (pass == 0) m += xn;
        if (TILED) m = fmaxf(m, 0.0f);
        take(__shfl_xor(m, 4), __shfl_xor(mi, 4));
        m_out = m;
        i_out = mi;
        if (!(m < 0.f)) return;
    }
}

template <int DP, bool TILED>
__device__ __forceinline__ void split_near_rows(unsigned long long rows, const float* __restrict__ x0, int64_t ldx,
                                                const float* __restrict__ C, int K, int64_t ldc, int D, int p, float& m,
                                                int& mi) {
    while (rows) {
        const int r = __builtin_ctzll(rows);
        rows &= rows - 1;
        float nm;
        int ni;
        const float* x = x0 + int64_t(r) * ldx;
        // half of the fp32 kernels' padded width: 24 for 17 to 24 features, else the one here
        if (DP == 32 && D <= 24) split_near_row<12, TILED>(x, C, K, ldc, D, nm, ni);
        else split_near_row<DP / 2, TILED>(x, C, K, ldc, D, nm, ni);
        if (p == r) {
            m = nm;
            mi = ni;
        }
    }
}

// One unit of the pipeline below: the products of one centroid block with one point block, from the norms c0; between
// the matrix instructions the pieces of the scan of an earlier unit's results (SCAN), and (RELOAD) the operand
// registers are refilled for the next block as soon as their last reader has been issued.
template <int DP, bool SCAN, bool RELOAD>
__device__ __forceinline__ floatx16 split_unit(halfx8 (&ch)[DP / 16], halfx8 (&cl)[DP / 16], const floatx16& c0,
                                               const halfx8 (&xh)[DP / 16], const halfx8 (&xl)[DP / 16],
                                               const floatx16& old, int cb_old, SplitBest& best,
                                               const _Float16* const (&next)[DP / 16]) {
    constexpr int NS = DP / 16;
    SplitScan sc{};
    floatx16 acc = c0;
#pragma unroll
    for (int i = 0; i < 3 * NS; ++i) {
        const int st = i / 3, t = i % 3;
        if (t == 0) acc = MFMA_F16(cl[st], xh[st], acc);
        if (t == 1) acc = MFMA_F16(ch[st], xl[st], acc);
        if (t == 2) acc = MFMA_F16(ch[st], xh[st], acc);
        if (RELOAD) {
            if (t == 0) cl[st] = ld_half8(next[st] + 32 * DP);
            if (t == 2) ch[st] = ld_half8(next[st]);
        }
        if (SCAN) {
            if (i == 1) split_scan_piece<0>(sc, old, cb_old, best);
            if (i == 2) split_scan_piece<1>(sc, old, cb_old, best);
            if (i == 3) split_scan_piece<2>(sc, old, cb_old, best);
        }
        __builtin_amdgcn_sched_barrier(0);
    }
    return acc;
}

// Scan of all centroid blocks for point blocks that take the shared scale, as a software pipeline: a wave issues in
// order, and the vector ALU works beside the matrix core only on what is issued between its instructions, so the
// scan of one unit's results sits between the matrix instructions of the next unit, and the LDS reads of the next
// centroid block between those of the block before it.  Two centroid blocks per trip, so that the norms of a block
// become the accumulators of its last unit in place.
// The running minima (best) are carried over from the blocks before; the first block here has the number cb0.
template <int DP, int PB>
__device__ __forceinline__ void split_scan(const _Float16* planes, const float* sCn, int ncb, int cb0, int p, int h,
                                           const halfx8 (&xh)[PB][DP / 16], const halfx8 (&xl)[PB][DP / 16],
                                           SplitBest (&best)[PB]) {
    constexpr int NS = DP / 16, P1 = PB - 1;
    const _Float16* next[NS];
    halfx8 ch[NS], cl[NS];
#pragma unroll
    for (int st = 0; st < NS; ++st) {
        next[st] = planes + split_off<DP>(p, h, st);
        ch[st] = ld_half8(next[st]);
        cl[st] = ld_half8(next[st] + 32 * DP);
    }
    const float* next_cn = sCn + 4 * h;
    // the block after cb (behind the last one that block again: read, not used)
    auto advance = [&](int cb) {
        const int by = cb + 1 < ncb ? 1 : 0;
#pragma unroll
        for (int st = 0; st < NS; ++st) next[st] += by * (64 * DP);
        next_cn += by * 32;
    };
    floatx16 c0a = load_cn16(next_cn), c0b;
    floatx16 acc0, acc1;
    if constexpr (PB == 2) {
        acc0 = split_unit<DP, false, false>(ch, cl, c0a, xh[0], xl[0], c0a, 0, best[0], next);
        int cb = 0;
#pragma unroll 1
        for (; cb + 2 < ncb; cb += 2) {
            advance(cb);
            c0b = load_cn16(next_cn);
            acc1 = split_unit<DP, true, true>(ch, cl, c0a, xh[P1], xl[P1], acc0, cb0 + cb, best[0], next);
            acc0 = split_unit<DP, true, false>(ch, cl, c0b, xh[0], xl[0], acc1, cb0 + cb, best[P1], next);
            advance(cb + 1);
            c0a = load_cn16(next_cn);
            acc1 = split_unit<DP, true, true>(ch, cl, c0b, xh[P1], xl[P1], acc0, cb0 + cb + 1, best[0], next);
            acc0 = split_unit<DP, true, false>(ch, cl, c0a, xh[0], xl[0], acc1, cb0 + cb + 1, best[P1], next);
        }
        if (cb + 1 < ncb) {
            advance(cb);
            c0b = load_cn16(next_cn);
            acc1 = split_unit<DP, true, true>(ch, cl, c0a, xh[P1], xl[P1], acc0, cb0 + cb, best[0], next);
            acc0 = split_unit<DP, true, false>(ch, cl, c0b, xh[0], xl[0], acc1, cb0 + cb, best[P1], next);
            acc1 = split_unit<DP, true, false>(ch, cl, c0b, xh[P1], xl[P1], acc0, cb0 + cb + 1, best[0], next);
        } else {
            acc1 = split_unit<DP, true, false>(ch, cl, c0a, xh[P1], xl[P1], acc0, cb0 + cb, best[0], next);
        }
        split_scan_all(acc1, cb0 + ncb - 1, best[P1]);
    } else {
        advance(0);
        c0b = load_cn16(next_cn);
        acc0 = split_unit<DP, false, true>(ch, cl, c0a, xh[0], xl[0], c0a, 0, best[0], next);
        int cb = 1;
#pragma unroll 1
        for (; cb + 1 < ncb; cb += 2) {
            advance(cb);
            c0a = load_cn16(next_cn);
            acc1 = split_unit<DP, true, true>(ch, cl, c0b, xh[0], xl[0], acc0, cb0 + cb - 1, best[0], next);
            advance(cb + 1);
            c0b = load_cn16(next_cn);
            acc0 = split_unit<DP, true, true>(ch, cl, c0a, xh[0], xl[0], acc1, cb0 + cb, best[0], next);
        }
        if (cb < ncb) acc0 = split_unit<DP, true, false>(ch, cl, c0b, xh[0], xl[0], acc0, cb0 + cb - 1, best[0], next);
        split_scan_all(acc0, cb0 + ncb - 1, best[0]);
    }
}

// operand parts of a lane's half row, scaled by s (a power of two)
template <int NS>
__device__ __forceinline__ void split_row(const floatx4 (&b)[2 * NS], float s, halfx8 (&xh)[NS], halfx8 (&xl)[NS]) {
#pragma unroll
    for (int st = 0; st < NS; ++st)
#pragma unroll
        for (int q = 0; q < 8; q += 2) {
            const floatx4& g = b[2 * st + (q >> 2)];
            const floatx2 v = {g[q & 3] * s, g[(q & 3) + 1] * s};
            const halfx2 v1 = __builtin_convertvector(v, halfx2);
            const floatx2 r = {fmaf(g[q & 3], s, -float(v1[0])), fmaf(g[(q & 3) + 1], s, -float(v1[1]))};
            const halfx2 v2 = __builtin_convertvector(r, halfx2);
#pragma unroll
            for (int e = 0; e < 2; ++e) {
                xh[st][q + e] = v1[e];
                xl[st][q + e] = v2[e];
            }
        }
}

// |x|^2 of a row from its two lanes, in eight chains: one chain of D terms would be the largest error of a distance
template <int NJ>
__device__ __forceinline__ float row_norm(const floatx4 (&b)[NJ]) {
    floatx4 n = b[0] * b[0];
#pragma unroll
    for (int j = 1; j < NJ; ++j)
#pragma unroll
        for (int t = 0; t < 4; ++t) n[t] = fmaf(b[j][t], b[j][t], n[t]);
    const float s = (n[0] + n[1]) + (n[2] + n[3]);
    return s + __shfl_xor(s, 32);
}

// Rows with a non-finite |x|^2, in fp32 on the vector ALU: the minimum of |c|^2 - 2 x.c over all centroids (NaNs
// never win).  The two lanes that share a row add their halves; both end with the same result.
template <int DP>
__device__ void split_scan_plain(const float* __restrict__ C, int K, int64_t ldc, int D, int h,
                                 const floatx4 (&b)[DP / 8], float& m, int& mi) {
    m = HKM_INF;
    mi = 0;
    for (int k = 0; k < K; ++k) {
        const float* c = C + int64_t(k) * ldc;
        float s = 0.f, cn = 0.f;
        for (int d = 0; d < D; ++d) cn = fmaf(c[d], c[d], cn);
#pragma unroll
        for (int j = 0; j < DP / 8; ++j)
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                const int d = h * (DP / 2) + 4 * j + t;
                if (d < D) s = fmaf(-2.0f * c[d], b[j][t], s);
            }
        s += __shfl_xor(s, 32);
        s += cn;
        if (s < m) {
            m = s;
            mi = k;
        }
    }
}

// Threads of a workgroup: the step keeps one workgroup per CU (its sums fill the LDS); the assignment alone two.
__host__ __device__ constexpr int split_pb(int dp) { return dp <= 32 ? 2 : 1; }
__host__ __device__ constexpr int split_threads(int dp, bool fused) {
    return !fused ? 256 : 512;
}

// FUSED: also the per-cluster sums (fsum / fcnt / flags as in lloyd_mfma_resident_kernel)
template <int DP, bool FULL, bool FUSED>
__global__ __launch_bounds__(split_threads(DP, FUSED)) void split_resident_kernel(
    const float* __restrict__ X, int64_t N, int D, int64_t ldx, const float* __restrict__ C, int K,
    int64_t ldc, int32_t* __restrict__ labels, float* __restrict__ min_d2, int64_t ntiles,
    double* __restrict__ fsum, int32_t* __restrict__ fcnt, int32_t* __restrict__ flags, int range_bits, int nrep) {
    extern __shared__ __align__(16) unsigned char lds_raw[];
    constexpr int PB = split_pb(DP);
    constexpr int NJ = DP / 8;   // 16-byte groups of fp32 per lane-half
    constexpr int NS = DP / 16;  // k-steps of the matrix instruction
    const int LDA = D | 1;       // odd row stride (in doubles): rows of different clusters spread over the banks
    const int KP = (K + 31) & ~31;
    _Float16* planes = reinterpret_cast<_Float16*>(lds_raw);    // [KP / 32][2][32][DP]
    float* sCn = reinterpret_cast<float*>(planes + 2 * KP * DP);  // [KP] S^2 |c|^2, +inf beyond K
    float* sI = sCn + KP;                                       // [KP] S / scale of the centroid
    int* sMeta = reinterpret_cast<int*>(sI + KP);               // [8]
    const size_t rstride = size_t(K) * LDA + 1;
    double* sA = reinterpret_cast<double*>(sMeta + 8);          // FUSED: [nrep][K][LDA] (+ 1 pad per copy)
    int* sN = reinterpret_cast<int*>(sA + (FUSED ? nrep * rstride : 0));  // FUSED: [nrep][K] counts
    const int tid = threadIdx.x, nthr = blockDim.x;

    // sMeta: Emin, Emax, non-finite, largest / smallest non-zero centroid norm, largest |coordinate|, no shared scale
    if (tid < 8) sMeta[tid] = tid == 0 || tid == 4 ? 0x7fffffff : tid == 1 ? -0x7fffffff : 0;
    __syncthreads();
    // eight lanes per centroid row (KP is a multiple of 32, the workgroup of 64: no lane group is cut)
    constexpr int EPL = DP / 8;
    for (int i = tid; i < KP * 8; i += nthr) {
        const int r = i >> 3, d0 = (i & 7) * EPL;
        float s = 0.f;
        int mx = 0;
        if (r < K)
#pragma unroll
            for (int e = 0; e < EPL; ++e)
                if (d0 + e < D) {
                    const float c = C[int64_t(r) * ldc + d0 + e];
                    s = fmaf(c, c, s);
                    mx = max(mx, __float_as_int(c) & 0x7fffffff);  // bits of non-negative floats order like integers
                }
#pragma unroll
        for (int o = 1; o < 8; o <<= 1) {
            s += __shfl_xor(s, o);
            mx = max(mx, __shfl_xor(mx, o));
        }
        if ((i & 7) == 0) {
            sCn[r] = s;
            sI[r] = __int_as_float(mx);
            if (r < K) {
                const int b = __float_as_int(s) & 0x7fffffff;
                atomicMax(&sMeta[3], b);
                if (b != 0) atomicMin(&sMeta[4], b);
                atomicMax(&sMeta[5], mx);
            }
        }
    }
    if (FUSED) {
        for (int i = tid; i < int(nrep * rstride); i += nthr) sA[i] = 0.0;
        for (int i = tid; i < nrep * K; i += nthr) sN[i] = 0;
    }
    __syncthreads();
    const float cmax = __int_as_float(sMeta[5]);
    const int ecm = (sMeta[5] >> 23) - 126;  // cmax < 2^ecm
    if (ecm < -20 || ecm > 40) {
        if (tid == 0) sMeta[6] = 1;
    } else {
        const float least = float(D) * cmax * cmax * 0x1p-12f;
        for (int r = tid; r < K; r += nthr)
            if (sI[r] != 0.f && sCn[r] < least) sMeta[6] = 1;
    }
    __syncthreads();
    const bool shared_scale = sMeta[6] == 0;
    const float S = shared_scale ? ldexpf(1.0f, 8 - ecm) : 1.0f;
    const float S2 = S * S, inv_s2 = 1.0f / S2;
    // position of coordinate c of centroid r's high part; the low part lies 32 rows further
    auto plane_at = [](int r, int c) {
        return (r >> 5) * (64 * DP) + (r & 31) * DP + 8 * ((c >> 3) ^ split_swz<DP>(r & 31)) + (c & 7);
    };
    // scale of centroid r, from its largest |coordinate|
    auto cscale = [&](float mx) {
        const int e = (__float_as_int(mx) >> 23) - 126;
        return mx == 0.f || e > 128 ? 1.0f : ldexpf(1.0f, 8 - max(e, -100));
    };
    for (int i = tid; i < KP * 8; i += nthr) {
        const int r = i >> 3, d0 = (i & 7) * EPL;
        const float s = shared_scale ? S : cscale(sI[r]);
        double n = 0.0;  // |c|^2 of the split centroid (the planes hold -2 s c)
#pragma unroll
        for (int e = 0; e < EPL; e += 2) {
            halfx2 v1, v2;
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                const float v = (r < K && d0 + e + q < D) ? -2.0f * s * C[int64_t(r) * ldc + d0 + e + q] : 0.f;
                v1[q] = _Float16(v);
                v2[q] = _Float16(v - float(v1[q]));
                const double w = double(float(v1[q]) + float(v2[q]));
                n += w * w;
            }
            const int o = plane_at(r, d0 + e);
            *reinterpret_cast<halfx2*>(planes + o) = v1;
            *reinterpret_cast<halfx2*>(planes + o + 32 * DP) = v2;
        }
#pragma unroll
        for (int o = 1; o < 8; o <<= 1) n += __shfl_xor(n, o);
        const float f = S / s;
        if ((i & 7) == 0) {  // (the lanes of a row are in one wave: its scale has been read)
            sCn[r] = r < K ? 0.25f * float(n) * f * f : HKM_INF;  // padding rows can never win
            sI[r] = f;
        }
    }
    __syncthreads();
    // quanta of the pre-rounded rows: see lloyd_mfma_resident_kernel
    int e_floor = -0x3fffffff;
    if (FUSED) {
        const int cexp = (sMeta[3] >> 23) & 0xff, cexp_min = (sMeta[4] >> 23) & 0xff;
        if (cexp != 0 && cexp != 255) {
            const int e_ref = ((cexp - 127) >> 1) + 2, e_min = ((cexp_min - 127) >> 1) + 2;
            const int head = range_bits < 4 ? (range_bits < 0 ? 0 : range_bits) : 4;
            e_floor = min(e_ref + head - range_bits, e_min + 4);
        }
    }
    // |x|^2 of the rows that may take the shared scale
    const float xn_lo = shared_scale ? float(D) * inv_s2 : HKM_INF, xn_hi = shared_scale ? 0x1p28f * inv_s2 : 0.f;

    const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), nw = nthr >> 6;
    const int p = lane & 31, h = lane >> 5;
    const int ncb = KP >> 5;
    const int64_t tile_rows = int64_t(nw) * PB * 32;
    const bool fast = ldx < (int64_t(1) << 24);
    const unsigned lane_off = unsigned((int64_t(p) * ldx + h * (DP / 2)) * 4);
    double* sA_lane = sA + (FUSED ? (p & (nrep - 1)) * rstride : 0);
    int* sN_lane = sN + (FUSED ? (p & (nrep - 1)) * K : 0);
    int emin = 0x7fffffff, emax = -0x7fffffff;
    int nonfinite = 0;

    auto step = [&](int64_t tile, const floatx4 (&b)[PB][NJ], floatx4 (&bnext)[PB][NJ]) {
        const int64_t row0 = tile * tile_rows + wave * (PB * 32);
        float xnr[PB], m[PB], rx[PB];
        int mi[PB];
        bool in[PB];  // the row takes the shared scale
        bool near[PB];
        halfx8 xh[PB][NS], xl[PB][NS];
        bool rest = false;
#pragma unroll
        for (int pb = 0; pb < PB; ++pb) {
            xnr[pb] = row_norm<NJ>(b[pb]);
            in[pb] = (xnr[pb] >= xn_lo && xnr[pb] <= xn_hi) || (shared_scale && xnr[pb] == 0.f);
            rest |= !in[pb];
            rx[pb] = 1.0f;
            near[pb] = false;
        }
        if (tile + gridDim.x < ntiles)
            fetch_rows_any<DP, PB, FULL>(X, N, D, ldx, row0 + int64_t(gridDim.x) * tile_rows, p, h, fast, lane_off, bnext);

        if (shared_scale) {
#pragma unroll
            for (int pb = 0; pb < PB; ++pb) split_row<NS>(b[pb], S, xh[pb], xl[pb]);
            SplitBest best[PB];
#pragma unroll
            for (int pb = 0; pb < PB; ++pb) split_best_init(best[pb]);
            split_scan<DP, PB>(planes, sCn, ncb, 0, p, h, xh, xl, best);
#pragma unroll
            for (int pb = 0; pb < PB; ++pb) {
                near[pb] = split_is_near(best[pb], xnr[pb] * S2) && in[pb];
                mi[pb] = split_best_index(best[pb]);
                m[pb] = fmaf(best[pb].m, inv_s2, xnr[pb]);
                rest |= m[pb] < 0.f;
            }
        }
        if (__any(rest)) {
            // rows outside the shared scale's range, and rows whose distance came out below 0
            float m1[PB];
            int mi1[PB];
            bool odd[PB], neg = false;
#pragma unroll
            for (int pb = 0; pb < PB; ++pb) {
                odd[pb] = ((__float_as_int(xnr[pb]) >> 23) & 0xff) == 255;
                const int e = ((((__float_as_int(xnr[pb]) >> 23) & 0xff) - 127) >> 1) + 1;  // |x_d| < 2^e
                const float sx = xnr[pb] > 0.f ? ldexpf(1.0f, 14 - e) : 1.0f;
                rx[pb] = S / sx;
                split_row<NS>(b[pb], sx, xh[pb], xl[pb]);
            }
            auto scan_own = [&](auto clamp) {
                int blk[PB];
                floatx16 keep[PB];
#pragma unroll
                for (int pb = 0; pb < PB; ++pb) {
                    m1[pb] = HKM_INF;
                    blk[pb] = 0;
                    keep_undefined(keep[pb]);
                }
                split_scan_own<DP, PB, decltype(clamp)::value>(planes, sCn, sI, ncb, 0, p, h, xh, xl, rx, inv_s2, xnr, m1,
                                                               blk, keep);
#pragma unroll
                for (int pb = 0; pb < PB; ++pb) mi1[pb] = kept_argmin(keep[pb], m1[pb], blk[pb]);
            };
            scan_own(std::integral_constant<bool, false>{});
#pragma unroll
            for (int pb = 0; pb < PB; ++pb) {
                m[pb] = in[pb] ? m[pb] : fmaf(m1[pb], inv_s2, xnr[pb]);
                mi[pb] = in[pb] ? mi[pb] : mi1[pb];
                neg |= m[pb] < 0.f;
            }
            if (__any(neg)) {
                scan_own(std::integral_constant<bool, true>{});
#pragma unroll
                for (int pb = 0; pb < PB; ++pb) {
                    mi[pb] = m[pb] < 0.f ? mi1[pb] : mi[pb];
                    m[pb] = m[pb] < 0.f ? m1[pb] : m[pb];
                }
            }
#pragma unroll
            for (int pb = 0; pb < PB; ++pb) {
                if (__any(odd[pb])) {
                    float mp;
                    int mip;
                    split_scan_plain<DP>(C, K, ldc, D, h, b[pb], mp, mip);
                    if (odd[pb]) {
                        m[pb] = mp + xnr[pb];
                        mi[pb] = mip - 4 * h;  // the lane-half term is added below
                    }
                }
            }
        }

#pragma unroll
        for (int pb = 0; pb < PB; ++pb) {
            mi[pb] += 4 * h;
            merge_halves(m[pb], mi[pb]);
            const int64_t rb = row0 + pb * 32;  // wave-uniform: the stores take it as their scalar base
            const bool valid = rb + p < N;
            const unsigned long long ties = __ballot(near[pb] && valid && h == 0);
            if (ties) split_near_rows<DP, false>(ties, X + rb * ldx, ldx, C, K, ldc, D, p, m[pb], mi[pb]);
            if (h == 0 && valid) {
                labels[rb + p] = mi[pb];
                if (min_d2) min_d2[rb + p] = m[pb];
                if (FUSED) atomicAdd(&sN_lane[mi[pb]], 1);
            }
            if (FUSED && valid && xnr[pb] != 0.f) {  // an all-zero row adds nothing
                // |x_d| < 2^E: |x|^2 < 2^(e2+1) up to rounding, one more bit of slack
                const int e2 = (__float_as_int(xnr[pb]) >> 23) - 127;
                nonfinite |= int((e2 & 0xff) == 128);  // exponent field 255 (the sign bit of |x|^2 is clear or NaN)
                const int E = max((e2 >> 1) + 2, e_floor);
                emin = min(emin, E);
                emax = max(emax, E);
                const double B = __hiloint2double(((1023 + 52 - SPLIT_QBITS + E) << 20) | 0x80000, 0);
                double* row = sA_lane + mi[pb] * LDA + h * (DP / 2);
#pragma unroll
                for (int j = 0; j < NJ; ++j)
#pragma unroll
                    for (int t = 0; t < 4; ++t) {
                        const double v = (double(b[pb][j][t]) + B) - B;
                        if (FULL || h * (DP / 2) + 4 * j + t < D)
                            __hip_atomic_fetch_add(row + 4 * j + t, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                    }
            }
        }
    };

    floatx4 b0[PB][NJ], b1[PB][NJ];
    if (int64_t(blockIdx.x) < ntiles)
        fetch_rows_any<DP, PB, FULL>(X, N, D, ldx, int64_t(blockIdx.x) * tile_rows + wave * (PB * 32), p, h, fast,
                                     lane_off, b0);
    for (int64_t tile = blockIdx.x; tile < ntiles; tile += 2 * int64_t(gridDim.x)) {
        step(tile, b0, b1);
        if (tile + gridDim.x < ntiles) step(tile + gridDim.x, b1, b0);
    }

    if (FUSED) {
        atomicMin(&sMeta[0], emin);
        atomicMax(&sMeta[1], emax);
        if (nonfinite) atomicOr(&sMeta[2], 1);
        __syncthreads();
        double* gs = fsum + size_t(blockIdx.x) * K * D;
        for (int i = tid; i < K * D; i += nthr) {
            const int k = i / D, d = i - k * D;
            double v = 0.0;  // exact whatever the order (or the flag is up and the value unused)
            for (int r = 0; r < nrep; ++r) v += sA[r * rstride + size_t(k) * LDA + d];
            gs[i] = v;
        }
        for (int i = tid; i < K; i += nthr) {
            int c = 0;
            for (int r = 0; r < nrep; ++r) c += sN[r * K + i];
            fcnt[size_t(blockIdx.x) * K + i] = c;
        }
        if (tid == 0) {
            const int l = sMeta[0], u = sMeta[1];
            flags[blockIdx.x] = ((u >= l && u - l > range_bits) || sMeta[2]) ? 1 : 0;
        }
    }
}

// feature padding of the split kernels: whole k-steps of 16
static int split_dp(int32_t D) { return D <= 32 ? 32 : D <= 48 ? 48 : 64; }

static size_t split_lds_bytes(int32_t D, int32_t K, bool fused, int nrep) {
    const size_t kp = (size_t(K) + 31) / 32 * 32;
    size_t b = kp * split_dp(D) * 4 + kp * 8 + 32;
    if (fused) b += size_t(nrep) * ((size_t(K) * (D | 1) + 1) * sizeof(double) + size_t(K) * sizeof(int)) + 16;
    return b;
}

// copies of the fp64 accumulators: see fused_replicas (hkm_assign_mfma.hip)
static int split_replicas(int32_t D, int32_t K) {
    int r = K <= 32 ? 16 : K <= 64 ? 4 : 1;
    while (r > 1 && split_lds_bytes(D, K, true, r) > size_t(128) * 1024) r >>= 1;
    return r;
}

// Rows of more than 16 features; a few shapes of 17 to 24 features with 400 clusters or more, whose rows padded to
// 32 features do not fit the LDS beside the sums, stay on the fp32 kernel.
bool split_eligible(int32_t D, int32_t K, bool fused) {
    if (D <= 16 || D > 64) return false;
    return split_lds_bytes(D, K, fused, fused ? split_replicas(D, K) : 1) <= (fused ? size_t(160) : size_t(80)) * 1024;
}

int split_point_blocks(int32_t D) { return split_pb(split_dp(D)); }

int split_fused_grid(int64_t N, int32_t D) {
    const int dp = split_dp(D);
    const int64_t tile_rows = int64_t(split_threads(dp, true) / 64) * split_pb(dp) * 32;
    const int64_t ntiles = (N + tile_rows - 1) / tile_rows;
    int64_t grid = num_cus();
    if (grid > FUSED_MAX_GRID) grid = FUSED_MAX_GRID;
    if (grid > ntiles) grid = ntiles;
    return int(grid < 1 ? 1 : grid);
}

template <int DP, bool FULL, bool FUSED>
static int launch_split_t(const float* X, int64_t N, int32_t D, int64_t ldx, const float* C, int32_t K,
                          int64_t ldc, int32_t* labels, float* min_d2, double* fsum, int32_t* fcnt,
                          int32_t* flags, hipStream_t st) {
    constexpr int THREADS = split_threads(DP, FUSED);
    const int64_t tile_rows = int64_t(THREADS / 64) * split_pb(DP) * 32;
    const int64_t ntiles = (N + tile_rows - 1) / tile_rows;
    const int nrep = FUSED ? split_replicas(D, K) : 1;
    const size_t lds = split_lds_bytes(D, K, FUSED, nrep);
    auto kern = split_resident_kernel<DP, FULL, FUSED>;
    if (lds > 64 * 1024) {
        hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                                           hipFuncAttributeMaxDynamicSharedMemorySize, int(lds));
        if (e != hipSuccess) return fail(HKM_EHIP, "hipFuncSetAttribute: %s", hipGetErrorString(e));
    }
    int64_t grid = 0;
    int range_bits = 0;
    if (FUSED) {
        grid = split_fused_grid(N, D);
        // rows one workgroup adds up, as a power of two
        const int64_t per_wg = (ntiles + grid - 1) / grid * tile_rows;
        int lg = 0;
        while ((int64_t(1) << lg) < per_wg) ++lg;
        range_bits = 53 - SPLIT_QBITS - lg;
    } else {
        // persistent grid: as many workgroups as are resident at once
        int per_cu = 0;
        hipError_t oe = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, reinterpret_cast<const void*>(kern), THREADS, lds);
        if (oe != hipSuccess) return fail(HKM_EHIP, "hipOccupancyMaxActiveBlocksPerMultiprocessor: %s", hipGetErrorString(oe));
        per_cu = per_cu < 1 ? 1 : per_cu > 4 ? 4 : per_cu;
        grid = int64_t(num_cus()) * per_cu;
        if (grid > ntiles) grid = ntiles;
    }
    prof_begin(st);
    hipLaunchKernelGGL(kern, dim3((unsigned)grid), dim3(THREADS), lds, st, X, N, D, ldx, C, K, ldc, labels,
                       min_d2, ntiles, fsum, fcnt, flags, range_bits, nrep);
    prof_end(st);
    return check_launch("split_resident_kernel");
}

// fsum == NULL: distance + argmin only
int launch_split_resident(const float* X, int64_t N, int32_t D, int64_t ldx, const float* C, int32_t K,
                          int64_t ldc, int32_t* labels, float* min_d2, double* fsum, int32_t* fcnt,
                          int32_t* flags, hipStream_t st) {
    const int dp = split_dp(D);
    const bool full = D == dp, fused = fsum != nullptr;
#define HKM_CASE(d)                                                                                              \
    case d:                                                                                                      \
        if (fused)                                                                                               \
            return full ? launch_split_t<d, true, true>(X, N, D, ldx, C, K, ldc, labels, min_d2, fsum, fcnt, flags, st)  \
                        : launch_split_t<d, false, true>(X, N, D, ldx, C, K, ldc, labels, min_d2, fsum, fcnt, flags, st); \
        return full ? launch_split_t<d, true, false>(X, N, D, ldx, C, K, ldc, labels, min_d2, fsum, fcnt, flags, st)     \
                    : launch_split_t<d, false, false>(X, N, D, ldx, C, K, ldc, labels, min_d2, fsum, fcnt, flags, st);
    switch (dp) {
        HKM_CASE(32) HKM_CASE(48) HKM_CASE(64)
        default:
            return fail(HKM_EUNSUPPORTED, "split_resident: D=%d", D);
    }
#undef HKM_CASE
}

// ------------------------------------------------------------------------------------------------
// 16 < D <= 64 with more centroids than LDS holds: a wave keeps the parts of its 64 rows in registers and scans
// centroid tiles of 128 rows that all threads split on their way into one of two LDS buffers, one barrier per tile.  The
// running minima are carried across tiles and the clamp at 0 is applied to the final minimum: where several centroids
// coincide with a point up to rounding (several negative values) the most negative one wins instead of the first -- a tie
// at the resolution of the formula.  Squared centroid norms come from global memory (cn, +inf beyond K).  Rows outside
// the shared scale's range (here S takes the largest centroid norm into [2^9, 2^10)) make their workgroup walk the
// tiles once more with scales of their own.
//
// What bounds it (1M x 64, K = 1024: 0.505 ms a call, 0.466 without the rule for tied rows): the matrix cores 40 % of the cycles; the waits at the barrier
// per tile and the first operand reads behind it most of the rest.  fp32 kernel -> this one: 1M x 64, K = 1024: 1043 ->
// 478 us; x 48, 1500: 1180 -> 435; x 32, 1500: 821 -> 265; 300k x 33, 700: 235 -> 122; 1000 x 64, 2048: 81 -> 55.
// ------------------------------------------------------------------------------------------------
static constexpr int TILED_TC = 128, TILED_THREADS = 512;

template <int DP, bool FULL>
__global__ __launch_bounds__(TILED_THREADS) void split_tiled_kernel(
    const float* __restrict__ X, int64_t N, int D, int64_t ldx, const float* __restrict__ C, int K, int64_t ldc,
    const float* __restrict__ cn, int32_t* __restrict__ labels, float* __restrict__ min_d2, int64_t ntiles) {
    constexpr int PB = 2, NJ = DP / 8, NS = DP / 16, TC = TILED_TC, TCB = TC / 32;
    constexpr int GPR = DP / 4, NQ = TC * GPR / TILED_THREADS;  // 16-byte groups per centroid row; per thread and tile
    __shared__ __align__(16) _Float16 sP[2][2 * TC * DP];
    __shared__ __align__(16) float sCn[2][TC], sI[2][TC];
    __shared__ int sMeta[2];
    const int tid = threadIdx.x;
    const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int p = lane & 31, h = lane >> 5;
    const int nct = (K + TC - 1) / TC;

    if (tid < 2) sMeta[tid] = 0;
    __syncthreads();
    int mxn = 0;
    for (int k = tid; k < K; k += TILED_THREADS) mxn = max(mxn, __float_as_int(cn[k]) & 0x7fffffff);
    atomicMax(&sMeta[0], mxn);
    __syncthreads();
    auto norm_exp = [](float n) { return ((((__float_as_int(n) >> 23) & 0xff) - 127) >> 1) + 1; };  // |c| < 2^e
    const float nmax = __int_as_float(sMeta[0]);
    const int ecm = norm_exp(nmax);
    float S = ldexpf(1.0f, 10 - ecm);
    if (((sMeta[0] >> 23) & 0xff) == 255 || ecm < -20 || ecm > 40) {
        if (tid == 0) sMeta[1] = 1;
    } else {
        for (int k = tid; k < K; k += TILED_THREADS)
            if (cn[k] != 0.f && cn[k] * S * S < float(D)) sMeta[1] = 1;
    }
    __syncthreads();
    const bool shared_scale = sMeta[1] == 0;
    if (!shared_scale) S = 1.0f;
    const float S2 = S * S, inv_s2 = 1.0f / S2;
    auto cscale = [&](float n) {
        const int f = (__float_as_int(n) >> 23) & 0xff;
        return shared_scale ? S : n == 0.f || f == 255 ? 1.0f : ldexpf(1.0f, 10 - norm_exp(n));
    };
    const float xn_lo = shared_scale ? 0.25f * float(D) * inv_s2 : HKM_INF, xn_hi = shared_scale ? 0x1p28f * inv_s2 : 0.f;

    floatx4 pc[NQ];
    float pcn = 0.f;   // |c|^2 of row `tid` of the tile being fetched (threads 0..127)
    auto issue = [&](int ct) {
#pragma unroll
        for (int q = 0; q < NQ; ++q) {
            const int g = tid + TILED_THREADS * q;
            const int r = ct * TC + g / GPR, c = (g % GPR) * 4;
            floatx4 v = {0.f, 0.f, 0.f, 0.f};
            if (r < K) {
                const float* row = C + int64_t(r) * ldc;
                if (FULL) v = ld4_any(row + c);
                else v = load_row4<false>(row, c, D);
            }
            pc[q] = v;
        }
        if (tid < TC) pcn = cn[ct * TC + tid];
    };
    auto stage = [&](int buf, int ct) {
#pragma unroll
        for (int q = 0; q < NQ; ++q) {
            const int g = tid + TILED_THREADS * q;
            const int r = g / GPR, c = (g % GPR) * 4;
            const float s = -2.0f * (shared_scale ? S : cscale(cn[ct * TC + r]));
            _Float16* at = sP[buf] + (r >> 5) * (64 * DP) + (r & 31) * DP + 8 * ((c >> 3) ^ split_swz<DP>(r & 31)) + (c & 4);
#pragma unroll
            for (int t = 0; t < 4; t += 2) {
                const floatx2 v = {pc[q][t] * s, pc[q][t + 1] * s};
                const halfx2 v1 = __builtin_convertvector(v, halfx2);
                const floatx2 w = {fmaf(pc[q][t], s, -float(v1[0])), fmaf(pc[q][t + 1], s, -float(v1[1]))};
                *reinterpret_cast<halfx2*>(at + t) = v1;
                *reinterpret_cast<halfx2*>(at + t + 32 * DP) = __builtin_convertvector(w, halfx2);
            }
        }
        if (tid < TC) {
            sCn[buf][tid] = pcn * S2;
            sI[buf][tid] = S / cscale(pcn);
        }
    };

    const bool fast = ldx < (int64_t(1) << 24);
    const unsigned lane_off = unsigned((int64_t(p) * ldx + h * (DP / 2)) * 4);
    int buf = 0;
    issue(0);
    for (int64_t tile = blockIdx.x; tile < ntiles; tile += gridDim.x) {
        const int64_t row0 = tile * (TILED_THREADS * PB / 2) + wave * (PB * 32);
        floatx4 b[PB][NJ];
        fetch_rows_any<DP, PB, FULL>(X, N, D, ldx, row0, p, h, fast, lane_off, b);
        float xn[PB], m[PB], rx[PB];
        int mi[PB];
        bool in[PB], rest = false;
        halfx8 xh[PB][NS], xl[PB][NS];
        SplitBest best[PB];
#pragma unroll
        for (int pb = 0; pb < PB; ++pb) {
            xn[pb] = row_norm<NJ>(b[pb]);
            in[pb] = (xn[pb] >= xn_lo && xn[pb] <= xn_hi) || (shared_scale && xn[pb] == 0.f);
            rest |= !in[pb];
            split_row<NS>(b[pb], S, xh[pb], xl[pb]);
            split_best_init(best[pb]);
        }
        if (shared_scale) {
            for (int ct = 0; ct < nct; ++ct) {
                stage(buf, ct);
                __syncthreads();
                issue(ct + 1 < nct ? ct + 1 : 0);  // (tile 0 again for the next rows)
                split_scan<DP, PB>(sP[buf], sCn[buf], TCB, ct * TCB, p, h, xh, xl, best);
                buf ^= 1;
            }
        }
        bool near[PB];
#pragma unroll
        for (int pb = 0; pb < PB; ++pb) {
            near[pb] = split_is_near(best[pb], xn[pb] * S2) && in[pb];
            mi[pb] = split_best_index(best[pb]);
            m[pb] = fmaf(best[pb].m, inv_s2, xn[pb]);
        }
        if (__syncthreads_or(rest)) {
            // rows with scales of their own
            floatx16 keep[PB];
            float m1[PB];
            int blk[PB];
            bool odd[PB];
            fetch_rows_any<DP, PB, FULL>(X, N, D, ldx, row0, p, h, fast, lane_off, b);
#pragma unroll
            for (int pb = 0; pb < PB; ++pb) {
                odd[pb] = ((__float_as_int(xn[pb]) >> 23) & 0xff) == 255;
                const float sx = xn[pb] > 0.f && !odd[pb] ? ldexpf(1.0f, 14 - norm_exp(xn[pb])) : 1.0f;
                rx[pb] = S / sx;
                split_row<NS>(b[pb], sx, xh[pb], xl[pb]);
                m1[pb] = HKM_INF;
                blk[pb] = 0;
                keep_undefined(keep[pb]);
            }
            for (int ct = 0; ct < nct; ++ct) {
                stage(buf, ct);
                __syncthreads();
                issue(ct + 1 < nct ? ct + 1 : 0);
                split_scan_own<DP, PB, false>(sP[buf], sCn[buf], sI[buf], TCB, ct * TCB, p, h, xh, xl, rx, inv_s2, xn, m1,
                                              blk, keep);
                buf ^= 1;
            }
#pragma unroll
            for (int pb = 0; pb < PB; ++pb) {
                if (!in[pb]) {
                    m[pb] = fmaf(m1[pb], inv_s2, xn[pb]);
                    mi[pb] = kept_argmin(keep[pb], m1[pb], blk[pb]);
                }
                if (__any(odd[pb])) {
                    float mp;
                    int mip;
                    split_scan_plain<DP>(C, K, ldc, D, h, b[pb], mp, mip);
                    if (odd[pb]) {
                        m[pb] = mp + xn[pb];
                        mi[pb] = mip - 4 * h;  // the lane-half term is added below
                    }
                }
            }
        }
#pragma unroll
        for (int pb = 0; pb < PB; ++pb) {
            m[pb] = fmaxf(m[pb], 0.0f);
            mi[pb] += 4 * h;
            merge_halves(m[pb], mi[pb]);
            const int64_t r = row0 + pb * 32 + p;
            const unsigned long long ties = __ballot(near[pb] && r < N && h == 0);
            if (ties) split_near_rows<DP, true>(ties, X + (row0 + pb * 32) * ldx, ldx, C, K, ldc, D, p, m[pb], mi[pb]);
            if (h == 0 && r < N) {
                labels[r] = mi[pb];
                if (min_d2) min_d2[r] = m[pb];
            }
        }
    }
}

template <int DP, bool FULL>
static int launch_tiled_t(const float* X, int64_t N, int32_t D, int64_t ldx, const float* C, int32_t K, int64_t ldc,
                          const float* cn, int32_t* labels, float* min_d2, hipStream_t st) {
    const int64_t ntiles = (N + TILED_THREADS - 1) / TILED_THREADS;
    int64_t grid = int64_t(num_cus());
    if (grid > ntiles) grid = ntiles;
    prof_begin(st);
    hipLaunchKernelGGL((split_tiled_kernel<DP, FULL>), dim3((unsigned)grid), dim3(TILED_THREADS), 0, st, X, N, D, ldx, C, K, ldc, cn,
                       labels, min_d2, ntiles);
    prof_end(st);
    return check_launch("split_tiled_kernel");
}

int launch_split_tiled(const float* X, int64_t N, int32_t D, int64_t ldx, const float* C, int32_t K, int64_t ldc,
                       const float* cn, int32_t* labels, float* min_d2, hipStream_t st) {
    const int dp = split_dp(D);
#define HKM_CASE(d)                                                                                     \
    case d:                                                                                             \
        return D == d ? launch_tiled_t<d, true>(X, N, D, ldx, C, K, ldc, cn, labels, min_d2, st)        \
                      : launch_tiled_t<d, false>(X, N, D, ldx, C, K, ldc, cn, labels, min_d2, st);
    switch (dp) {
        HKM_CASE(32) HKM_CASE(48) HKM_CASE(64)
        default:
            return fail(HKM_EUNSUPPORTED, "split_tiled: D=%d", D);
    }
#undef HKM_CASE
}

}  // namespace hkm
