// Distance + argmin for rows of more than 128 features and any K, 2-D decomposition, with the cross term on the fp16 matrix cores from operands split into two fp16 parts (the arithmetic
// of hkm_assign_split.hip: three products per 16 features, fp32 sums).
//
// A work item is a tile of 256 points x a tile of 64 CB centroids over all features in chunks of 32; eight waves as a
// 4 x 2 grid, each 64 points x 32 CB centroids per chunk.  Both operand panels are fetched with 16-byte loads two
// chunks ahead by all threads, and scaled and split into their fp16 parts on the way into double-buffered LDS between
// the matrix instructions of the chunk before (16-byte groups permuted by the row: operand reads meet no bank twice).
// Splitting happens per item because a copy of the split centroids in global memory would not fit the callers' scratch.
//
// What bounds it (200 000 rows of 512, K = 1024): the matrix cores 40 % of the cycles, reads and writes of the panels
// in LDS 35 %, the barrier per chunk and the operand reads behind it most of the rest.  Tried: four waves of 128 x 64
// with all registers of a SIMD each (1.31x longer: nothing overlaps within one wave per SIMD), 64 x 128 per wave (the
// accumulators leave no room for the panels in flight: spills, 2.4x longer).
// Assignment alone, fp32 kernel (128 x 128 tiles) -> this one: 200k x 512, K = 1024: 1708 -> 710 us; 200k x 130, 300:
// 335 -> 136; 20k x 512, 100: 91 -> 42; 5000 x 512, 1024: 139 -> 41.
// Measured rms error of min |x - c|^2 against float64 in units of 2^-24 (|x|^2 + |c|^2), blobs: 4.88 -> 2.62 (512
// features), 3.18 -> 1.72 (200), 2.60 -> 1.36 (128); normal rows 1.64 -> 1.24, 1.17 -> 0.82, 1.01 -> 0.79.
//
// Scaling (powers of two, exact): a centroid by its own norm; rows by one S that takes the centroids' average root mean
// square to 8.  A row between 1/16 of that and a norm of 2^15 / S is at least as precise as in fp32 (its parts end at
// 2^-25 / S); if a tile holds a row outside, the item runs again with such rows scaled by their own norm -- the norms
// are known by then -- and the others as before, so a row's result does not depend on its neighbours.  Rows and
// centroids with a norm of inf or NaN take fp32 products on the vector ALU.
//
// The workgroups of one XCD (workgroup b runs on XCD b % 8) work on the same few point tiles at the same time, one
// centroid tile each: a point tile is read from HBM once and served to the others from that XCD's L2.  The per-item
// (min, argmin) of a point are merged across centroid tiles with a 64-bit unsigned atomic min on the key (bits of the
// clamped d2) << 32 | index: for non-negative floats the bit pattern orders like the value, so the smallest distance
// wins and, among equal distances, the smallest index -- an order-independent, hence deterministic, merge.
#include "hkm_common.h"
#include "hkm_mfma_util.h"

namespace hkm {

static constexpr int WIDE_THREADS = 512, WIDE_TP = 256, WIDE_DC = 32;

__global__ void fill_keys_kernel(unsigned long long* __restrict__ keys, int64_t n) {
    for (int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < n;
         i += int64_t(gridDim.x) * blockDim.x)
        keys[i] = ~0ull;
}

__global__ void unpack_keys_kernel(const unsigned long long* __restrict__ keys, int64_t n,
                                   int32_t* __restrict__ labels, float* __restrict__ min_d2) {
    for (int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < n;
         i += int64_t(gridDim.x) * blockDim.x) {
        const unsigned long long k = keys[i];
        const unsigned hi = unsigned(k >> 32);
        // a row whose distances were all infinite never lowered its key: label 0 like the reference's
        // torch.min on such a row
        labels[i] = hi == 0xffffffffu ? 0 : int32_t(unsigned(k));
        if (min_d2) min_d2[i] = __uint_as_float(hi);
    }
}

__device__ __forceinline__ bool wide_odd(float norm) { return ((__float_as_int(norm) >> 23) & 0xff) == 255; }

// 2^(bits - E) with |v_d| < 2^E from the squared norm of v
__device__ __forceinline__ float wide_scale(float norm, int bits) {
    if (norm == 0.f || wide_odd(norm)) return 1.0f;
    const int e = ((((__float_as_int(norm) >> 23) & 0xff) - 127) >> 1) + 1;
    return ldexpf(1.0f, bits - e);
}

// the squared distance as (x.c - |c|^2/2) - |x|^2/2 = -d2/2, clamped there at 0 -- a NaN becomes 0
__device__ __forceinline__ unsigned long long wide_plain_key(float dot, float cn, float xn, int k) {
    const float g = fminf((dot - 0.5f * cn) - 0.5f * xn, 0.0f);
    const float d = -2.0f * g + 0.0f;  // the "+ 0" turns -0.0 into +0.0, whose bit pattern is the smallest key
    return d < HKM_INF ? (static_cast<unsigned long long>(__float_as_uint(d)) << 32) | unsigned(k) : ~0ull;
}

template <int CB>
__global__ __launch_bounds__(WIDE_THREADS) void assign_wide_kernel(
    const float* __restrict__ X, int64_t N, int D, int64_t ldx, const float* __restrict__ C, int K, int64_t ldc,
    const float* __restrict__ cn, unsigned long long* __restrict__ keys, int64_t ntiles, int nct, int ndc) {
    constexpr int WP = WIDE_THREADS / 128, PB = 8 / WP;  // waves along the points, each with PB blocks of 32 of them
    constexpr int TP = WIDE_TP, TC = 64 * CB, DC = WIDE_DC;
    constexpr int SR = WIDE_THREADS / 8, RX = TP / SR, RC = TC / SR, STEPS = 2 * CB;  // staged rows per thread and panel; steps of a chunk
    __shared__ __align__(16) _Float16 sX[2][2][TP * DC];  // [buffer][part]
    __shared__ __align__(16) _Float16 sC[2][2][TC * DC];
    __shared__ float sM[2][TP];
    __shared__ int sI[2][TP];
    __shared__ float sXn[TP], sXs[TP];                          // the tile's |x|^2 and, in a second run, scales
    __shared__ __align__(16) float sCn[TC];                     // |c|^2 (+inf: padding, or not finite)
    __shared__ __align__(16) float sCi[TC];                     // 1 / scale
    __shared__ int sStat[2];
    __shared__ int sOddC;
    const int tid = threadIdx.x;
    const int lane = tid & 63, wave = tid >> 6;
    const int wp = wave & (WP - 1), wc = wave / WP;  // this wave: points [32 PB wp, ...), centroids [32 CB wc, ...)
    const int p = lane & 31, h = lane >> 5;

    // S from the average exponent of the centroids' squared norms
    if (tid < 2) sStat[tid] = 0;
    __syncthreads();
    {
        int es = 0, n = 0;
        for (int k = tid; k < K; k += WIDE_THREADS) {
            const int e = (__float_as_int(cn[k]) >> 23) & 0xff;
            if (e != 0 && e != 255) {
                es += e - 127;
                ++n;
            }
        }
        atomicAdd(&sStat[0], es);
        atomicAdd(&sStat[1], n);
    }
    __syncthreads();
    float S = 1.0f;
    if (sStat[1] > 0) {
        const float lg = 0.5f * (float(sStat[0]) / float(sStat[1]) - log2f(float(D)));
        S = ldexpf(1.0f, 3 - int(rintf(fminf(fmaxf(lg, -50.f), 50.f))));
    }
    const float inv_s2 = 1.0f / (S * S);
    const float xn_lo = 0.25f * float(D) * inv_s2, xn_hi = 0x1p30f * inv_s2;
    auto in_range = [&](float xn) { return (xn >= xn_lo && xn <= xn_hi) || xn == 0.f; };

    // items of this workgroup: the l-th, (l + per XCD)-th, ... of its XCD's point tiles x centroid tiles
    const int xcd = blockIdx.x & 7, nl = gridDim.x >> 3;
    const int64_t nx = xcd < ntiles ? (ntiles - xcd + 7) / 8 : 0;
    if (int64_t(blockIdx.x >> 3) >= nx * nct) return;
    // an item as (point tile, centroid tile) of this XCD; the next item of this workgroup without a division
    struct Item {
        int64_t x;
        int c;
    };
    const int step_x = nl / nct, step_c = nl - step_x * nct;
    auto next_item = [&](Item& i) {
        i.x += step_x;
        i.c += step_c;
        if (i.c >= nct) {
            i.c -= nct;
            ++i.x;
        }
    };
    Item cur;
    cur.x = int(blockIdx.x >> 3) / nct;
    cur.c = int(blockIdx.x >> 3) - int(cur.x) * nct;

    const int sr = tid >> 3;         // staging: rows sr + SR q of both panels
    const int sc = (tid & 7) * 4;    // column group
    floatx4 pa[RC], pb_[RX];         // a chunk on its way to LDS
    float scA[RC], scB[RX];          // scales of the rows being staged
    float ncA[RC];                   // squared norms of the fetched item's centroid rows
    float xsq[RX];                   // |x|^2 of the staged rows over this thread's column group

    // The next chunk to fetch.  Rows beyond K or N are clamped to the last valid row (a padding centroid has
    // |c|^2 = +inf and never wins; a padding point is never stored), column groups to the last one inside the row
    // (tail() moves such a group's elements to their places).
    Item fitem = cur;
    int fdc = 0;
    unsigned offA[RC], offB[RX];
    const char *baseA = nullptr, *baseB = nullptr;
    bool ftail = false, stail = false;  // the chunk being fetched resp. staged is the ragged last one
    const unsigned lda4 = unsigned(ldc) * 4u, ldb4 = unsigned(ldx) * 4u;
    auto fetch_begin = [&]() {
        const bool more = fitem.x < nx;  // (behind the last item: fetched, not used)
        const int64_t x0 = (xcd + 8 * (more ? fitem.x : cur.x)) * TP;
        const int c0 = (more ? fitem.c : cur.c) * TC, d0 = fdc * DC;
        stail = ftail;
        ftail = d0 + DC > D;
        const int back = ftail ? 4 : 0;  // (the group may begin before the chunk)
        baseA = reinterpret_cast<const char*>(C + int64_t(c0) * ldc + d0 - back);
        baseB = reinterpret_cast<const char*>(X + x0 * ldx + d0 - back);
        if (fdc == 0 || ftail) {
            const int lastA = K - 1 - c0, lastB = int(N - 1 - x0 < TP ? N - 1 - x0 : TP);
            const unsigned vcol = unsigned((ftail ? min(sc, D - 4 - d0) : sc) + back) * 4u;
#pragma unroll
            for (int q = 0; q < RX; ++q) offB[q] = unsigned(min(sr + SR * q, lastB)) * ldb4 + vcol;
#pragma unroll
            for (int q = 0; q < RC; ++q) {
                const int r = min(sr + SR * q, lastA);
                offA[q] = unsigned(r) * lda4 + vcol;
                if (fdc == 0) ncA[q] = cn[c0 + r];
            }
        }
        if (++fdc == ndc) {
            fdc = 0;
            next_item(fitem);
        }
    };
    auto fetch_x = [&](int q) { pb_[q] = ld4_any(baseB + offB[q]); };
    auto fetch_c = [&](int q) { pa[q] = ld4_any(baseA + offA[q]); };
    // a group fetched `by` elements ahead of its place; what lies beyond the row becomes 0
    const int by = sc - (D - 4 - (ndc - 1) * DC);
    auto tail = [&](floatx4 v) {
        if (by & 1) v = floatx4{v[1], v[2], v[3], 0.f};
        if (by & 2) v = floatx4{v[2], v[3], 0.f, 0.f};
        if (by >= 4) v = floatx4{0.f, 0.f, 0.f, 0.f};
        return v;
    };
    auto fix_tail = [&]() {
        if (!stail) return;
#pragma unroll
        for (int q = 0; q < RX; ++q) pb_[q] = by > 0 ? tail(pb_[q]) : pb_[q];
#pragma unroll
        for (int q = 0; q < RC; ++q) pa[q] = by > 0 ? tail(pa[q]) : pa[q];
        asm volatile("" ::: "memory");  // a branch: the chunks before it take none of this
    };
    // position of 16-byte group g of a panel row
    auto at = [](int r, int g) { return r * DC + 8 * (g ^ ((r >> 2) & 3)); };
    auto split_store = [&](const floatx4& v, float s, _Float16* hi, _Float16* lo) {
        typedef _Float16 halfx4 __attribute__((ext_vector_type(4)));
        halfx4 a, b;
#pragma unroll
        for (int t = 0; t < 4; t += 2) {
            const floatx2 w = {v[t] * s, v[t + 1] * s};
            const halfx2 w1 = __builtin_convertvector(w, halfx2);
            const floatx2 r = {fmaf(v[t], s, -float(w1[0])), fmaf(v[t + 1], s, -float(w1[1]))};
            const halfx2 w2 = __builtin_convertvector(r, halfx2);
            a[t] = w1[0];
            a[t + 1] = w1[1];
            b[t] = w2[0];
            b[t + 1] = w2[1];
        }
        *reinterpret_cast<halfx4*>(hi) = a;
        *reinterpret_cast<halfx4*>(lo) = b;
    };
    const int w0 = at(sr, sc >> 3) + 4 * (tid & 1);  // (rows 32 or 64 apart permute alike)
    auto stage_x = [&](int b, int q) {
        split_store(pb_[q], scB[q], &sX[b][0][w0 + SR * DC * q], &sX[b][1][w0 + SR * DC * q]);
#pragma unroll
        for (int t = 0; t < 4; ++t) xsq[q] = fmaf(pb_[q][t], pb_[q][t], xsq[q]);
    };
    auto stage_c = [&](int b, int q) {
        split_store(pa[q], scA[q], &sC[b][0][w0 + SR * DC * q], &sC[b][1][w0 + SR * DC * q]);
    };
    // scales of the item whose first chunk is staged next
    auto set_scales = [&](bool own_rows) {
#pragma unroll
        for (int q = 0; q < RX; ++q) {
            scB[q] = own_rows ? sXs[sr + SR * q] : S;
            xsq[q] = 0.f;
        }
#pragma unroll
        for (int q = 0; q < RC; ++q) scA[q] = wide_scale(ncA[q], 12);
    };
    auto stage_first = [&](int b, bool own_rows) {
        fetch_begin();
#pragma unroll
        for (int q = 0; q < RX; ++q) fetch_x(q);
#pragma unroll
        for (int q = 0; q < RC; ++q) fetch_c(q);
        set_scales(own_rows);
        fetch_begin();
        fix_tail();
#pragma unroll
        for (int q = 0; q < RX; ++q) {
            stage_x(b, q);
            fetch_x(q);
        }
#pragma unroll
        for (int q = 0; q < RC; ++q) {
            stage_c(b, q);
            fetch_c(q);
        }
    };

    bool own = false;  // this run of the item uses the rows' own scales where needed
    int dc = 0, buf = 0;
    floatx16 acc[PB][CB];
    auto clear = [&]() {
#pragma unroll
        for (int pb = 0; pb < PB; ++pb)
#pragma unroll
            for (int cb = 0; cb < CB; ++cb)
#pragma unroll
                for (int v = 0; v < 16; ++v) acc[pb][cb][v] = 0.f;
    };
    clear();
    stage_first(0, false);
    const int rX = wp * (32 * PB) + p, rC = wc * (32 * CB) + p;
    const int fX[2] = {at(rX, h), at(rX, 2 + h)}, fC[2] = {at(rC, h), at(rC, 2 + h)};

    while (true) {
        // the accumulators live in accumulation registers from chunk to chunk (left to itself the compiler carries half
        // of them in vector registers and copies them over and back in every chunk)
#pragma unroll
        for (int pb = 0; pb < PB; ++pb)
#pragma unroll
            for (int cb = 0; cb < CB; ++cb) asm volatile("" : "+v"(acc[pb][cb]));
        __syncthreads();
        const bool last = dc == ndc - 1;
        const int c_lo = cur.c * TC;
        float cur_cn = HKM_INF;
        if (last) {
            if (tid < TC && tid < K - c_lo) cur_cn = cn[c_lo + tid];
            if (tid == 0) sOddC = 0;
            // squared norms of the tile's points: the eight threads that staged a row add their parts
#pragma unroll
            for (int q = 0; q < RX; ++q) {
                float v = xsq[q];
                v += __shfl_xor(v, 1);
                v += __shfl_xor(v, 2);
                v += __shfl_xor(v, 4);
                if ((tid & 7) == 0) sXn[sr + SR * q] = v;
            }
            set_scales(false);  // the next item's first chunk is staged below
        }
        // k-step st of the matrix instruction covers features 16 st .. 16 st + 15 of the chunk, 8 per lane-half.  The
        // operands of a step are read one step ahead; the next chunk is split into the other buffer, and the one
        // after it fetched, between the matrix instructions.
        fetch_begin();
        fix_tail();
        const _Float16* bX = &sX[buf][0][0];
        const _Float16* bC = &sC[buf][0][0];
        halfx8 xh[PB], xl[PB], ch[2], cl[2];
        auto read_x = [&](int st) {
#pragma unroll
            for (int pb = 0; pb < PB; ++pb) {
                xh[pb] = *reinterpret_cast<const halfx8*>(bX + fX[st] + pb * 32 * DC);
                xl[pb] = *reinterpret_cast<const halfx8*>(bX + fX[st] + pb * 32 * DC + TP * DC);
            }
        };
        auto read_c = [&](int step) {
            const int st = step / CB, cb = step % CB;
            ch[step & 1] = *reinterpret_cast<const halfx8*>(bC + fC[st] + cb * 32 * DC);
            cl[step & 1] = *reinterpret_cast<const halfx8*>(bC + fC[st] + cb * 32 * DC + TC * DC);
        };
        read_c(0);
        read_x(0);
#pragma unroll
        for (int step = 0; step < STEPS; ++step) {
            const int cb = step % CB;
            if (step == CB) read_x(1);
            if (step + 1 < STEPS) read_c(step + 1);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int pb = 0; pb < PB; ++pb) acc[pb][cb] = MFMA_F16(cl[step & 1], xh[pb], acc[pb][cb]);
#pragma unroll
            for (int q = step * RX / STEPS; q < (step + 1) * RX / STEPS; ++q) {
                stage_x(buf ^ 1, q);
                fetch_x(q);
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int pb = 0; pb < PB; ++pb) acc[pb][cb] = MFMA_F16(ch[step & 1], xl[pb], acc[pb][cb]);
#pragma unroll
            for (int q = step * RC / STEPS; q < (step + 1) * RC / STEPS; ++q) {
                stage_c(buf ^ 1, q);
                fetch_c(q);
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int pb = 0; pb < PB; ++pb) acc[pb][cb] = MFMA_F16(ch[step & 1], xh[pb], acc[pb][cb]);
            __builtin_amdgcn_sched_barrier(0);
        }
        buf ^= 1;
        if (!last) {
            ++dc;
            continue;
        }
        dc = 0;

        // ---- the item is complete ----
        __syncthreads();
        const int64_t x_lo = (xcd + 8 * cur.x) * TP;
        const int64_t left = N - x_lo;
        int out = 0;
        if (tid < TP && tid < left) out = !in_range(sXn[tid]) && !wide_odd(sXn[tid]);
        if (tid < TC) {
            const bool odd = tid < K - c_lo && wide_odd(cur_cn);
            sCn[tid] = odd ? HKM_INF : cur_cn;
            sCi[tid] = -2.0f / (S * wide_scale(cur_cn, 12));
            if (odd) sOddC = 1;
        }
        if (__syncthreads_or(out) && !own) {
            // once more, with scales of their own for the rows that need one
            if (tid < TP) sXs[tid] = in_range(sXn[tid]) || wide_odd(sXn[tid]) ? S : wide_scale(sXn[tid], 14);
            __syncthreads();
            own = true;
            fitem = cur;
            fdc = 0;
            clear();
            stage_first(buf, true);
            continue;
        }
        auto scan = [&](bool clamp, int pb, float xn, float f, float& m, int& mi) {
            m = HKM_INF;
            int blk = 0;
            floatx16 keep;
            keep_undefined(keep);
#pragma unroll
            for (int cb = 0; cb < CB; ++cb) {
                const int kb = wc * (32 * CB) + cb * 32;
                const floatx16 c0 = load_cn16(sCn + kb + 4 * h), ci = load_cn16(sCi + kb + 4 * h);
                floatx16 d;
#pragma unroll
                for (int v = 0; v < 16; ++v) d[v] = fmaf(own ? acc[pb][cb][v] * f : acc[pb][cb][v], ci[v], c0[v]);
                if (clamp) {
#pragma unroll
                    for (int v = 0; v < 16; ++v) d[v] = fmaxf(d[v] + xn, 0.0f);
                }
                block_min_keep(d, cb, m, blk, keep);
            }
            mi = kept_argmin(keep, m, blk) + c_lo + wc * (32 * CB);
        };
#pragma unroll
        for (int pb = 0; pb < PB; ++pb) {
            const int r = rX + pb * 32;
            const float xn = sXn[r], f = own ? S / sXs[r] : 1.0f;
            float m;
            int mi;
            scan(false, pb, xn, f, m, mi);
            m += xn;
            if (__any(m < 0.f)) {
                float m1;
                int mi1;
                scan(true, pb, xn, f, m1, mi1);
                mi = m < 0.f ? mi1 : mi;
                m = m < 0.f ? m1 : m;
            }
            // merge lane halves, then the two waves that cover the same points
            mi += 4 * h;
            merge_halves(m, mi);
            if (h == 0) {
                sM[wc][r] = m;
                sI[wc][r] = mi;
            }
        }
        __syncthreads();
        if (tid < TP && tid < left && !wide_odd(sXn[tid])) {
            float m0 = sM[0][tid];
            int i0 = sI[0][tid];
            const float m1 = sM[1][tid];
            const int i1 = sI[1][tid];
            if (m1 < m0 || (m1 == m0 && i1 < i0)) {
                m0 = m1;
                i0 = i1;
            }
            if (m0 < HKM_INF)
                atomicMin(keys + x_lo + tid, (static_cast<unsigned long long>(__float_as_uint(m0 + 0.0f)) << 32) | unsigned(i0));
        }
        // rows and centroids that are not finite: fp32 products, each pair by itself
        const int kn = min(TC, K - c_lo);
        const bool odd_row = tid < TP && tid < left && wide_odd(sXn[tid]);
        if (__syncthreads_or(odd_row)) {
            for (int r = 0; r < TP && r < left; ++r) {
                if (!wide_odd(sXn[r])) continue;
                const float* x = X + (x_lo + r) * ldx;
                for (int k = tid; k < kn; k += WIDE_THREADS) {
                    const float* c = C + int64_t(c_lo + k) * ldc;
                    float s = 0.f;
                    for (int d = 0; d < D; ++d) s = fmaf(x[d], c[d], s);
                    atomicMin(keys + x_lo + r, wide_plain_key(s, cn[c_lo + k], sXn[r], c_lo + k));
                }
            }
        }
        if (sOddC) {
            for (int k = 0; k < kn; ++k) {
                const float nk = cn[c_lo + k];
                if (!wide_odd(nk)) continue;
                const float* c = C + int64_t(c_lo + k) * ldc;
                if (tid < TP && tid < left && !wide_odd(sXn[tid])) {
                    const float* x = X + (x_lo + tid) * ldx;
                    float s = 0.f;
                    for (int d = 0; d < D; ++d) s = fmaf(x[d], c[d], s);
                    atomicMin(keys + x_lo + tid, wide_plain_key(s, nk, sXn[tid], c_lo + k));
                }
            }
        }
        own = false;
        next_item(cur);
        if (cur.x >= nx) return;
        clear();
    }
}

static unsigned keys_grid(int64_t N) {
    const int64_t g = (N + 255) / 256, cap = int64_t(num_cus()) * 8;
    return unsigned(g < cap ? g : cap);
}

int launch_fill_keys(unsigned long long* keys, int64_t N, hipStream_t st) {
    hipLaunchKernelGGL(fill_keys_kernel, dim3(keys_grid(N)), dim3(256), 0, st, keys, N);
    return check_launch("fill_keys_kernel");
}

int launch_unpack_keys(const unsigned long long* keys, int64_t N, int32_t* labels, float* min_d2, hipStream_t st) {
    hipLaunchKernelGGL(unpack_keys_kernel, dim3(keys_grid(N)), dim3(256), 0, st, keys, N, labels, min_d2);
    return check_launch("unpack_keys_kernel");
}

int launch_assign_wide(const float* X, int64_t N, int32_t D, int64_t ldx, const float* C, int32_t K, int64_t ldc,
                       const float* cn, unsigned long long* keys, int32_t* labels, float* min_d2, hipStream_t st) {
    // per-thread offsets inside a tile are 32-bit byte offsets
    if (ldx >= (int64_t(1) << 22) || ldc >= (int64_t(1) << 22))
        return fail(HKM_EUNSUPPORTED, "assign_mfma_stream: leading dimension of 2^22 elements or more");
    const int64_t ntiles = (N + WIDE_TP - 1) / WIDE_TP;
    const int ndc = (D + WIDE_DC - 1) / WIDE_DC;
    int rc = launch_fill_keys(keys, N, st);
    if (rc) return rc;
    // centroids per tile: the padding of the last tile is work done for nothing, narrower tiles read more operand
    // bytes per product
    const int cb = K <= 64 ? 1 : 2;
    const int nct = (K + 64 * cb - 1) / (64 * cb);
    const int64_t per_xcd = (ntiles + 7) / 8 * nct;
    const int64_t wgs = num_cus() / 8 < 1 ? 1 : num_cus() / 8;
    const unsigned grid = unsigned(8 * (per_xcd < wgs ? per_xcd : wgs));
    prof_begin(st);
#define HKM_WIDE(b)                                                                                                \
    if (cb == b)                                                                                                   \
        hipLaunchKernelGGL(assign_wide_kernel<b>, dim3(grid), dim3(WIDE_THREADS), 0, st, X, N, D, ldx, C, K, ldc,  \
                           cn, keys, ntiles, nct, ndc);
    HKM_WIDE(1) HKM_WIDE(2)
#undef HKM_WIDE
    prof_end(st);
    if ((rc = check_launch("assign_wide_kernel"))) return rc;
    return launch_unpack_keys(keys, N, labels, min_d2, st);
}

}  // namespace hkm
