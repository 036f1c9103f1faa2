// Distance + argmin for rows of more than 128 features and any K (the second part, assign_panel_kernel: 65 to 512 features):
// labels and distances are those of fp32 products in the order of assign_mfma_stream_kernel (hkm_assign_mfma.hip), bit for
// bit; most of the work is done by fp16 products.
//
// First part, three products: rows of more than 512 features, few centroids, small calls (panel_eligible).
//
// assign_wide_kernel finds the nearest centroid with the cross term on the fp16 matrix cores, from operands split into two
// fp16 parts (the arithmetic of hkm_assign_split.hip: three products per 16 features, fp32 sums), and marks the rows that
// have another centroid within wide_limit() of it.  wide_exact_kernel decides those with fp32 products.
//
// A work item is a tile of 256 points x a tile of 64 CB centroids over all features in chunks of 32; eight waves as a
// 4 x 2 grid, each 64 points x 32 CB centroids per chunk.  Both operand panels are fetched with 16-byte loads two
// chunks ahead by all threads, and scaled and split into their fp16 parts on the way into double-buffered LDS between
// the matrix instructions of the chunk before (16-byte groups permuted by the row: operand reads meet no bank twice).
// Splitting happens per item because a copy of the split centroids in global memory would not fit the callers' scratch.
//
// What bounds it (2M rows of 512, K = 1024: 7.6 ms, and 0.1 ms for 2000 tied rows; fp32 products alone 16.4): the matrix
// cores 40 % of the cycles, reads and writes of the panels in LDS 35 %, the barrier per chunk and the operand reads behind
// it most of the rest.  Tried: four waves of 128 x 64 with all registers of a SIMD each (1.31x longer: nothing overlaps
// within one wave per SIMD), 64 x 128 per wave (the accumulators leave no room for the panels in flight: spills, 2.4x
// longer).  Without the tied rows' part the call above took 7.2 ms, and labels of 0.05 % of the rows were other ones.
//
// Scaling (powers of two, exact): a centroid by its own norm; rows by one S that takes the centroids' average root mean
// square to 8.  A row between 1/16 of that and a norm of 2^15 / S is at least as precise as in fp32 (its parts end at
// 2^-25 / S); if a tile holds a row outside, the item runs again with such rows scaled by their own norm -- the norms
// are known by then -- and the others as before, so a row's result does not depend on its neighbours.  Rows with a norm
// of inf or NaN, and all rows where a centroid has one, are marked.
//
// The workgroups of one XCD (workgroup b runs on XCD b % 8) work on the same few point tiles at the same time, one
// centroid tile each: a point tile is read from HBM once and served to the others from that XCD's L2.  The per-item
// (min, argmin) of a point are merged across centroid tiles with a 64-bit unsigned atomic min on a key that orders like
// (distance, index): for non-negative floats the bit pattern orders like the value.
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

// ---- keys of the wide rows: bit 63 set, distance, index << 1, tied ----
// An exact key (WIDE_FOUND clear) is smaller than any other, whatever its distance, so the exact products of a row need
// not wait for its first key to be taken away.
static constexpr unsigned long long WIDE_FOUND = 1ull << 63;
__device__ __forceinline__ unsigned long long wide_key(float d, int k, bool tied) {
    return WIDE_FOUND | (static_cast<unsigned long long>(__float_as_uint(d)) << 32) | (unsigned(k) << 1) | unsigned(tied);
}
__device__ __forceinline__ float wide_key_distance(unsigned long long key) {
    return __uint_as_float(unsigned(key >> 32) & 0x7fffffffu);
}
// mark: the row's entry in `labels` until the last launch: the bits of the smallest distance that was found tied with
// another tile's, 0 if the row is to be decided by exact products in any case.  It counts if it is the row's smallest
// distance in the end (equal centroids far from a row -- empty clusters are all zero -- tie without a consequence).
static constexpr unsigned WIDE_NO_MARK = 0xffffffffu;
__device__ __forceinline__ bool wide_is_tied(unsigned long long key, unsigned mark) {
    return !(key & WIDE_FOUND) || (key & 1) || key == ~0ull || mark <= (unsigned(key >> 32) & 0x7fffffffu);
}

// norms of the centroids by the first `nb` workgroups, no key and no mark for every row by the others
__global__ __launch_bounds__(64) void wide_begin_kernel(const float* __restrict__ C, int K, int D, int64_t ldc,
                                                        float* __restrict__ cn, int kpad, int nb,
                                                        unsigned long long* __restrict__ keys,
                                                        unsigned* __restrict__ marks, int64_t n) {
    if (int(blockIdx.x) < nb) {
        norms_of_rows(C, K, D, ldc, cn, kpad, int(blockIdx.x) * NORM_ROWS);
        return;
    }
    for (int64_t i = int64_t(blockIdx.x - nb) * 64 + threadIdx.x; i < n; i += int64_t(gridDim.x - nb) * 64) {
        keys[i] = ~0ull;
        marks[i] = WIDE_NO_MARK;
    }
}

__device__ __forceinline__ bool wide_odd(float norm) { return ((__float_as_int(norm) >> 23) & 0xff) == 255; }

// 2^(bits - E) with |v_d| < 2^E from the squared norm of v
__device__ __forceinline__ float wide_scale(float norm, int bits) {
    if (norm == 0.f || wide_odd(norm)) return 1.0f;
    const int e = ((((__float_as_int(norm) >> 23) & 0xff) - 127) >> 1) + 1;
    return ldexpf(1.0f, bits - e);
}

// what the rounding of a row's distances is measured in: about 2^-24 (|x|^2 + |c|^2) for a centroid at distance d
__device__ __forceinline__ float wide_unit(float xn, float d) { return 0x1p-24f * fmaf(2.5f, xn, 2.0f * d); }

template <int CB>
__global__ __launch_bounds__(WIDE_THREADS) void assign_wide_kernel(
    const float* __restrict__ X, int64_t N, int D, int64_t ldx, const float* __restrict__ C, int K, int64_t ldc,
    const float* __restrict__ cn, unsigned long long* __restrict__ keys, unsigned* __restrict__ marks, float limit,
    int64_t ntiles, int nct, int ndc) {
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
    __shared__ int sNear[TP];  // distances of the tile within the limit of the row's smallest one
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

    const int probe_gap = nct / nl + 3;
    int probe_in = probe_gap;
    int64_t probe_row = (xcd + 8 * cur.x) * TP;
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
            if (tid < TP) sNear[tid] = 0;
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
        floatx16 keep[PB];  // of the block that holds a lane's smallest distance
        float other[PB];    // smallest distance of the other block
#pragma unroll
        for (int pb = 0; pb < PB; ++pb) {
            const int r = rX + pb * 32;
            const float xn = sXn[r], f = own ? S / sXs[r] : 1.0f;
            float m = HKM_INF;
            int blk = 0;
            other[pb] = HKM_INF;
#pragma unroll
            for (int v = 0; v < 16; ++v) keep[pb][v] = HKM_INF;
#pragma unroll
            for (int cb = 0; cb < CB; ++cb) {
                const int kb = wc * (32 * CB) + cb * 32;
                const floatx16 c0 = load_cn16(sCn + kb + 4 * h), ci = load_cn16(sCi + kb + 4 * h);
                floatx16 d;
#pragma unroll
                for (int v = 0; v < 16; ++v) d[v] = fmaf(own ? acc[pb][cb][v] * f : acc[pb][cb][v], ci[v], c0[v]);
                const float bm = block_min16(d);
                other[pb] = fminf(other[pb], fmaxf(m, bm));
                if (bm < m) {
                    m = bm;
                    blk = cb;
                    keep[pb] = d;
                }
            }
            int mi = kept_argmin(keep[pb], m, blk) + c_lo + wc * (32 * CB) + 4 * h;
            // merge lane halves, then the two waves that cover the same points.  (Several distances at or below 0 are
            // tied, so it does not matter which of them is found here.)
            m = fmaxf(m + xn, 0.0f);
            merge_halves(m, mi);
            if (h == 0) {
                sM[wc][r] = m;
                sI[wc][r] = mi;
            }
        }
        __syncthreads();
        // how many distances lie within the limit of the tile's smallest
#pragma unroll
        for (int pb = 0; pb < PB; ++pb) {
            const int r = rX + pb * 32;
            const float xn = sXn[r];
            const float m = fminf(sM[0][r], sM[1][r]);
            const float top = (m - xn) + limit * wide_unit(xn, m);
            int n = other[pb] <= top ? 1 : 0;
#pragma unroll
            for (int v = 0; v < 16; ++v) n += keep[pb][v] <= top ? 1 : 0;
            if (n) atomicAdd(&sNear[r], n);
        }
        __syncthreads();
        if (tid < TP && tid < left) {
            const float xn = sXn[tid];
            float m0 = sM[0][tid];
            int i0 = sI[0][tid];
            const float m1 = sM[1][tid];
            const int i1 = sI[1][tid];
            if (m1 < m0 || (m1 == m0 && i1 < i0)) {
                m0 = m1;
                i0 = i1;
            }
            const bool tied = sNear[tid] > 1;
            if (wide_odd(xn) || sOddC) {
                atomicMin(marks + x_lo + tid, 0u);
            } else if (m0 < HKM_INF) {
                // Whichever of a row's two nearest centroids comes second meets the other one's key, or that of a
                // centroid between them: no tie is missed, in whatever order the tiles arrive.
                const unsigned long long old = atomicMin(keys + x_lo + tid, wide_key(m0, i0, tied));
                const float od = wide_key_distance(old);
                const float both = fminf(od, m0);
                if (old != ~0ull && fabsf(od - m0) <= limit * wide_unit(xn, both))
                    atomicMin(marks + x_lo + tid, __float_as_uint(both));
            }
        }
        // Where most rows are tied (far from the origin, many equal centroids) the rest of this workgroup's items would be
        // worked off twice: their rows are all marked instead.  Looked at: the rows of an item that the other workgroups
        // have long been done with, too.
        if (--probe_in == 0) {
            bool tied = false;
            if (tid < TP && probe_row + tid < N)
                tied = wide_is_tied(__hip_atomic_load(keys + probe_row + tid, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT),
                                    __hip_atomic_load(marks + probe_row + tid, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
            if (2 * __syncthreads_count(tied) > TP) {
                for (next_item(cur); cur.x < nx; next_item(cur)) {
                    const int64_t r = (xcd + 8 * cur.x) * TP + tid;
                    if (tid < TP && r < N) atomicMin(marks + r, 0u);
                }
                return;
            }
            probe_in = 4 * probe_gap;
            probe_row = x_lo;
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

// ------------------------------------------------------------------------------------------------
// The tied rows, with fp32 products in the order of assign_mfma_stream_kernel (hkm_assign_mfma.hip): chunks of 32
// features, then -|c|^2 / 2 and -|x|^2 / 2.  A workgroup looks through its range of rows, gathers the tied ones and
// multiplies 128 of them at a time -- the last ones of the range, if they are few, 32 at a time -- with its tile of
// 128 centroids.
//
// Two workgroups share a CU: while one waits for its scattered rows or a barrier the other multiplies, and the launches make
// so many.  That takes all 256 registers of a thread: with chunks fetched two and three ahead, not one, a CU held a single
// workgroup (400k x 600, K = 1000, every centroid close to another one: whole call 4.31 ms with two, 5.15 with one; 1M x 256, K = 32: 314
// and 322 us; 1M x 100, K = 1000 by one product: 425 and 445).
// ------------------------------------------------------------------------------------------------
static constexpr int EXACT_TC = 128, EXACT_LD = WIDE_DC + 4, EXACT_SCAN = 1024;  // rows looked at at a time

// WP waves side by side along the points, PB blocks of 32 points each; the others along the centroids
template <int WP, int PB>
__device__ __forceinline__ void wide_exact_tile(const float* __restrict__ X, int D, int64_t ldx,
                                                const float* __restrict__ C, int K, int64_t ldc,
                                                const float* __restrict__ cn, unsigned long long* __restrict__ keys,
                                                int64_t row0, const unsigned* list, int n, int c_lo, int ndc,
                                                float* sA, float* sB) {
    constexpr int TP = 32 * PB * WP, WC = 4 / WP, CB = 4 / WC, RB = TP / 32;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wp = wave % WP, wc = wave / WP;
    const int p = lane & 31, h = lane >> 5;
    const int sr = tid >> 3, sc = (tid & 7) * 4;
    const float* rowA[4];
    const float* rowB[RB];
#pragma unroll
    for (int q = 0; q < 4; ++q) rowA[q] = C + int64_t(min(c_lo + sr + 32 * q, K - 1)) * ldc;
#pragma unroll
    for (int q = 0; q < RB; ++q) rowB[q] = X + (row0 + list[min(sr + 32 * q, n - 1)]) * ldx;
    floatx4 pa[4], pb_[RB];  // the next chunk, on its way
    auto issue = [&](int dc) {
        const int c = dc * WIDE_DC + sc;
        const bool whole = c + 4 <= D;
#pragma unroll
        for (int q = 0; q < 4; ++q) pa[q] = whole ? ld4_any(rowA[q] + c) : load_row4<false>(rowA[q], c, D);
#pragma unroll
        for (int q = 0; q < RB; ++q) pb_[q] = whole ? ld4_any(rowB[q] + c) : load_row4<false>(rowB[q], c, D);
    };
    floatx16 acc[PB][CB];
#pragma unroll
    for (int pb = 0; pb < PB; ++pb)
#pragma unroll
        for (int cb = 0; cb < CB; ++cb)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[pb][cb][v] = 0.f;
    float xsq[RB];
#pragma unroll
    for (int q = 0; q < RB; ++q) xsq[q] = 0.f;
    issue(0);
    for (int dc = 0; dc < ndc; ++dc) {
        float* bufA = sA + (dc & 1) * (EXACT_TC * EXACT_LD);
        float* bufB = sB + (dc & 1) * (128 * EXACT_LD);
#pragma unroll
        for (int q = 0; q < 4; ++q) *reinterpret_cast<floatx4*>(bufA + (sr + 32 * q) * EXACT_LD + sc) = pa[q];
#pragma unroll
        for (int q = 0; q < RB; ++q) {
            *reinterpret_cast<floatx4*>(bufB + (sr + 32 * q) * EXACT_LD + sc) = pb_[q];
#pragma unroll
            for (int t = 0; t < 4; ++t) xsq[q] = fmaf(pb_[q][t], pb_[q][t], xsq[q]);
        }
        __syncthreads();
        if (dc + 1 < ndc) issue(dc + 1);
        floatx4 b[PB][4];
#pragma unroll
        for (int pb = 0; pb < PB; ++pb)
#pragma unroll
            for (int j = 0; j < 4; ++j) b[pb][j] = ld4(bufB + (wp * 32 * PB + pb * 32 + p) * EXACT_LD + h * 16 + 4 * j);
#pragma unroll
        for (int cb = 0; cb < CB; ++cb)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const floatx4 a = ld4(bufA + (wc * 32 * CB + cb * 32 + p) * EXACT_LD + h * 16 + 4 * j);
#pragma unroll
                for (int t = 0; t < 4; ++t)
#pragma unroll
                    for (int pb = 0; pb < PB; ++pb) acc[pb][cb] = MFMA32(a[t], b[pb][j][t], acc[pb][cb]);
            }
    }
    __syncthreads();
    // the panels' memory from here on: |x|^2, and each wave's smallest distances and their indices
    float* sXn = sA;
    float(*sM)[128] = reinterpret_cast<float(*)[128]>(sA + 128);
    int(*sI)[128] = reinterpret_cast<int(*)[128]>(sB);
#pragma unroll
    for (int q = 0; q < RB; ++q) {
        float v = xsq[q];
        v += __shfl_xor(v, 1);
        v += __shfl_xor(v, 2);
        v += __shfl_xor(v, 4);
        if ((tid & 7) == 0) sXn[sr + 32 * q] = v;
    }
    __syncthreads();
#pragma unroll
    for (int pb = 0; pb < PB; ++pb) {
        const int r = wp * 32 * PB + pb * 32 + p;
        const float baug = h ? -0.5f * sXn[r] : 1.0f;
        float m = -HKM_INF;
        int mi = 0;
#pragma unroll
        for (int cb = 0; cb < CB; ++cb) {
            const int kb = c_lo + wc * 32 * CB + cb * 32;
            const float aaug = h ? 1.0f : -0.5f * cn[kb + p];
            // -d2/2, the largest is the nearest; a NaN counts as distance 0
            const floatx16 g16 = MFMA32(aaug, baug, acc[pb][cb]);
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                const float g = fminf(g16[v], 0.0f);
                const bool gt = g > m;
                mi = gt ? kb + 8 * (v >> 2) + (v & 3) : mi;
                m = gt ? g : m;
            }
        }
        mi += 4 * h;
        m = -2.0f * m + 0.0f;  // the "+ 0" turns -0.0 into +0.0, whose bit pattern is the smallest key
        merge_halves(m, mi);
        if (h == 0) {
            sM[wc][r] = m;
            sI[wc][r] = mi;
        }
    }
    __syncthreads();
    if (tid < n) {
        float m = sM[0][tid];
        int mi = sI[0][tid];
#pragma unroll
        for (int w = 1; w < WC; ++w) {
            const float om = sM[w][tid];
            const int oi = sI[w][tid];
            if (om < m || (om == m && oi < mi)) {
                m = om;
                mi = oi;
            }
        }
        if (m < HKM_INF)
            atomicMin(keys + row0 + list[tid], (static_cast<unsigned long long>(__float_as_uint(m)) << 32) | (unsigned(mi) << 1));
    }
    __syncthreads();
}

__global__ __launch_bounds__(256, 2) void wide_exact_kernel(const float* __restrict__ X, int64_t N, int D, int64_t ldx,
                                                            const float* __restrict__ C, int K, int64_t ldc,
                                                            const float* __restrict__ cn,
                                                            unsigned long long* __restrict__ keys,
                                                            const unsigned* __restrict__ marks, int64_t per, int ctiles,
                                                            int ndc) {
    __shared__ __align__(16) float sA[2 * EXACT_TC * EXACT_LD];
    __shared__ __align__(16) float sB[2 * 128 * EXACT_LD];
    __shared__ unsigned list[128 + EXACT_SCAN];  // rows of the range
    __shared__ int found[4];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int range = int(blockIdx.x) / ctiles, c_lo = (int(blockIdx.x) - range * ctiles) * EXACT_TC;
    const int64_t lo = range * per, hi = min(N, lo + per);
    int pending = 0;
    for (int64_t at = lo; at < hi; at += EXACT_SCAN) {
        unsigned long long lanes[EXACT_SCAN / 256];
        int mine = 0;
#pragma unroll
        for (int q = 0; q < EXACT_SCAN / 256; ++q) {
            const int64_t i = at + 256 * q + tid;
            // (another workgroup's exact key in place of the row's own says the same: tied)
            lanes[q] = __ballot(i < hi && wide_is_tied(keys[min(i, hi - 1)], marks[min(i, hi - 1)]));
            mine += __popcll(lanes[q]);
        }
        if (lane == 0) found[wave] = mine;
        __syncthreads();
        int put = pending;
        for (int w = 0; w < 4; ++w) {
            if (w < wave) put += found[w];
            pending += found[w];
        }
#pragma unroll
        for (int q = 0; q < EXACT_SCAN / 256; ++q) {
            if (lanes[q] >> lane & 1) list[put + __popcll(lanes[q] & ((1ull << lane) - 1))] = unsigned(at - lo) + 256 * q + tid;
            put += __popcll(lanes[q]);
        }
        __syncthreads();
        const bool end = at + EXACT_SCAN >= hi;
        while (pending >= 128 || (end && pending > 0)) {
            // from the end of the list: what stays behind stays in place
            const int n = pending > 32 ? min(pending, 128) : pending;
            pending -= n;
            if (n > 32) wide_exact_tile<2, 2>(X, D, ldx, C, K, ldc, cn, keys, lo, list + pending, n, c_lo, ndc, sA, sB);
            else wide_exact_tile<1, 1>(X, D, ldx, C, K, ldc, cn, keys, lo, list + pending, n, c_lo, ndc, sA, sB);
        }
    }
}

__global__ __launch_bounds__(256) void wide_labels_kernel(const unsigned long long* __restrict__ keys, int64_t n,
                                                          int32_t* __restrict__ labels) {
    for (int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += int64_t(gridDim.x) * blockDim.x) {
        const unsigned long long key = keys[i];
        // tied, and no exact key: all distances were infinite
        const bool none = (key & WIDE_FOUND) && wide_is_tied(key, unsigned(labels[i]));
        labels[i] = none ? 0 : int32_t(unsigned(key) >> 1);
    }
}

// Labels and the distances that go with them: for the rows that were not tied the distance to their centroid is computed
// here, as fp32 products give it (the order of wide_exact_tile).  One row per lane; rows and their centroids come through
// LDS in chunks of 32 features, eight lanes to a row, the next chunk on its way while one is added up.  Bound by reading
// the rows once more (1M x 208: 0.2 ms; each lane reading its own row: 0.36).
// PANEL: of assign_panel_kernel (labels are final but for the rows decided by all centroids: PANEL_HARD still, their label and
// distance are in the key, which nothing lowered where all distances are infinite).
template <bool PANEL>
__global__ __launch_bounds__(64) void wide_distances_kernel(const float* __restrict__ X, int64_t n, int D, int64_t ldx,
                                                            const float* __restrict__ C, int64_t ldc,
                                                            const float* __restrict__ cn,
                                                            const unsigned long long* __restrict__ keys,
                                                            int32_t* __restrict__ labels, float* __restrict__ min_d2) {
    __shared__ __align__(16) float sX[64 * EXACT_LD], sC[64 * EXACT_LD];
    const int lane = threadIdx.x;
    const int64_t row0 = int64_t(blockIdx.x) * 64, i = row0 + lane;
    const int lab = PANEL && i < n ? labels[i] : 0;
    const unsigned long long key = i < n && !(PANEL && lab >= 0) ? keys[i] : 0;
    const bool exact = PANEL ? lab < 0 && key != ~0ull : !(key & WIDE_FOUND);
    const bool none = PANEL ? lab < 0 && key == ~0ull : !exact && wide_is_tied(key, unsigned(labels[i]));
    const int k = none || i >= n ? 0 : PANEL && lab >= 0 ? lab : int(unsigned(key) >> 1);
    const int sr = lane >> 3, sc = (lane & 7) * 4;
    const float *x[8], *c[8];
#pragma unroll
    for (int q = 0; q < 8; ++q) {
        x[q] = X + min(row0 + sr + 8 * q, n - 1) * ldx;
        c[q] = C + int64_t(__shfl(k, sr + 8 * q)) * ldc;
    }
    floatx4 xv[8], cv[8];
    auto issue = [&](int col) {
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            xv[q] = col + 4 <= D ? ld4_any(x[q] + col) : load_row4<false>(x[q], col, D);
            cv[q] = col + 4 <= D ? ld4_any(c[q] + col) : load_row4<false>(c[q], col, D);
        }
    };
    issue(sc);
    float dot = 0.f, s[8] = {};
    for (int d = 0; d < D; d += WIDE_DC) {
        __syncthreads();
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            *reinterpret_cast<floatx4*>(sX + (sr + 8 * q) * EXACT_LD + sc) = xv[q];
            *reinterpret_cast<floatx4*>(sC + (sr + 8 * q) * EXACT_LD + sc) = cv[q];
        }
        __syncthreads();
        if (d + WIDE_DC < D) issue(d + WIDE_DC + sc);
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            const floatx4 x0 = ld4(sX + lane * EXACT_LD + 4 * g), x1 = ld4(sX + lane * EXACT_LD + 16 + 4 * g);
            const floatx4 c0 = ld4(sC + lane * EXACT_LD + 4 * g), c1 = ld4(sC + lane * EXACT_LD + 16 + 4 * g);
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                dot = fmaf(c0[t], x0[t], dot);
                dot = fmaf(c1[t], x1[t], dot);
                s[g] = fmaf(x0[t], x0[t], s[g]);
                s[4 + g] = fmaf(x1[t], x1[t], s[4 + g]);
            }
        }
    }
    if (i >= n) return;
    labels[i] = k;
    const float xn = ((s[0] + s[1]) + (s[2] + s[3])) + ((s[4] + s[5]) + (s[6] + s[7]));
    const float g = fminf((dot - 0.5f * cn[k]) - 0.5f * xn, 0.0f);
    min_d2[i] = exact ? __uint_as_float(unsigned(key >> 32)) : none ? __uint_as_float(0xffffffffu) : -2.0f * g + 0.0f;
}

// Distances within this many units (wide_unit) are tied.  The two arithmetics differ by a sum of roundings that grows with
// the square root of the row: the root mean square of the difference of two distances' differences is about 0.35 sqrt(D) units
// on blobs (7.8 at 512 features, 4.9 at 200), so this is more than six times it.
static float wide_limit(int32_t D) { return 4.0f + 2.25f * sqrtf(float(D)); }


// ------------------------------------------------------------------------------------------------
// 65 to 512 features with the centroids as one fp16 panel in global memory: ONE product per feature finds the nearest
// centroid of nearly every row, fp32 products decide the others.
//
// Rows and centroids are moved by the mean mu of a few centroids (a distance does not change) and rounded to fp16.  A
// distance of the rounded points differs from the true one by at most t = |x - x1| + sigma (triangle inequality; sigma: the
// largest |c - c1|; both taken from the values), so with u the smallest squared distance of a row, every
// centroid with u' > (sqrt(u) + 2 t)^2 + t^2 + 2 eta is farther than the nearest one, also in the fp32 products' rounding
// (eta = wide_limit() units).  A row with one centroid below that has its label; a row with two (2 to 6 % of the rows of
// blobs) is decided between them by fp32 chains in the order of assign_mfma_stream_kernel, one lane per pair; a row with
// more, or out of fp16's range, by the fp32 products of all centroids (wide_exact_tile).
//
// A workgroup holds a tile of 128 rows as fp16 in LDS, all features, and goes through all centroids: the panel is laid
// out as the matrix instruction reads it (16 bytes per lane, 1 KB per block of 32 centroids and k-step of 16), so its
// fragments go from L2 straight to registers, four k-steps ahead, and no barrier stands between two centroid blocks.  A
// wave multiplies 32 RB rows by 64 centroids at a time.  Norms take part as five more features (three fp16 parts of
// |c1|^2 against powers of two, and two that put a padding centroid behind every other).
//
// What bounds it: the matrix cores (one product: a third of assign_wide_kernel's), then the rows' way into LDS, which
// only other workgroups' products hide: two workgroups of four waves per CU up to 267 features, one of eight beyond.
// Whole call, three products (65 to 128 features: fp32 products) -> one, by all launches: 2M x 512, K = 1024: 7.6 -> 2.8 ms (products
// 2.46 = 0.85 PFLOP/s, rows by all centroids 0.11, pairs 0.05, the rest 0.02; many first centroids in each of clusters far apart: 8.4
// -> 5.1); 400k x 512, 1024: 1610 -> 675 us; 1M x 200, 300: 785 -> 385; 1M x 100, 1000: 2450 -> 450; 400k x 80, 700: 635 -> 154.
// ------------------------------------------------------------------------------------------------
static constexpr int PANEL_TP = 128, PANEL_SAMPLE = 16, PANEL_ROWS = 4, PANEL_MAX_D = 512, PANEL_MIN_D = 65;
static constexpr int PANEL_SMALL_D = 267;  // a tile of so many features leaves room for another workgroup in the LDS
static constexpr int PANEL_HARD = -1, PANEL_PAIR = -2;  // in place of a label: decided by all centroids, by the two in the key

__host__ __device__ constexpr int panel_steps(int D) { return (D + 5 + 15) / 16; }
// scratch: [0] S, [64 ...] S mu, then sigma^2 of every PANEL_ROWS centroids, then the panel
__host__ __device__ inline size_t panel_head_floats(int D, int K) {
    return (size_t(64 + D) + size_t((K + 63) / 64 * 64) / PANEL_ROWS + 63) / 64 * 64;
}
size_t panel_bytes(int32_t D, int32_t K) {
    return panel_head_floats(D, K) * sizeof(float) + size_t((K + 63) / 64 * 64) * panel_steps(D) * 32;
}
// Where one product pays (four launches, and rows decided afterwards), whatever the rows are.  The price of rows that stay open
// depends on the data: few in blobs, more in noise around converged centroids, a quarter of the rows where many first centroids share
// clusters that lie far apart (centres in +-100, spread 1: "far"), and their fp32 products hardly get cheaper in small calls.
// Times as fast as without one product, blobs and noise; far, over 129 to 4096 centroids --
// 24 million rows x centroids: 70 to 128 features 1.13 to 2.0; 0.89 to 1.35; 140 to 256 0.81 to 1.4; 0.59 to 0.84;
// 48 million: 140 to 256 features 1.30 to 1.7; 0.82 to 1.13; 268 to 512, K >= 500: 1.32 to 1.6; 0.83 to 1.17;
// 64 million: 140 to 256 1.4 to 1.8; 0.92 to 1.15; 267 to 512, K >= 500: 1.44 to 1.9; 0.97 to 1.27, fewer: 1.26 to 1.6; 0.81 to 1.07;
// 127 million: 268 to 512, K of 129 to 300: 1.30 to 1.6; 0.91 to 1.12.
// Up to 128 clusters of more than 128 features, where reading the rows bounds both, large calls lose too: 400k x 300, K = 100:
// blobs 214 and 222, noise 221 and 270, far 233 and 294; 4M x 129, 65: 985 and 737, but far 958 and 1242.
// More than 4096 clusters: off since a call of 65 536 clusters (8192 x 70) ended in a memory fault on the GPU whose cause is open.
bool panel_eligible(int64_t N, int32_t D, int32_t K) {
    const int64_t least = D <= 128 ? 32000000 : D <= 256 || K >= 500 ? 64000000 : 128000000;
    return panel_room(N, D, K) && (D <= 128 || K > 128) && N >= (least + K - 1) / K;
}
// Scratch has room for the fp16 centroids (at most 4 MB) from fewer rows on: hkm_workspace_bytes gives the sizes it gave while
// the line lay there.
bool panel_room(int64_t N, int32_t D, int32_t K) {
    return D >= PANEL_MIN_D && D <= PANEL_MAX_D && K <= 4096 && (D <= 128 || K > 64) && N >= 8000000 / K;
}

// the point operand of the norms' parts, and a norm in those parts (n < 0: a padding centroid)
__device__ __forceinline__ _Float16 panel_unit(int i) {
    return _Float16(i == 0 ? 0x1p15f : i == 1 ? 0x1p4f : i == 2 ? 0x1p-7f : i < 5 ? 0x1p15f : 0.0f);
}
__device__ __forceinline__ _Float16 panel_norm(float n, int i) {
    if (n < 0.f) return _Float16(i < 3 ? 0.f : 65504.0f);
    const _Float16 a = _Float16(n * 0x1p-15f);
    n = fmaf(float(a), -0x1p15f, n);
    const _Float16 b = _Float16(n * 0x1p-4f);
    n = fmaf(float(b), -0x1p4f, n);
    return i == 0 ? a : i == 1 ? b : i == 2 ? _Float16(n * 0x1p7f) : _Float16(0.f);
}

// Norms of the centroids as they are (the first nb workgroups, one wave of each), and the panel (the others, one centroid
// per wave).  Every workgroup takes the mean and the scale from the same sample by itself: one launch less.
__global__ __launch_bounds__(64 * PANEL_ROWS) void panel_begin_kernel(const float* __restrict__ C, int K, int D, int64_t ldc,
                                                                      float* __restrict__ cn, int kpad, int nb,
                                                                      float* __restrict__ head, _Float16* __restrict__ panel,
                                                                      int sig_at) {
    if (int(blockIdx.x) < nb) {
        if (threadIdx.x < 64) norms_of_rows(C, K, D, ldc, cn, kpad, int(blockIdx.x) * NORM_ROWS);
        return;
    }
    __shared__ float sMu[PANEL_MAX_D];
    __shared__ float sDev[PANEL_ROWS], sSig[PANEL_ROWS];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, blk = int(blockIdx.x) - nb;
    const int ns = min(K, PANEL_SAMPLE);
    float dev = 0.f;
    for (int d = tid; d < D; d += 64 * PANEL_ROWS) {
        float v[PANEL_SAMPLE], mean = 0.f;
#pragma unroll
        for (int i = 0; i < PANEL_SAMPLE; ++i) v[i] = i < ns ? C[(int64_t(i) * K / ns) * ldc + d] : 0.f;
#pragma unroll
        for (int i = 0; i < PANEL_SAMPLE; ++i) mean += v[i];
        mean /= float(ns);
#pragma unroll
        for (int i = 0; i < PANEL_SAMPLE; ++i) dev += i < ns ? (v[i] - mean) * (v[i] - mean) : 0.f;
        sMu[d] = mean;
    }
    auto sum = [](float v) {
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) v += __shfl_xor(v, o);
        return v;
    };
    dev = sum(dev);
    if (lane == 0) sDev[wave] = dev;
    __syncthreads();
    dev = 0.f;
#pragma unroll
    for (int w = 0; w < PANEL_ROWS; ++w) dev += sDev[w];
    // S takes the sample's root mean square to 4 .. 8 (a power of two; nothing to go by: 1)
    const float ms = dev / (float(ns) * float(D));
    float S = 1.0f;
    if (ms > 0x1p-80f && ms < 0x1p80f) S = ldexpf(1.0f, 2 - ((((__float_as_int(ms) >> 23) & 0xff) - 127) >> 1));
    if (blk == 0) {
        if (tid == 0) head[0] = S;
        for (int d = tid; d < D; d += 64 * PANEL_ROWS) head[64 + d] = S * sMu[d];
    }
    const int steps = panel_steps(D), whole = D >> 3, groups = 2 * steps;
    const int r = blk * PANEL_ROWS + wave;
    const float* row = C + int64_t(min(r, K - 1)) * ldc;
    float n = 0.f, miss = 0.f, top = 0.f;
    bool zero = true;
    auto convert = [&](int g) {
        halfx8 v = {};
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const int d = 8 * g + e;
            if (r < K && d < D) {
                const float c = row[d], w = fmaf(c, -2.0f * S, 2.0f * S * sMu[d]);
                zero = zero && c == 0.f;
                v[e] = _Float16(w);
                const float q = float(v[e]);
                n = fmaf(q, q, n);
                miss = fmaf(w - q, w - q, miss);
                top = fmaxf(top, fabsf(w));
                if (!(w == w)) top = HKM_INF;
            }
        }
        return v;
    };
    auto place = [&](int g) { return panel + ((int64_t(r >> 5) * steps + (g >> 1)) * 64 + (g & 1) * 32 + (r & 31)) * 8; };
    for (int g = lane; g < whole; g += 64) *reinterpret_cast<halfx8*>(place(g)) = convert(g);
    const int tail = whole + lane;  // at most three groups hold the last features and the norm's parts
    halfx8 t = {};
    if (tail < groups) t = convert(tail);
    n = sum(n);
    miss = sum(miss);
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) top = fmaxf(top, __shfl_xor(top, o));
    // Empty clusters are all zero, and of equal centroids the first wins: the others take no part (with them every row
    // near the origin would be left to the fp32 products).
    bool out = r >= K;
    if (!out && __all(zero)) {
        for (int j0 = 0; j0 < r && !out; j0 += 64) {
            const float* c = C + int64_t(min(j0 + lane, r)) * ldc;
            unsigned long long left = __ballot(j0 + lane < r && c[0] == 0.f && c[D >> 1] == 0.f && c[D - 1] == 0.f);
            while (left && !out) {
                c = C + int64_t(j0 + __ffsll(left) - 1) * ldc;
                left &= left - 1;
                bool z = true;
                for (int d = lane; d < D; d += 64) z = z && c[d] == 0.f;
                out = __all(z);
            }
        }
    }
    n = out ? -1.0f : 0.25f * n;
    if (tail < groups) {
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const int q = 8 * tail + e - D;
            if (q >= 0 && q < 5) t[e] = panel_norm(n, q);
        }
        *reinterpret_cast<halfx8*>(place(tail)) = t;
    }
    // beyond fp16, or not finite: no bound, every row is decided by fp32 products
    if (lane == 0) sSig[wave] = top <= 60000.0f && n < 0x1p30f ? 0.25f * miss : HKM_INF;
    __syncthreads();
    if (tid == 0) {
        float sigma = sSig[0];
#pragma unroll
        for (int w = 1; w < PANEL_ROWS; ++w) sigma = fmaxf(sigma, sSig[w]);
        head[sig_at + blk] = sigma;
    }
}

__device__ __forceinline__ float vmin(float a, float b) {
    float r;
    asm("v_min_f32 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
}
__device__ __forceinline__ float vmax(float a, float b) {
    float r;
    asm("v_max_f32 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
}
__device__ __forceinline__ float vmin3(float a, float b, float c) {
    float r;
    asm("v_min3_f32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
    return r;
}
// smallest and second smallest of the 16 distances of a lane
__device__ __forceinline__ void block_two(floatx16& d, float& m, float& s) {
    // the first read is the compiler's own (it knows how long a read of fresh matrix results has to wait), and the
    // others depend on it
    const float t0 = __builtin_canonicalizef(d[0]);
    asm volatile("" : "+v"(d) : "v"(t0));
    float lo[8], hi[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        lo[i] = vmin(d[2 * i], d[2 * i + 1]);
        hi[i] = vmax(d[2 * i], d[2 * i + 1]);
    }
#pragma unroll
    for (int w = 4; w > 0; w >>= 1)
#pragma unroll
        for (int i = 0; i < w; ++i) {
            const float x = vmax(lo[i], lo[i + w]);
            lo[i] = vmin(lo[i], lo[i + w]);
            hi[i] = vmin3(x, hi[i], hi[i + w]);
        }
    m = lo[0];
    s = hi[0];
}

// NW waves: 4 / RB of them (at most NW) side by side along the rows, the others along the centroids
template <int NW, int RB>
__global__ __launch_bounds__(64 * NW, 2) void assign_panel_kernel(
    const float* __restrict__ X, int64_t N, int D, int64_t ldx, int K, const float* __restrict__ head, int nsig, int sig_at,
    const _Float16* __restrict__ panel, unsigned long long* __restrict__ keys, int32_t* __restrict__ labels, float limit,
    int64_t ntiles) {
    constexpr int TP = PANEL_TP, CB = 2, WR = 4 / RB, WC = NW / WR, TPR = 64 * NW / TP, AHEAD = 4;
    extern __shared__ __align__(16) unsigned char lds_raw[];
    const int steps = panel_steps(D), groups = 2 * steps, stride = groups + 1;  // 16-byte groups of a row, odd: rows spread over the banks
    _Float16* sX = reinterpret_cast<_Float16*>(lds_raw);  // [TP][stride][8]
    float* sMu = reinterpret_cast<float*>(sX + size_t(TP) * stride * 8);  // [groups * 8]
    float* sYn = sMu + groups * 8;                                       // [TP]
    float* sXn = sYn + TP;
    float* sT = sXn + TP;
    float* sM = sT + TP;                               // [WC][TP]
    int* sCand = reinterpret_cast<int*>(sM + WC * TP);  // [2][TP]
    int* sCnt = sCand + 2 * TP;                         // [TP]
    int* sStat = sCnt + TP;                             // [2] (the bits of the largest sigma; later rows of a tile left open, by wave)
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int p = lane & 31, h = lane >> 5;
    const int wr = wave % WR, wc = wave / WR;
    const float S = head[0], S2 = S * S;
    if (tid < 2) sStat[tid] = 0;
    for (int d = tid; d < groups * 8; d += 64 * NW) sMu[d] = d < D ? head[64 + d] : 0.f;
    __syncthreads();
    {
        int mx = 0;
        for (int i = tid; i < nsig; i += 64 * NW) mx = max(mx, __float_as_int(head[sig_at + i]));
        atomicMax(&sStat[0], mx);
    }
    __syncthreads();
    // what subnormal parts and the rounding of the moved values miss is in the second term
    const float sigma = fmaf(sqrtf(__int_as_float(sStat[0])), 0x1.01p0f, 0x1p-14f * sqrtf(float(D)));
    const int ngroups = (K + 63) / 64;
    const int sr = tid / TPR, sq = tid % TPR;
    int heat = 0, skip = 0;  // tiles in a row that were no use; tiles to be left out

    for (int64_t tile = blockIdx.x; tile < ntiles; tile += gridDim.x) {
        const int64_t row0 = tile * TP;
        if (skip > 0) {
            --skip;
            if (skip == 0) heat = 2;
            if (tid < TP && row0 + tid < N) {
                labels[row0 + tid] = PANEL_HARD;
                keys[row0 + tid] = ~0ull;
            }
            continue;
        }
        // ---- the rows into LDS ----
        {
            const int64_t r = min(row0 + sr, N - 1);
            const float* row = X + r * ldx;
            float yn = 0.f, xn = 0.f, miss = 0.f;
            _Float16* dst = sX + size_t(sr) * stride * 8;
            const int whole = D >> 3;
            auto put = [&](int g, const floatx4& a, const floatx4& b) {
                const floatx4 m0 = ld4(sMu + 8 * g), m1 = ld4(sMu + 8 * g + 4);
                halfx8 o;
#pragma unroll
                for (int q = 0; q < 8; q += 2) {
                    const floatx4& v = q < 4 ? a : b;
                    const floatx4& m = q < 4 ? m0 : m1;
                    const floatx2 w = {fmaf(v[q & 3], S, -m[q & 3]), fmaf(v[(q & 3) + 1], S, -m[(q & 3) + 1])};
                    const halfx2 w1 = __builtin_convertvector(w, halfx2);
                    const float r0 = w[0] - float(w1[0]), r1 = w[1] - float(w1[1]);
                    yn = __builtin_amdgcn_fdot2(w1, w1, yn, false);
                    miss = fmaf(r0, r0, miss);
                    miss = fmaf(r1, r1, miss);
                    xn = fmaf(v[q & 3], v[q & 3], xn);
                    xn = fmaf(v[(q & 3) + 1], v[(q & 3) + 1], xn);
                    o[q] = w1[0];
                    o[q + 1] = w1[1];
                }
                return o;
            };
            constexpr int U = 4;
            int g = sq;
            for (; g + (U - 1) * TPR < whole; g += U * TPR) {
                floatx4 a[U], b[U];
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    a[u] = ld4_any(row + 8 * (g + u * TPR));
                    b[u] = ld4_any(row + 8 * (g + u * TPR) + 4);
                }
#pragma unroll
                for (int u = 0; u < U; ++u) *reinterpret_cast<halfx8*>(dst + 8 * (g + u * TPR)) = put(g + u * TPR, a[u], b[u]);
            }
            for (; g < groups; g += TPR) {
                floatx4 a = {0.f, 0.f, 0.f, 0.f}, b = a;
                if (g < whole) {
                    a = ld4_any(row + 8 * g);
                    b = ld4_any(row + 8 * g + 4);
                } else {
                    a = load_row4<false>(row, 8 * g, D);
                    b = load_row4<false>(row, 8 * g + 4, D);
                }
                halfx8 o = put(g, a, b);
#pragma unroll
                for (int e = 0; e < 8; ++e)
                    if (8 * g + e >= D) o[e] = panel_unit(8 * g + e - D);
                *reinterpret_cast<halfx8*>(dst + 8 * g) = o;
            }
#pragma unroll
            for (int o = 1; o < TPR; o <<= 1) {
                yn += __shfl_xor(yn, o);
                xn += __shfl_xor(xn, o);
                miss += __shfl_xor(miss, o);
            }
            if (sq == 0) {
                sYn[sr] = yn;
                sXn[sr] = xn;
                // what rounding moves the row and a centroid by, at most
                sT[sr] = fmaf(sqrtf(miss), 0x1.01p0f, fmaf(sqrtf(yn), 0x1p-22f, sigma));
                sCnt[sr] = 0;
            }
        }
        __syncthreads();

        // ---- all centroids ----
        float m[RB], m2[RB];
        int mi[RB];
#pragma unroll
        for (int rb = 0; rb < RB; ++rb) {
            m[rb] = HKM_INF;
            m2[rb] = HKM_INF;
            mi[rb] = 0;
        }
        const _Float16* bp[RB];
#pragma unroll
        for (int rb = 0; rb < RB; ++rb) bp[rb] = sX + size_t((wr * RB + rb) * 32 + p) * stride * 8 + 8 * h;
        for (int g = wc; g < ngroups; g += WC) {
            const _Float16* ap = panel + (int64_t(2 * g) * steps * 64 + lane) * 8;
            halfx8 a[AHEAD][CB], b[2][RB];
            auto load_a = [&](int st, halfx8 (&dst)[CB]) {
                const int s = min(st, steps - 1);  // (behind the last step that one again: read, not used)
#pragma unroll
                for (int cb = 0; cb < CB; ++cb) dst[cb] = *reinterpret_cast<const halfx8*>(ap + (int64_t(cb) * steps + s) * 512);
            };
            auto load_b = [&](int st, halfx8 (&dst)[RB]) {
                const int s = min(st, steps - 1);
#pragma unroll
                for (int rb = 0; rb < RB; ++rb) dst[rb] = *reinterpret_cast<const halfx8*>(bp[rb] + 16 * s);
            };
            floatx16 acc[RB][CB];
#pragma unroll
            for (int rb = 0; rb < RB; ++rb)
#pragma unroll
                for (int cb = 0; cb < CB; ++cb)
#pragma unroll
                    for (int v = 0; v < 16; ++v) acc[rb][cb][v] = 0.f;
#pragma unroll
            for (int j = 0; j < AHEAD; ++j) load_a(j, a[j]);
            load_b(0, b[0]);
            auto step = [&](int st, int j) {
                load_b(st + 1, b[(j + 1) & 1]);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int cb = 0; cb < CB; ++cb)
#pragma unroll
                    for (int rb = 0; rb < RB; ++rb) acc[rb][cb] = MFMA_F16(a[j][cb], b[j & 1][rb], acc[rb][cb]);
                load_a(st + AHEAD, a[j]);
                __builtin_amdgcn_sched_barrier(0);
            };
            int st = 0;
#pragma unroll 1
            for (; st + AHEAD <= steps; st += AHEAD) {
#pragma unroll
                for (int j = 0; j < AHEAD; ++j) step(st + j, j);
            }
#pragma unroll
            for (int j = 0; j < AHEAD - 1; ++j)
                if (st + j < steps) step(st + j, j);
#pragma unroll
            for (int rb = 0; rb < RB; ++rb)
#pragma unroll
                for (int cb = 0; cb < CB; ++cb) {
                    float bm, bs;
                    block_two(acc[rb][cb], bm, bs);
                    const bool up = bm < m[rb];
                    m2[rb] = up ? fminf(m[rb], bs) : fminf(m2[rb], bm);
                    if (up) {
                        mi[rb] = (2 * g + cb) * 32 + block_pos16(acc[rb][cb], bm);
                        m[rb] = bm;
                    }
                }
        }

        // ---- the rows' smallest distances, and who is near them ----
#pragma unroll
        for (int rb = 0; rb < RB; ++rb) {
            const float o = fminf(m[rb], __shfl_xor(m[rb], 32));
            if (h == 0) sM[wc * TP + (wr * RB + rb) * 32 + p] = o;
        }
        __syncthreads();
#pragma unroll
        for (int rb = 0; rb < RB; ++rb) {
            const int r = (wr * RB + rb) * 32 + p;
            float all = sM[r];
#pragma unroll
            for (int w = 1; w < WC; ++w) all = fminf(all, sM[w * TP + r]);
            const float yn = sYn[r], u = fmaxf(all + yn, 0.f);
            const float t = sT[r];
            const float eta = 0x1p-24f * limit * (2.5f * (S2 * sXn[r] + yn) + 2.0f * u);
            const float lim = all + (4.0f * t * __builtin_amdgcn_sqrtf(u) + 7.0f * t * t + 4.0f * eta);
            if (m[rb] <= lim) {
                const int at = atomicAdd(&sCnt[r], m2[rb] <= lim ? 64 : 1);
                if (at < 2) sCand[at * TP + r] = mi[rb] + 4 * h;
            }
        }
        __syncthreads();
        bool hard = false;
        if (tid < TP && row0 + tid < N) {
            int t = tid;
            asm("" : "+v"(t));  // (its address in LDS is not kept from tile to tile: it was spilled)
            const int cnt = sCnt[t], c0 = sCand[t], c1 = sCand[TP + t];
            const bool in = sYn[t] <= 0x1p28f;  // (not so for NaN)
            int lab = PANEL_HARD;
            const bool in0 = unsigned(c0) < unsigned(K), in1 = unsigned(c1) < unsigned(K);
            if (in && cnt == 1 && in0) lab = c0;
            if (in && cnt == 2 && in0 && in1) {
                lab = PANEL_PAIR;
                keys[row0 + tid] = static_cast<unsigned long long>(unsigned(max(c0, c1))) << 32 | unsigned(min(c0, c1));
            }
            if (lab == PANEL_HARD) {
                keys[row0 + tid] = ~0ull;
                hard = true;
            }
            labels[row0 + tid] = lab;
        }
        // Where most rows are left to the fp32 products (many equal centroids, far from any mean), looking first is waste:
        // after three such tiles in a row the next 29 are left out.
        // (Counted here: __syncthreads_count has two barriers more and keeps a register that was spilled.)
        const unsigned long long open = __ballot(hard);
        if (lane == 0 && wave < TP / 64) sStat[wave] = __popcll(open);
        __syncthreads();
        heat = 2 * (sStat[0] + sStat[1]) > TP ? heat + 1 : 0;
        if (heat >= 3) skip = 29;
    }
}

// The rows to be decided by all centroids: as wide_exact_kernel, which looks for its rows in the keys.
__global__ __launch_bounds__(256, 2) void panel_exact_kernel(const float* __restrict__ X, int64_t N, int D, int64_t ldx,
                                                             const float* __restrict__ C, int K, int64_t ldc,
                                                             const float* __restrict__ cn,
                                                             unsigned long long* __restrict__ keys,
                                                             const int32_t* __restrict__ labels, int64_t per, int ctiles, int ndc) {
    __shared__ __align__(16) float sA[2 * EXACT_TC * EXACT_LD];
    __shared__ __align__(16) float sB[2 * 128 * EXACT_LD];
    __shared__ unsigned list[128 + EXACT_SCAN];  // rows of the range
    __shared__ int found[4];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int range = int(blockIdx.x) / ctiles, c_lo = (int(blockIdx.x) - range * ctiles) * EXACT_TC;
    const int64_t lo = range * per, hi = min(N, lo + per);
    int next[EXACT_SCAN / 256];  // the labels looked at next
#pragma unroll
    for (int q = 0; q < EXACT_SCAN / 256; ++q) next[q] = lo + 256 * q + tid < hi ? labels[lo + 256 * q + tid] : 0;
    int pending = 0;
    for (int64_t at = lo; at < hi; at += EXACT_SCAN) {
        unsigned long long lanes[EXACT_SCAN / 256];
        int mine = 0;
#pragma unroll
        for (int q = 0; q < EXACT_SCAN / 256; ++q) {
            const int64_t i = at + EXACT_SCAN + 256 * q + tid;
            lanes[q] = __ballot(next[q] == PANEL_HARD);
            mine += __popcll(lanes[q]);
            next[q] = i < hi ? labels[i] : 0;
        }
        const bool end = at + EXACT_SCAN >= hi;
        if (!__syncthreads_or(mine) && !(end && pending > 0)) continue;
        if (lane == 0) found[wave] = mine;
        __syncthreads();
        int put = pending;
        for (int w = 0; w < 4; ++w) {
            if (w < wave) put += found[w];
            pending += found[w];
        }
#pragma unroll
        for (int q = 0; q < EXACT_SCAN / 256; ++q) {
            if (lanes[q] >> lane & 1) list[put + __popcll(lanes[q] & ((1ull << lane) - 1))] = unsigned(at - lo) + 256 * q + tid;
            put += __popcll(lanes[q]);
        }
        __syncthreads();
        while (pending >= 128 || (end && pending > 0)) {
            // from the end of the list: what stays behind stays in place
            const int n = pending > 32 ? min(pending, 128) : pending;
            pending -= n;
            if (n > 32) wide_exact_tile<2, 2>(X, D, ldx, C, K, ldc, cn, keys, lo, list + pending, n, c_lo, ndc, sA, sB);
            else wide_exact_tile<1, 1>(X, D, ldx, C, K, ldc, cn, keys, lo, list + pending, n, c_lo, ndc, sA, sB);
        }
    }
}

// The labels that are still missing: of two centroids by one chain each, or by the keys of panel_exact_kernel (not if
// wide_distances_kernel follows, which takes label and distance from there).  One wave
// looks through PANEL_LOOK rows and decides 32 pairs at a time, two lanes each; rows and centroids come through LDS in chunks
// of 32 features, eight lanes to a row, two chunks ahead.  Bound by the way of scattered rows from memory: small workgroups,
// eight on a CU (as a part of panel_exact_kernel: 2M x 512, K = 1024, 5 % pairs: 260 us, 140 here).
static constexpr int PANEL_LOOK = 512;
__global__ __launch_bounds__(64) void panel_finish_kernel(const float* __restrict__ X, int64_t N, int D, int64_t ldx,
                                                          const float* __restrict__ C, int64_t ldc, const float* __restrict__ cn,
                                                          const unsigned long long* __restrict__ keys,
                                                          int32_t* __restrict__ labels, bool distances_follow) {
    __shared__ __align__(16) float sXr[32 * EXACT_LD], sCr[64 * EXACT_LD];
    __shared__ unsigned short list[PANEL_LOOK];
    const int lane = threadIdx.x;
    const int64_t lo = int64_t(blockIdx.x) * PANEL_LOOK;
    int lab[PANEL_LOOK / 64];
#pragma unroll
    for (int q = 0; q < PANEL_LOOK / 64; ++q) lab[q] = lo + 64 * q + lane < N ? labels[lo + 64 * q + lane] : 0;
    int pairs = 0;
#pragma unroll
    for (int q = 0; q < PANEL_LOOK / 64; ++q) {
        const int64_t i = lo + 64 * q + lane;
        if (lab[q] == PANEL_HARD && !distances_follow) labels[i] = keys[i] == ~0ull ? 0 : int32_t(unsigned(keys[i]) >> 1);
        const unsigned long long two = __ballot(lab[q] == PANEL_PAIR);
        if (two >> lane & 1) list[pairs + __popcll(two & ((1ull << lane) - 1))] = static_cast<unsigned short>(64 * q + lane);
        pairs += __popcll(two);
    }
    wave_lds_sync();
    for (int first = 0; first < pairs; first += 32) {
        const int n = min(32, pairs - first);
        const int pr = lane >> 1;
        const int64_t r = lo + list[first + min(pr, n - 1)];
        const unsigned long long key = keys[r];
        const int k = int(lane & 1 ? unsigned(key >> 32) : unsigned(key));
        const int sr = lane >> 3, sc = (lane & 7) * 4;
        const float *x[4], *c[8];
#pragma unroll
        for (int q = 0; q < 4; ++q) x[q] = X + (lo + list[first + min(sr + 8 * q, n - 1)]) * ldx;
#pragma unroll
        for (int q = 0; q < 8; ++q) c[q] = C + int64_t(__shfl(k, sr + 8 * q)) * ldc;
        floatx4 xv[2][4], cv[2][8];  // chunks on their way, two ahead
        auto issue = [&](int col, floatx4 (&xd)[4], floatx4 (&cd)[8]) {
#pragma unroll
            for (int q = 0; q < 4; ++q) xd[q] = col + 4 <= D ? ld4_any(x[q] + col) : load_row4<false>(x[q], col, D);
#pragma unroll
            for (int q = 0; q < 8; ++q) cd[q] = col + 4 <= D ? ld4_any(c[q] + col) : load_row4<false>(c[q], col, D);
        };
        issue(sc, xv[0], cv[0]);
        issue(WIDE_DC + sc, xv[1], cv[1]);
        float dot = 0.f, s[8] = {};
        for (int d0 = 0; d0 < D; d0 += 2 * WIDE_DC) {
#pragma unroll
            for (int half = 0; half < 2; ++half) {
                const int d = d0 + half * WIDE_DC;
                if (d >= D) break;
                wave_lds_sync();
#pragma unroll
                for (int q = 0; q < 4; ++q) *reinterpret_cast<floatx4*>(sXr + (sr + 8 * q) * EXACT_LD + sc) = xv[half][q];
#pragma unroll
                for (int q = 0; q < 8; ++q) *reinterpret_cast<floatx4*>(sCr + (sr + 8 * q) * EXACT_LD + sc) = cv[half][q];
                wave_lds_sync();
                issue(d + 2 * WIDE_DC + sc, xv[half], cv[half]);  // (behind the row: nothing is read)
#pragma unroll
                for (int g = 0; g < 4; ++g) {
                    const floatx4 x0 = ld4(sXr + pr * EXACT_LD + 4 * g), x1 = ld4(sXr + pr * EXACT_LD + 16 + 4 * g);
                    const floatx4 c0 = ld4(sCr + lane * EXACT_LD + 4 * g), c1 = ld4(sCr + lane * EXACT_LD + 16 + 4 * g);
#pragma unroll
                    for (int t = 0; t < 4; ++t) {
                        dot = fmaf(c0[t], x0[t], dot);
                        dot = fmaf(c1[t], x1[t], dot);
                        s[g] = fmaf(x0[t], x0[t], s[g]);
                        s[4 + g] = fmaf(x1[t], x1[t], s[4 + g]);
                    }
                }
            }
        }
        const float xn = ((s[0] + s[1]) + (s[2] + s[3])) + ((s[4] + s[5]) + (s[6] + s[7]));
        const float g = fminf((dot - 0.5f * cn[k]) - 0.5f * xn, 0.0f), other = __shfl_xor(g, 1);
        // -d2/2: the larger one is nearer; the even lane has the lower index
        if ((lane & 1) == 0 && pr < n) labels[r] = other > g ? int(unsigned(key >> 32)) : k;
    }
}

template <int NW, int RB>
static int launch_panel_t(const float* X, int64_t N, int32_t D, int64_t ldx, int32_t K, const float* head, int nsig, int sig_at,
                          const _Float16* panel, unsigned long long* keys, int32_t* labels, hipStream_t st) {
    constexpr int WC = NW / (4 / RB);
    const int groups = 2 * panel_steps(D);
    const size_t lds = size_t(PANEL_TP) * (groups + 1) * 16 + (size_t(groups) * 8 + PANEL_TP * (3 + WC) + 3 * PANEL_TP + 2) * 4;
    auto kern = assign_panel_kernel<NW, RB>;
    if (lds > 64 * 1024) {
        hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, int(lds));
        if (e != hipSuccess) return fail(HKM_EHIP, "hipFuncSetAttribute: %s", hipGetErrorString(e));
    }
    const int64_t ntiles = (N + PANEL_TP - 1) / PANEL_TP;
    const int64_t wgs = int64_t(num_cus()) * (NW == 4 ? 2 : 1);
    prof_begin(st);
    hipLaunchKernelGGL(kern, dim3(unsigned(ntiles < wgs ? ntiles : wgs)), dim3(64 * NW), lds, st, X, N, D, ldx, K, head, nsig, sig_at,
                       panel, keys, labels, wide_limit(D), ntiles);
    prof_end(st);
    return check_launch("assign_panel_kernel");
}

int launch_assign_panel(const float* X, int64_t N, int32_t D, int64_t ldx, const float* C, int32_t K, int64_t ldc, float* cn,
                        unsigned long long* keys, void* scratch, int32_t* labels, float* min_d2, hipStream_t st) {
    if (ldx >= (int64_t(1) << 22) || ldc >= (int64_t(1) << 22))  // as the kernels it stands in for
        return fail(HKM_EUNSUPPORTED, "assign_mfma_stream: leading dimension of 2^22 elements or more");
    const int kpad = (K + 127) / 128 * 128, nb = kpad / NORM_ROWS, kp = (K + 63) / 64 * 64, nsig = kp / PANEL_ROWS;
    const int sig_at = 64 + D, ndc = (D + WIDE_DC - 1) / WIDE_DC;
    float* head = static_cast<float*>(scratch);
    _Float16* panel = reinterpret_cast<_Float16*>(head + panel_head_floats(D, K));
    hipLaunchKernelGGL(panel_begin_kernel, dim3(unsigned(nb + nsig)), dim3(64 * PANEL_ROWS), 0, st, C, K, D, ldc, cn, kpad, nb, head, panel, sig_at);
    int rc = check_launch("panel_begin_kernel");
    if (rc) return rc;
    // Waves along the centroids in tiles of 64, as many as there are; those left over divide the rows, which costs operand
    // reads (RB rows blocks share a panel fragment).
    const int tiles = kp / 64;
#define HKM_PANEL(nw, rb) rc = launch_panel_t<nw, rb>(X, N, D, ldx, K, head, nsig, sig_at, panel, keys, labels, st)
    if (D <= PANEL_SMALL_D) {
        if (tiles == 1) HKM_PANEL(4, 1);
        else if (tiles == 2 || tiles == 5 || tiles == 6) HKM_PANEL(4, 2);
        else HKM_PANEL(4, 4);
    } else {
        if (tiles <= 2) HKM_PANEL(8, 1);
        else if (tiles <= 4 || (tiles > 8 && tiles <= 12)) HKM_PANEL(8, 2);
        else HKM_PANEL(8, 4);
    }
#undef HKM_PANEL
    if (rc) return rc;
    // ranges of rows: with the tiles of centroids the two workgroups that a CU holds, 64 rows or more each
    const int ctiles = (K + EXACT_TC - 1) / EXACT_TC;
    int64_t ranges = int64_t(num_cus()) * 2 / ctiles;
    if (ranges > (N + 63) / 64) ranges = (N + 63) / 64;
    if (ranges < (N >> 30) + 1) ranges = (N >> 30) + 1;  // (row numbers inside a range are 32-bit)
    hipLaunchKernelGGL(panel_exact_kernel, dim3(unsigned(ranges * ctiles)), dim3(256), 0, st, X, N, D, ldx, C, K, ldc, cn, keys,
                       labels, (N + ranges - 1) / ranges, ctiles, ndc);
    if ((rc = check_launch("panel_exact_kernel"))) return rc;
    hipLaunchKernelGGL(panel_finish_kernel, dim3(unsigned((N + PANEL_LOOK - 1) / PANEL_LOOK)), dim3(64), 0, st, X, N, D, ldx, C, ldc,
                       cn, keys, labels, min_d2 != nullptr);
    if ((rc = check_launch("panel_finish_kernel")) || !min_d2) return rc;
    hipLaunchKernelGGL(wide_distances_kernel<true>, dim3(unsigned((N + 63) / 64)), dim3(64), 0, st, X, N, D, ldx, C, ldc, cn, keys,
                       labels, min_d2);
    return check_launch("wide_distances_kernel");
}

int launch_assign_wide(const float* X, int64_t N, int32_t D, int64_t ldx, const float* C, int32_t K, int64_t ldc,
                       float* cn, unsigned long long* keys, int32_t* labels, float* min_d2, hipStream_t st) {
    // per-thread offsets inside a tile are 32-bit byte offsets
    if (ldx >= (int64_t(1) << 22) || ldc >= (int64_t(1) << 22))
        return fail(HKM_EUNSUPPORTED, "assign_mfma_stream: leading dimension of 2^22 elements or more");
    const int64_t ntiles = (N + WIDE_TP - 1) / WIDE_TP;
    const int ndc = (D + WIDE_DC - 1) / WIDE_DC;
    const int kpad = (K + 127) / 128 * 128, nb = kpad / NORM_ROWS;
    const int64_t fill = (N + 255) / 256, fcap = int64_t(num_cus()) * 16;
    unsigned* marks = reinterpret_cast<unsigned*>(labels);
    hipLaunchKernelGGL(wide_begin_kernel, dim3(unsigned(nb + (fill < fcap ? fill : fcap))), dim3(64), 0, st, C, K, D, ldc, cn,
                       kpad, nb, keys, marks, N);
    int rc = check_launch("wide_begin_kernel");
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
                           cn, keys, marks, wide_limit(D), ntiles, nct, ndc);
    HKM_WIDE(1) HKM_WIDE(2)
#undef HKM_WIDE
    prof_end(st);
    if ((rc = check_launch("assign_wide_kernel"))) return rc;
    // ranges of rows: with the tiles of centroids the two workgroups that a CU holds, 64 rows or more each
    const int ctiles = (K + EXACT_TC - 1) / EXACT_TC;
    int64_t ranges = int64_t(num_cus()) * 2 / ctiles;
    if (ranges > (N + 63) / 64) ranges = (N + 63) / 64;
    if (ranges < (N >> 30) + 1) ranges = (N >> 30) + 1;  // (row numbers inside a range are 32-bit)
    hipLaunchKernelGGL(wide_exact_kernel, dim3(unsigned(ranges * ctiles)), dim3(256), 0, st, X, N, D, ldx, C, K, ldc, cn,
                       keys, marks, (N + ranges - 1) / ranges, ctiles, ndc);
    if ((rc = check_launch("wide_exact_kernel"))) return rc;
    if (!min_d2) {
        hipLaunchKernelGGL(wide_labels_kernel, dim3(keys_grid(N)), dim3(256), 0, st, keys, N, labels);
        return check_launch("wide_labels_kernel");
    }
    hipLaunchKernelGGL(wide_distances_kernel<false>, dim3(unsigned((N + 63) / 64)), dim3(64), 0, st, X, N, D, ldx, C, ldc, cn, keys,
                       labels, min_d2);
    return check_launch("wide_distances_kernel");
}

}  // namespace hkm
