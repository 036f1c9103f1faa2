// The update, and the whole step, of few clusters of float64 rows: per-cluster sums as a product of matrices on the fp64 matrix cores.
//
// S = P X with P[k][row] = 1 where the row's label is k: v_mfma_f64_16x16x4 takes 16 clusters, 4 rows and 16 columns at a
// time, every product is exact and every sum has a fixed order -- a wave's rows in ascending order, then the waves of a
// workgroup, then the workgroups -- so the means depend on the labels and rows alone.  A column of ones counts the rows.
//
// What it replaces for these shapes: a stable counting sort of the rows and segmented sums, seven launches of which three
// pass over memory.  Bound by reading the rows once: 1M x 18, K = 16: 77 us in seven launches -> 47 in three (36 of them
// here, 4.0 TB/s); ten iterations of the fit 1.33 -> 1.02 ms.
//
// 0 x inf is NaN, so values that are not finite do not take part in the product: they enter as 0 and leave a mark (+inf,
// -inf or NaN) with their cluster and column, and the finishing kernel puts what their sum is into the mean.
#include "hkm_common.h"

namespace hkm {

typedef double doublex4 __attribute__((ext_vector_type(4)));

static constexpr int OH_THREADS = 512, OH_MAX_TILES = 8;

// The product multiplies every row by all clusters, sixteen at a time; the sort it replaces does not, but it is seven launches, which
// small calls feel.  Update alone of more than 32 clusters, product as many times as fast as the sort, over 1 to 31 columns --
// three tiles (up to 48 clusters of up to 15 columns): 1M rows 1.42 to 1.53, 2M 1.07 to 1.37, 4M of 1 column 0.94, of 5 1.00, of 7 1.05, of 15 1.43;
// four (64): 1M 1.20 to 1.33, 2M of 1 0.90, of 9 1.01, of 12 1.01 (4M: 1.08), of 15 1.12; five (80): 1M 1.12 to 1.17, 2M 0.78 to 0.98;
// six: 700 000 rows 1.10 to 1.25, 1M 0.88 to 1.12; seven: 700 000 1.09 to 1.13, 1M 0.89 to 0.94; eight: 500 000 1.10 to 1.29, 700 000
// 0.93 to 1.04, 1M of 18 0.77.  Up to 32 clusters: 1M x 18: 67 -> 61 us, 20M x 18: 1.07 times as fast.
bool onehot_eligible(int64_t N, int32_t D, int32_t K) {
    const int64_t tiles = int64_t((K + 15) / 16) * ((D + 16) / 16);
    if (N < 4096 || K > 128 || D > 128 || tiles > OH_MAX_TILES) return false;
    if (K <= 32 || N <= 500000) return true;
    if (tiles <= 3) return N <= 2000000 || D >= 7;
    if (tiles <= 5) return N <= 1000000 || (tiles == 4 && D >= 12);
    return tiles <= 7 && N <= 700000;
}
static int onehot_grid(int64_t N) {
    const int64_t want = (N + 511) / 512;  // 64 rows a wave at least
    return int(want < OH_MAX_GRID ? want : OH_MAX_GRID);
}

// U of a wave's groups of four rows: their share of the KT x DT tiles of 16 clusters x 16 columns (column D holds ones).
// value(u, d): the lane's of group u and column tile d, 0 behind the rows' ends; label(u): that of its row, -1 behind the last.
template <int KT, int DT, int U, class V, class L>
__device__ __forceinline__ void onehot_add(V value, L label, int D, int K, doublex4 (&acc)[KT][DT], unsigned* sOdd, int* sAny) {
    constexpr int COLS = DT * 16;
    const int j = threadIdx.x & 15;
    double x[U][DT];
    int lab[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
        lab[u] = label(u);
#pragma unroll
        for (int d = 0; d < DT; ++d) x[u][d] = value(u, d);
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
        bool bad = false;
#pragma unroll
        for (int d = 0; d < DT; ++d) bad = bad || !(fabs(x[u][d]) < HKM_INF);
        if (__any(bad)) {
#pragma unroll
            for (int d = 0; d < DT; ++d)
                if (!(fabs(x[u][d]) < HKM_INF)) {
                    const unsigned bit = x[u][d] != x[u][d] ? 4u : x[u][d] > 0.0 ? 1u : 2u;
                    if (lab[u] >= 0 && lab[u] < K) {
                        atomicOr(&sOdd[lab[u] * COLS + 16 * d + j], bit);
                        *sAny = 1;
                    }
                    x[u][d] = 0.0;
                }
        }
#pragma unroll
        for (int d = 0; d < DT; ++d) x[u][d] = 16 * d + j == D ? 1.0 : x[u][d];
#pragma unroll
        for (int k = 0; k < KT; ++k) {
            const double p = lab[u] == 16 * k + j ? 1.0 : 0.0;
#pragma unroll
            for (int d = 0; d < DT; ++d) acc[k][d] = __builtin_amdgcn_mfma_f64_16x16x4f64(p, x[u][d], acc[k][d], 0, 0, 0);
        }
    }
}

// The workgroup's sums out: the waves one after the other; register v of lane (q, j) is row q + 4 v of the tile, column j.
template <int KT, int DT>
__device__ __forceinline__ void onehot_out(const doublex4 (&acc)[KT][DT], int D, int K, double* sS, const unsigned* sOdd,
                                           const int* sAny, double* __restrict__ part, unsigned* __restrict__ odd,
                                           int32_t* __restrict__ odd_flag) {
    constexpr int WAVES = OH_THREADS / 64, COLS = DT * 16;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int j = lane & 15, q = lane >> 4;
    for (int w = 0; w < WAVES; ++w) {
        if (w == wave) {
#pragma unroll
            for (int k = 0; k < KT; ++k)
#pragma unroll
                for (int d = 0; d < DT; ++d)
#pragma unroll
                    for (int v = 0; v < 4; ++v) {
                        double& s = sS[(16 * k + q + 4 * v) * COLS + 16 * d + j];
                        s = w == 0 ? acc[k][d][v] : s + acc[k][d][v];
                    }
        }
        __syncthreads();
    }
    double* out = part + size_t(blockIdx.x) * K * (D + 1);
    for (int i = tid; i < K * (D + 1); i += OH_THREADS) {
        const int k = i / (D + 1), d = i - k * (D + 1);
        out[i] = sS[k * COLS + d];
    }
    if (tid == 0) odd_flag[blockIdx.x] = *sAny;
    if (*sAny) {
        unsigned* o = odd + size_t(blockIdx.x) * K * D;
        for (int i = tid; i < K * D; i += OH_THREADS) {
            const int k = i / D, d = i - k * D;
            o[i] = sOdd[k * COLS + d];
        }
    }
}

// rows of a wave, whole groups of four
__device__ __forceinline__ int64_t onehot_stretch(int64_t N) {
    const int64_t waves = int64_t(gridDim.x) * (OH_THREADS / 64);
    return ((N + waves - 1) / waves + 3) / 4 * 4;
}

template <int KT, int DT>
__global__ __launch_bounds__(OH_THREADS) void onehot_sum_kernel(const double* __restrict__ X, int64_t N, int D, int64_t ldx,
                                                                const int32_t* __restrict__ labels, int K,
                                                                double* __restrict__ part, unsigned* __restrict__ odd,
                                                                int32_t* __restrict__ odd_flag) {
    constexpr int WAVES = OH_THREADS / 64, COLS = DT * 16, ROWS = KT * 16;
    __shared__ double sS[ROWS * COLS];
    __shared__ unsigned sOdd[ROWS * COLS];
    __shared__ int sAny;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, j = lane & 15, q = lane >> 4;
    if (tid == 0) sAny = 0;
    for (int i = tid; i < ROWS * COLS; i += OH_THREADS) sOdd[i] = 0u;
    __syncthreads();
    doublex4 acc[KT][DT];
#pragma unroll
    for (int k = 0; k < KT; ++k)
#pragma unroll
        for (int d = 0; d < DT; ++d) acc[k][d] = doublex4{0.0, 0.0, 0.0, 0.0};
    const int64_t per = onehot_stretch(N), lo = (int64_t(blockIdx.x) * WAVES + wave) * per, hi = min(N, lo + per);
    constexpr int U = DT <= 2 ? 8 : 4;  // groups of four rows in flight
    for (int64_t r0 = lo; r0 < hi; r0 += 4 * U)
        onehot_add<KT, DT, U>(
            [&](int u, int d) {
                const int64_t r = r0 + 4 * u + q;
                return r < hi && 16 * d + j < D ? X[r * ldx + 16 * d + j] : 0.0;
            },
            [&](int u) { return r0 + 4 * u + q < hi ? labels[r0 + 4 * u + q] : -1; }, D, K, acc, sOdd, &sAny);
    onehot_out<KT, DT>(acc, D, K, sS, sOdd, &sAny, part, odd, odd_flag);
}

// Labels and sums in one pass over memory.  A wave takes 64 rows of its stretch at a time, loaded as the product wants them
// (whole lines) while the 64 before are worked on, and kept in LDS of its own: each lane finds the nearest centroid of one
// row (the sums of assign_f64_rows_kernel in its order: the same bits), then the wave multiplies the 64 rows as above.  Same
// stretches and order as onehot_sum_kernel: the same means.
//
// Bound by memory with few centroids (4M x 31, K = 2: 4.5 TB/s in all), by the way of the centroids through the scalar unit with
// more: eight waves on a CU do not hide it.  Step of 4M rows, assignment and update -> one pass: 31, K = 2: 561 -> 230 us; 24, 8: 376 ->
// 259; 18, 16: 319 -> 293; of 1M: 31, 5: 125 -> 78; 18, 4: 79 -> 65; 18, 16: 86 and 86; of 30 000: 21 -> 18 to 28 -> 25 (a launch less).
// (Each lane loading its own row, as assign_f64_rows_kernel does, and the product the rows again: 93 at 18, 16.)
template <int DP, int DT>
__global__ __launch_bounds__(OH_THREADS) void onehot_step_kernel(const double* __restrict__ X, int64_t N, int D, int64_t ldx,
                                                                 const double* __restrict__ C, int K, int32_t* __restrict__ labels,
                                                                 double* __restrict__ min_d2, double* __restrict__ part,
                                                                 unsigned* __restrict__ odd, int32_t* __restrict__ odd_flag) {
    constexpr int KT = 1, WAVES = OH_THREADS / 64, COLS = DT * 16, ROWS = KT * 16;
    constexpr int LD = DP + 1;  // odd: a lane's own row is read without conflicts
    extern __shared__ __align__(16) double lds_rows[];
    __shared__ double sS[ROWS * COLS];
    __shared__ double sCn[ROWS];
    __shared__ unsigned sOdd[ROWS * COLS];
    __shared__ int sAny;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, j = lane & 15, q = lane >> 4;
    if (tid == 0) sAny = 0;
    for (int i = tid; i < ROWS * COLS; i += OH_THREADS) sOdd[i] = 0u;
    for (int k = tid; k < K; k += OH_THREADS) {
        const double* row = C + k * D;
        double s = 0.0;
        for (int d = 0; d < D; ++d) s = fma(row[d], row[d], s);
        sCn[k] = s;
    }
    __syncthreads();
    doublex4 acc[KT][DT];
#pragma unroll
    for (int k = 0; k < KT; ++k)
#pragma unroll
        for (int d = 0; d < DT; ++d) acc[k][d] = doublex4{0.0, 0.0, 0.0, 0.0};
    const int64_t per = onehot_stretch(N), lo = (int64_t(blockIdx.x) * WAVES + wave) * per, hi = min(N, lo + per);
    double* sR = lds_rows + wave * 64 * LD;
    double next[16][DT];
    auto load = [&](int64_t r0) {
#pragma unroll
        for (int u = 0; u < 16; ++u)
#pragma unroll
            for (int d = 0; d < DT; ++d) {
                const int64_t r = r0 + 4 * u + q;
                next[u][d] = r < hi && 16 * d + j < D ? X[r * ldx + 16 * d + j] : 0.0;
            }
    };
    if (lo < hi) load(lo);
    for (int64_t r0 = lo; r0 < hi; r0 += 64) {
        wave_lds_sync();
#pragma unroll
        for (int u = 0; u < 16; ++u)
#pragma unroll
            for (int d = 0; d < DT; ++d)
                if (16 * d + j < DP) sR[(4 * u + q) * LD + 16 * d + j] = next[u][d];
        wave_lds_sync();
        if (r0 + 64 < hi) load(r0 + 64);
        double x[DP], xn = 0.0, m = __builtin_inf();
#pragma unroll
        for (int d = 0; d < DP; ++d) x[d] = sR[lane * LD + d];
        int mi = 0x7fffffff;
#pragma unroll
        for (int d = 0; d < DP; ++d)
            if (d < D) xn = fma(x[d], x[d], xn);
        auto offer = [&](double dot, int k) {
            double v = fma(-2.0, dot, xn + sCn[k]);
            v = v > 0.0 ? v : (v != v ? v : 0.0);
            if (v < m) {  // ascending index, strict '<': first index wins ties
                m = v;
                mi = k;
            }
        };
        int k = 0;
        for (; k + 2 <= K; k += 2) {
            const double *c = C + k * D, *e = c + D;
            double s = 0.0, t = 0.0;
#pragma unroll
            for (int d = 0; d < DP; ++d)
                if (d < DP - 8 || d < D) {
                    s = fma(x[d], c[d], s);
                    t = fma(x[d], e[d], t);
                }
            offer(s, k);
            offer(t, k + 1);
        }
        if (k < K) {
            const double* c = C + k * D;
            double s = 0.0;
#pragma unroll
            for (int d = 0; d < DP; ++d)
                if (d < DP - 8 || d < D) s = fma(x[d], c[d], s);
            offer(s, k);
        }
        const bool in = r0 + lane < hi;
        const int mine = in ? (mi == 0x7fffffff ? 0 : mi) : -1;
        if (in) {
            labels[r0 + lane] = mine;
            if (min_d2) min_d2[r0 + lane] = m;
        }
        constexpr int U = 4;
#pragma unroll 1
        for (int g = 0; g < 16; g += U)
            if (r0 + 4 * g < hi)  // uniform
                onehot_add<KT, DT, U>([&](int u, int d) { return 16 * d + j < DP ? sR[(4 * (g + u) + q) * LD + 16 * d + j] : 0.0; },
                                      [&](int u) { return __shfl(mine, 4 * (g + u) + q); }, D, K, acc, sOdd, &sAny);
    }
    onehot_out<KT, DT>(acc, D, K, sS, sOdd, &sAny, part, odd, odd_flag);
}

// Means and their share of the shift: a workgroup has 16 entries (cluster, column), 16 threads each add a stretch of the
// partial sums in order, then the stretches are added in order.
__global__ __launch_bounds__(256) void onehot_finalize_kernel(const double* __restrict__ part, const unsigned* __restrict__ odd,
                                                              const int32_t* __restrict__ odd_flag, int grid, int K, int D,
                                                              double* __restrict__ C_new, int64_t ldcn,
                                                              int64_t* __restrict__ counts_out,
                                                              const double* __restrict__ C_old, double* __restrict__ shift_part) {
    __shared__ double sS[16][17], sN[16][17];
    const int tid = threadIdx.x, e = tid & 15, sl = tid >> 4;
    const int i = blockIdx.x * 16 + e;
    const bool ok = i < K * D;
    const int k = ok ? i / D : 0, d = ok ? i - k * D : 0;
    const int per = (grid + 15) / 16, w0 = sl * per, w1 = min(grid, w0 + per);
    const size_t row = size_t(K) * (D + 1);
    double sum = 0.0, cnt = 0.0;
    const double* p = part + size_t(k) * (D + 1);
    for (int w = w0; w < w1; w += 8) {
        double v[8], c[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const bool in = w + u < w1;
            v[u] = in ? p[size_t(w + u) * row + d] : 0.0;
            c[u] = in ? p[size_t(w + u) * row + D] : 0.0;
        }
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            sum += v[u];
            cnt += c[u];
        }
    }
    sS[e][sl] = sum;
    sN[e][sl] = cnt;
    unsigned bits = 0;
    for (int w = w0; w < w1; ++w)
        if (odd_flag[w] && ok) bits |= odd[size_t(w) * K * D + i];
    __shared__ unsigned sBits[16];
    if (tid < 16) sBits[tid] = 0;
    __syncthreads();
    if (bits) atomicOr(&sBits[e], bits);
    __syncthreads();
    double sq = 0.0;
    if (sl == 0 && ok) {
        sum = 0.0;
        cnt = 0.0;
#pragma unroll
        for (int s = 0; s < 16; ++s) {
            sum += sS[e][s];
            cnt += sN[e][s];
        }
        const unsigned b = sBits[e];
        if (b & 1u) sum += __builtin_inf();
        if (b & 2u) sum -= __builtin_inf();
        if (b & 4u) sum = __builtin_nan("");
        const int64_t n = int64_t(cnt);
        const double cnew = sum / double(float(n < 1 ? 1 : n));
        C_new[int64_t(k) * ldcn + d] = cnew;
        if (d == 0 && counts_out) counts_out[k] = n;
        if (C_old) {
            const double df = C_old[int64_t(k) * D + d] - cnew;
            sq = df * df;
        }
    }
    if (C_old) {
        const double t = block_sum_256(sq);
        if (tid == 0) shift_part[blockIdx.x] = t;
    }
}

__global__ __launch_bounds__(256) void onehot_shift_kernel(const double* __restrict__ part, int nb, double* __restrict__ out) {
    double acc = 0.0;
    for (int i = threadIdx.x; i < nb; i += 256) acc += part[i];
    const double t = block_sum_256(acc);
    if (threadIdx.x == 0) *out = t;
}

template <int KT, int DT>
static void go(const double* X, int64_t N, int32_t D, int64_t ldx, const int32_t* labels, int32_t K, const OnehotWorkspace& w,
               int grid, hipStream_t st) {
    hipLaunchKernelGGL((onehot_sum_kernel<KT, DT>), dim3(unsigned(grid)), dim3(OH_THREADS), 0, st, X, N, D, ldx, labels, K, w.part,
                       w.odd, w.flag);
}

template <int DP, int DT>
static int go_step(const double* X, int64_t N, int32_t D, int64_t ldx, const double* C, int32_t K, int32_t* labels, double* min_d2,
                   const OnehotWorkspace& w, int grid, hipStream_t st) {
    const size_t lds = size_t(OH_THREADS) * (DP + 1) * sizeof(double);
    auto kern = onehot_step_kernel<DP, DT>;
    if (lds > 48 * 1024) {
        hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, int(lds));
        if (e != hipSuccess) return fail(HKM_EHIP, "hipFuncSetAttribute: %s", hipGetErrorString(e));
    }
    hipLaunchKernelGGL(kern, dim3(unsigned(grid)), dim3(OH_THREADS), lds, st, X, N, D, ldx, C, K, labels, min_d2, w.part, w.odd, w.flag);
    return check_launch("onehot_step_kernel");
}

static int finish(const OnehotWorkspace& w, int grid, int32_t K, int32_t D, double* C_new, int64_t ldcn, int64_t* counts,
                  const double* C_old, double* shift, hipStream_t st) {
    const int nb = (K * D + 15) / 16;
    hipLaunchKernelGGL(onehot_finalize_kernel, dim3(unsigned(nb)), dim3(256), 0, st, w.part, w.odd, w.flag, grid, K, D, C_new, ldcn,
                       counts, C_old, w.shift_part);
    int rc = check_launch("onehot_finalize_kernel");
    if (rc || !C_old) return rc;
    hipLaunchKernelGGL(onehot_shift_kernel, dim3(1), dim3(256), 0, st, w.shift_part, nb, shift);
    return check_launch("onehot_shift_kernel");
}

// From 9 features on: rows of up to 8 are read by the assignment at memory rate already (1M x 8, K = 16: 46 us in two passes, 61 in
// one).  More than 16 centroids: 1M x 18, K = 32: 116 and 137.  13 to 16 centroids of narrow rows: 1M x 9, 16: 56 and 58, x 13: 64 and 66,
// but 200 000 x 9: 25 -> 24.
bool onehot_step_eligible(int64_t N, int32_t D, int32_t K) {
    return onehot_eligible(N, D, K) && D > 8 && D <= 31 && K <= 16 && (K <= 12 || D > 13 || N < 500000);
}

// C and C_new with rows of D
int launch_step_onehot_f64(const double* X, int64_t N, int32_t D, int64_t ldx, const double* C, int32_t K, double* C_new, int32_t* labels,
                           double* min_d2, const OnehotWorkspace& w, double* shift, hipStream_t st) {
    const int grid = onehot_grid(N);
    int rc;
    // rows padded to a multiple of 8 features (the kernel tests only the last eight), a column more for the counts
    if (D <= 15) rc = go_step<16, 1>(X, N, D, ldx, C, K, labels, min_d2, w, grid, st);
    else if (D <= 16) rc = go_step<16, 2>(X, N, D, ldx, C, K, labels, min_d2, w, grid, st);
    else if (D <= 24) rc = go_step<24, 2>(X, N, D, ldx, C, K, labels, min_d2, w, grid, st);
    else rc = go_step<32, 2>(X, N, D, ldx, C, K, labels, min_d2, w, grid, st);
    if (rc) return rc;
    return finish(w, grid, K, D, C_new, D, nullptr, C, shift, st);
}

int launch_update_onehot_f64(const double* X, int64_t N, int32_t D, int64_t ldx, const int32_t* labels, int32_t K, double* C_new,
                             int64_t ldcn, int64_t* counts, const OnehotWorkspace& w, const double* C_old, double* shift,
                             hipStream_t st) {
    const int grid = onehot_grid(N), kt = (K + 15) / 16, dt = (D + 16) / 16;
#define HKM_OH(k, d)                                      \
    if (kt == k && dt == d) {                             \
        go<k, d>(X, N, D, ldx, labels, K, w, grid, st);   \
    }
    HKM_OH(1, 1) HKM_OH(1, 2) HKM_OH(1, 3) HKM_OH(1, 4) HKM_OH(1, 5) HKM_OH(1, 6) HKM_OH(1, 7) HKM_OH(1, 8)
    HKM_OH(2, 1) HKM_OH(2, 2) HKM_OH(2, 3) HKM_OH(2, 4) HKM_OH(3, 1) HKM_OH(3, 2) HKM_OH(4, 1) HKM_OH(4, 2)
    HKM_OH(5, 1) HKM_OH(6, 1) HKM_OH(7, 1) HKM_OH(8, 1)
#undef HKM_OH
    const int rc = check_launch("onehot_sum_kernel");
    return rc ? rc : finish(w, grid, K, D, C_new, ldcn, counts, C_old, shift, st);
}

}  // namespace hkm
