// The update of few clusters of float64 rows: per-cluster sums as a product of matrices on the fp64 matrix cores.
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

bool onehot_eligible(int64_t N, int32_t D, int32_t K) {
    return N >= 4096 && K <= 128 && D <= 128 && int64_t((K + 15) / 16) * ((D + 16) / 16) <= OH_MAX_TILES;
}
static int onehot_grid(int64_t N) {
    const int64_t want = (N + 511) / 512;  // 64 rows a wave at least
    return int(want < OH_MAX_GRID ? want : OH_MAX_GRID);
}

// KT x DT tiles of 16 clusters x 16 columns; column D holds ones
template <int KT, int DT>
__global__ __launch_bounds__(OH_THREADS) void onehot_sum_kernel(const double* __restrict__ X, int64_t N, int D, int64_t ldx,
                                                                const int32_t* __restrict__ labels, int K,
                                                                double* __restrict__ part, unsigned* __restrict__ odd,
                                                                int32_t* __restrict__ odd_flag) {
    constexpr int WAVES = OH_THREADS / 64, COLS = DT * 16, ROWS = KT * 16;
    __shared__ double sS[ROWS * COLS];
    __shared__ unsigned sOdd[ROWS * COLS];
    __shared__ int sAny;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int j = lane & 15, q = lane >> 4;
    if (tid == 0) sAny = 0;
    for (int i = tid; i < ROWS * COLS; i += OH_THREADS) sOdd[i] = 0u;
    __syncthreads();
    doublex4 acc[KT][DT];
#pragma unroll
    for (int k = 0; k < KT; ++k)
#pragma unroll
        for (int d = 0; d < DT; ++d) acc[k][d] = doublex4{0.0, 0.0, 0.0, 0.0};
    const int64_t waves = int64_t(gridDim.x) * WAVES, w0 = int64_t(blockIdx.x) * WAVES + wave;
    const int64_t per = ((N + waves - 1) / waves + 3) / 4 * 4;  // rows of a wave, whole groups of four
    const int64_t lo = w0 * per, hi = min(N, lo + per);
    constexpr int U = DT <= 2 ? 8 : 4;  // groups of four rows in flight
    for (int64_t r0 = lo; r0 < hi; r0 += 4 * U) {
        double x[U][DT];
        int lab[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int64_t r = r0 + 4 * u + q;
            const bool in = r < hi;
            lab[u] = in ? labels[r] : -1;
#pragma unroll
            for (int d = 0; d < DT; ++d) x[u][d] = in && 16 * d + j < D ? X[r * ldx + 16 * d + j] : 0.0;
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
                            sAny = 1;
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
    // the waves one after the other; register v of lane (q, j) is row q + 4 v of the tile, column j
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
    if (tid == 0) odd_flag[blockIdx.x] = sAny;
    if (sAny) {
        unsigned* o = odd + size_t(blockIdx.x) * K * D;
        for (int i = tid; i < K * D; i += OH_THREADS) {
            const int k = i / D, d = i - k * D;
            o[i] = sOdd[k * COLS + d];
        }
    }
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
    int rc = check_launch("onehot_sum_kernel");
    if (rc) return rc;
    const int nb = (K * D + 15) / 16;
    hipLaunchKernelGGL(onehot_finalize_kernel, dim3(unsigned(nb)), dim3(256), 0, st, w.part, w.odd, w.flag, grid, K, D, C_new, ldcn,
                       counts, C_old, w.shift_part);
    if ((rc = check_launch("onehot_finalize_kernel")) || !C_old) return rc;
    hipLaunchKernelGGL(onehot_shift_kernel, dim3(1), dim3(256), 0, st, w.shift_part, nb, shift);
    return check_launch("onehot_shift_kernel");
}

}  // namespace hkm
