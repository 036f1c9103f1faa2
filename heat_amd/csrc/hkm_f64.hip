// float64 data: fused quadratic-expansion distance + argmin on the fp64 vector ALU.  The reference
// runs float64 inputs through the same op sequence in float64 (promote(X, Y, float32) keeps float64,
// heat/spatial/distance.py:392-403), so d2 = max(0, (|x|^2 + |c|^2) - 2 x.c) is evaluated in fp64
// here as well; the N x K matrix is never written.  Same tiling as the Manhattan kernel: a workgroup
// owns 64 points and walks the centroids in tiles of 64 (4 x 4 register block per lane, 16-feature
// chunks through LDS); squared norms are accumulated from the staged tiles on the way.
#include "hkm_common.h"

namespace hkm {

static constexpr int F64_T = 64;
static constexpr int F64_KC = 16;

__global__ __launch_bounds__(256) void assign_f64_kernel(const double* __restrict__ X, int64_t N,
                                                         int64_t ldx, const double* __restrict__ C,
                                                         int K, int64_t ldc, int D,
                                                         int32_t* __restrict__ labels,
                                                         double* __restrict__ min_d2) {
    __shared__ double sX[F64_KC][F64_T + 2];
    __shared__ double sC[F64_KC][F64_T + 2];
    __shared__ double sXn[F64_T], sCn[F64_T];
    const int tid = threadIdx.x;
    const int tx = tid & 15, ty = tid >> 4;
    const int lk = tid & 15, lr = tid >> 4;
    const int64_t i0 = int64_t(blockIdx.x) * F64_T;

    // squared norms of the tile's points, summed in feature order
    if (tid < F64_T) {
        const int64_t g = i0 + tid;
        double s = 0.0;
        if (g < N) {
            const double* row = X + g * ldx;
            for (int d = 0; d < D; ++d) s = fma(row[d], row[d], s);
        }
        sXn[tid] = s;
    }

    double bd[4];
    int bi[4];
#pragma unroll
    for (int a = 0; a < 4; ++a) {
        bd[a] = __builtin_inf();
        bi[a] = 0x7fffffff;
    }

    for (int j0 = 0; j0 < K; j0 += F64_T) {
        __syncthreads();  // previous tile's sCn is no longer read
        if (tid < F64_T) {
            const int g = j0 + tid;
            double s = 0.0;
            if (g < K) {
                const double* row = C + int64_t(g) * ldc;
                for (int d = 0; d < D; ++d) s = fma(row[d], row[d], s);
            }
            sCn[tid] = s;
        }
        double acc[4][4];
#pragma unroll
        for (int a = 0; a < 4; ++a)
#pragma unroll
            for (int b = 0; b < 4; ++b) acc[a][b] = 0.0;
        for (int d0 = 0; d0 < D; d0 += F64_KC) {
            __syncthreads();
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int r = lr + 16 * q;
                const int d = d0 + lk;
                const int64_t gi = i0 + r;
                const int gj = j0 + r;
                sX[lk][r] = (gi < N && d < D) ? X[gi * ldx + d] : 0.0;
                sC[lk][r] = (gj < K && d < D) ? C[int64_t(gj) * ldc + d] : 0.0;
            }
            __syncthreads();
#pragma unroll
            for (int k = 0; k < F64_KC; ++k) {
                double xa[4], cb[4];
#pragma unroll
                for (int a = 0; a < 4; ++a) xa[a] = sX[k][ty * 4 + a];
#pragma unroll
                for (int b = 0; b < 4; ++b) cb[b] = sC[k][tx * 4 + b];
#pragma unroll
                for (int a = 0; a < 4; ++a)
#pragma unroll
                    for (int b = 0; b < 4; ++b) acc[a][b] = fma(xa[a], cb[b], acc[a][b]);
            }
        }
#pragma unroll
        for (int a = 0; a < 4; ++a) {
            const double xn = sXn[ty * 4 + a];
            double d = __builtin_inf();
            int i = 0x7fffffff;
#pragma unroll
            for (int b = 0; b < 4; ++b) {
                const int gj = j0 + tx * 4 + b;
                if (gj >= K) continue;
                double v = fma(-2.0, acc[a][b], xn + sCn[tx * 4 + b]);
                v = v > 0.0 ? v : (v != v ? v : 0.0);
                if (v < d) {  // ascending index, strict '<': first index wins ties
                    d = v;
                    i = gj;
                }
            }
#pragma unroll
            for (int w = 1; w < 16; w <<= 1) {
                const double od = __shfl_xor(d, w);
                const int oi = __shfl_xor(i, w);
                if (od < d || (od == d && oi < i)) {
                    d = od;
                    i = oi;
                }
            }
            if (d < bd[a] || (d == bd[a] && i < bi[a])) {
                bd[a] = d;
                bi[a] = i;
            }
        }
    }

    if (tx == 0) {
#pragma unroll
        for (int a = 0; a < 4; ++a) {
            const int64_t gi = i0 + ty * 4 + a;
            if (gi >= N) continue;
            labels[gi] = bi[a] == 0x7fffffff ? 0 : bi[a];
            if (min_d2) min_d2[gi] = bd[a];
        }
    }
}

// Narrow rows and few centroids (D <= 8, K (D + 1) <= F64S_LDS): the 64 x 64 tile would be mostly
// padding.  One point per lane, the centroids and their squared norms broadcast from LDS; every sum
// in feature order with fma, so the values equal those of the tiled kernel bit for bit.
static constexpr int F64S_THREADS = 256;
static constexpr int F64S_LDS = 2048;  // doubles: K rows of D coordinates + the squared norm

template <int D>
__global__ __launch_bounds__(F64S_THREADS) void assign_f64_small_kernel(
    const double* __restrict__ X, int64_t N, int64_t ldx, const double* __restrict__ C, int K, int64_t ldc,
    int32_t* __restrict__ labels, double* __restrict__ min_d2, int64_t nbatches) {
    __shared__ double sC[F64S_LDS];
    const int tid = threadIdx.x;
    for (int k = tid; k < K; k += F64S_THREADS) {
        const double* row = C + int64_t(k) * ldc;
        double s = 0.0;
#pragma unroll
        for (int d = 0; d < D; ++d) {
            sC[k * (D + 1) + d] = row[d];
            s = fma(row[d], row[d], s);
        }
        sC[k * (D + 1) + D] = s;
    }
    __syncthreads();
    for (int64_t b = blockIdx.x; b < nbatches; b += gridDim.x) {
        const int64_t i = b * F64S_THREADS + tid;
        const double* xp = X + (i < N ? i : N - 1) * ldx;
        double x[D], xn = 0.0;
#pragma unroll
        for (int d = 0; d < D; ++d) {
            x[d] = xp[d];
            xn = fma(x[d], x[d], xn);
        }
        double m = __builtin_inf();
        int mi = 0x7fffffff;
#pragma unroll 4
        for (int k = 0; k < K; ++k) {
            const double* c = sC + k * (D + 1);
            double dot = 0.0;
#pragma unroll
            for (int d = 0; d < D; ++d) dot = fma(x[d], c[d], dot);
            double v = fma(-2.0, dot, xn + c[D]);
            v = v > 0.0 ? v : (v != v ? v : 0.0);
            if (v < m) {  // ascending index, strict '<': first index wins ties
                m = v;
                mi = k;
            }
        }
        if (i < N) {
            labels[i] = mi == 0x7fffffff ? 0 : mi;
            if (min_d2) min_d2[i] = m;
        }
    }
}

// Up to 64 features and any number of centroids: one point per lane as well, the row in registers (in 16-byte loads at any
// 8-byte boundary), the centroids -- the same for all lanes -- through the scalar unit, their squared norms in LDS.  The
// 64 x 64 tiles above spent their time on 8-byte staging loads and two barriers per 16 features: 1M x 18, K = 16 took
// 218 us there.  Bound: fp64 fused multiply-adds, K D per row, and the rows' way from memory.  Every sum in feature
// order with fma, two centroids side by side, so the values equal those of the tiled kernel bit for bit.
static constexpr int F64R_KT = 1024;  // norms held in LDS at a time

template <int DP>
__global__ __launch_bounds__(256) void assign_f64_rows_kernel(
    const double* __restrict__ X, int64_t N, int64_t ldx, const double* __restrict__ C, int K, int64_t ldc, int D,
    int32_t* __restrict__ labels, double* __restrict__ min_d2, int64_t nbatches) {
    __shared__ double sCn[F64R_KT];
    struct __attribute__((packed, aligned(8))) any2 { double v[2]; };
    const int tid = threadIdx.x;
    const bool once = K <= F64R_KT;
    auto norms = [&](int k0) {
        for (int k = k0 + tid; k < K && k < k0 + F64R_KT; k += 256) {
            const double* row = C + int64_t(k) * ldc;
            double s = 0.0;
            for (int d = 0; d < D; ++d) s = fma(row[d], row[d], s);
            sCn[k - k0] = s;
        }
    };
    if (once) {
        norms(0);
        __syncthreads();
    }
    for (int64_t b = blockIdx.x; b < nbatches; b += gridDim.x) {
        const int64_t i = b * 256 + tid;
        const double* xp = X + (i < N ? i : N - 1) * ldx;
        double x[DP], xn = 0.0;
#pragma unroll
        for (int d = 0; d < DP; d += 2) {
            x[d] = 0.0;
            x[d + 1] = 0.0;
            if (d + 1 < D) {  // uniform
                const any2 v = *reinterpret_cast<const any2*>(xp + d);
                x[d] = v.v[0];
                x[d + 1] = v.v[1];
            } else if (d < D) {
                x[d] = xp[d];
            }
        }
#pragma unroll
        for (int d = 0; d < DP; ++d)
            if (d < D) xn = fma(x[d], x[d], xn);
        double m = __builtin_inf();
        int mi = 0x7fffffff;
        auto offer = [&](double dot, double cn, int k) {
            double v = fma(-2.0, dot, xn + cn);
            v = v > 0.0 ? v : (v != v ? v : 0.0);
            if (v < m) {  // ascending index, strict '<': first index wins ties
                m = v;
                mi = k;
            }
        };
        for (int k0 = 0; k0 < K; k0 += F64R_KT) {
            if (!once) {
                __syncthreads();
                norms(k0);
                __syncthreads();
            }
            const int k1 = min(K, k0 + F64R_KT);
            int k = k0;
            for (; k + 2 <= k1; k += 2) {
                const double* c = C + int64_t(k) * ldc;
                const double* e = c + ldc;
                double s = 0.0, t = 0.0;
#pragma unroll
                for (int d = 0; d < DP; ++d)
                    if (d < DP - 8 || d < D) {
                        s = fma(x[d], c[d], s);
                        t = fma(x[d], e[d], t);
                    }
                offer(s, sCn[k - k0], k);
                offer(t, sCn[k + 1 - k0], k + 1);
            }
            if (k < k1) {
                const double* c = C + int64_t(k) * ldc;
                double s = 0.0;
#pragma unroll
                for (int d = 0; d < DP; ++d)
                    if (d < DP - 8 || d < D) s = fma(x[d], c[d], s);
                offer(s, sCn[k - k0], k);
            }
        }
        if (i < N) {
            labels[i] = mi == 0x7fffffff ? 0 : mi;
            if (min_d2) min_d2[i] = m;
        }
    }
}

template <int DP>
static int launch_assign_f64_rows_t(const double* X, int64_t N, int64_t ldx, const double* C, int32_t K, int64_t ldc,
                                    int32_t D, int32_t* labels, double* min_d2, hipStream_t st) {
    const int64_t nbatches = (N + 255) / 256;
    int64_t grid = int64_t(num_cus()) * 8;
    if (grid > nbatches) grid = nbatches;
    hipLaunchKernelGGL(assign_f64_rows_kernel<DP>, dim3((unsigned)grid), dim3(256), 0, st, X, N, ldx, C, K, ldc, D, labels,
                       min_d2, nbatches);
    return check_launch("assign_f64_rows_kernel");
}

template <int D>
static int launch_assign_f64_small_t(const double* X, int64_t N, int64_t ldx, const double* C, int32_t K,
                                     int64_t ldc, int32_t* labels, double* min_d2, hipStream_t st) {
    const int64_t nbatches = (N + F64S_THREADS - 1) / F64S_THREADS;
    int64_t grid = int64_t(num_cus()) * 8;
    if (grid > nbatches) grid = nbatches;
    hipLaunchKernelGGL(assign_f64_small_kernel<D>, dim3((unsigned)grid), dim3(F64S_THREADS), 0, st, X, N, ldx, C, K,
                       ldc, labels, min_d2, nbatches);
    return check_launch("assign_f64_small_kernel");
}

int launch_assign_f64(const double* X, int64_t N, int32_t D, int64_t ldx, const double* C, int32_t K,
                      int64_t ldc, int32_t* labels, double* min_d2, hipStream_t st) {
    if (D <= 8 && int64_t(K) * (D + 1) <= F64S_LDS) {
#define HKM_CASE(d) \
    case d:         \
        return launch_assign_f64_small_t<d>(X, N, ldx, C, K, ldc, labels, min_d2, st);
        switch (D) {
            HKM_CASE(1) HKM_CASE(2) HKM_CASE(3) HKM_CASE(4) HKM_CASE(5) HKM_CASE(6) HKM_CASE(7) HKM_CASE(8)
        }
#undef HKM_CASE
    }
    if (N > 0 && D <= 64) {
        // padded to a multiple of 8 features (assign_f64_rows_kernel tests only the last eight)
#define HKM_CASE(d) \
    if (D <= d) return launch_assign_f64_rows_t<d>(X, N, ldx, C, K, ldc, D, labels, min_d2, st);
        HKM_CASE(8) HKM_CASE(16) HKM_CASE(24) HKM_CASE(32) HKM_CASE(40) HKM_CASE(48) HKM_CASE(56) HKM_CASE(64)
#undef HKM_CASE
    }
    const int64_t tiles = (N + F64_T - 1) / F64_T;
    if (tiles > 0x7fffffffLL) return fail(HKM_EUNSUPPORTED, "assign_f64: too many row tiles");
    hipLaunchKernelGGL(assign_f64_kernel, dim3((unsigned)tiles), dim3(256), 0, st, X, N, ldx, C, K, ldc, D,
                       labels, min_d2);
    return check_launch("assign_f64_kernel");
}

}  // namespace hkm
