// Full pairwise distance matrices for the public cdist / rbf / manhattan API
// (heat/spatial/distance.py:17-133): quadratic expansion max(0, (|x|^2 + |y|^2) - 2 x.y), the direct
// form sum((x-y)^2) and sum|x-y|, followed by sqrt or exp(-d2 / (2 sigma^2)).  The output is M x Nn
// floats, so for the feature counts these functions are used with the kernel is bound by writing the
// matrix; a 64 x 64 output tile per workgroup with a 4 x 4 register block per lane keeps the X / Y
// re-reads in L2 and the stores 16 bytes wide.
#include "hkm_common.h"

namespace hkm {

static constexpr int CD_T = 64;   // tile edge

// METRIC: 0 = quadratic expansion (squared, optional sqrt), 1 = direct sum((x-y)^2) (optional sqrt),
//         2 = sum |x-y|;  gauss != 0 applies exp(-d2 * gauss) to the squared distance instead of sqrt
// square roots of a lane's block: float takes the short correctly rounded form unless some lane of
// the wave holds a positive value below its range (one integer minimum tree decides)
__device__ __forceinline__ void cd_sqrt_block(float (&v)[4][4]) {
    unsigned m = 0xffffffffu;
#pragma unroll
    for (int a = 0; a < 4; ++a)
#pragma unroll
        for (int b = 0; b < 4; b += 2) m = min(m, min(sqrt_short_key(v[a][b]), sqrt_short_key(v[a][b + 1])));
    if (__builtin_amdgcn_ballot_w64(m < SQRT_SHORT_KEY_LIMIT) != 0) {
#pragma unroll
        for (int a = 0; a < 4; ++a)
#pragma unroll
            for (int b = 0; b < 4; ++b) v[a][b] = sqrtf(v[a][b]);
    } else {
#pragma unroll
        for (int a = 0; a < 4; ++a)
#pragma unroll
            for (int b = 0; b < 4; ++b) v[a][b] = sqrt_rn_short(v[a][b]);
    }
}
__device__ __forceinline__ void cd_sqrt_block(double (&v)[4][4]) {
#pragma unroll
    for (int a = 0; a < 4; ++a)
#pragma unroll
        for (int b = 0; b < 4; ++b) v[a][b] = sqrt(v[a][b]);
}
__device__ __forceinline__ void store_row4(float* p, const float (&v)[4]) {
    *reinterpret_cast<float4*>(p) = make_float4(v[0], v[1], v[2], v[3]);
}
__device__ __forceinline__ void store_row4(double* p, const double (&v)[4]) {
#pragma unroll
    for (int b = 0; b < 4; ++b) p[b] = v[b];
}
__device__ __forceinline__ float cd_exp(float v) { return expf(v); }
__device__ __forceinline__ double cd_exp(double v) { return exp(v); }
__device__ __forceinline__ float cd_abs(float v) { return fabsf(v); }
__device__ __forceinline__ double cd_abs(double v) { return fabs(v); }
__device__ __forceinline__ float cd_fma(float a, float b, float c) { return fmaf(a, b, c); }
__device__ __forceinline__ double cd_fma(double a, double b, double c) { return fma(a, b, c); }

// KU: features of a staged chunk that may take part in the arithmetic (rows of at most 4 / 8 features would otherwise
// spend their time testing for the end); the loop ends with the row, two features at a time.  (With chunks of 16
// always worked off in full, rows of 18 features paid for 32: 40 000 x 40 000 took 3.15 ms.)
//
// SYM: X and Y are the same matrix.  Every operation of an element commutes in its two rows (differences enter squared
// or as absolute values, products and the sum of the norms commute), so element (j, i) has the bits of (i, j): only the
// tiles on and below the diagonal are computed, and each is stored a second time as its transpose.  The arithmetic (2
// vector instructions per feature and the square root) bounds this kernel, not the matrix it writes: 40 000 x 40 000 of 18
// features 2.55 -> 1.92 ms (the turned tiles stored straight from registers, in pieces of 64 bytes: 2.11).
template <typename T, int METRIC, int KU, bool SYM>
__global__ __launch_bounds__(256) void cdist_kernel(const T* __restrict__ X, int64_t M,
                                                    int64_t ldx, const T* __restrict__ Y,
                                                    int64_t Nn, int64_t ldy, int D,
                                                    T* __restrict__ out, int64_t ldo,
                                                    int sqrt_flag, T gauss, int64_t tiles_n, bool vec_out) {
    constexpr int KC = KU <= 16 ? 16 : 32;  // feature chunk
    __shared__ __align__(16) T stage[2][KC][CD_T + 4];
    T(*sX)[CD_T + 4] = stage[0];
    T(*sY)[CD_T + 4] = stage[1];
    __shared__ T sXn[CD_T], sYn[CD_T];
    const int tid = threadIdx.x;
    int64_t tm = blockIdx.x / tiles_n, tn = blockIdx.x % tiles_n;
    if (SYM) {
        // tile blockIdx.x = tm (tm + 1) / 2 + tn of the lower triangle (the estimate is off by one at most)
        int64_t t = int64_t((sqrtf(8.0f * float(blockIdx.x) + 1.0f) - 1.0f) * 0.5f);
        while (t * (t + 1) / 2 > int64_t(blockIdx.x)) --t;
        while ((t + 1) * (t + 2) / 2 <= int64_t(blockIdx.x)) ++t;
        tm = t;
        tn = int64_t(blockIdx.x) - t * (t + 1) / 2;
    }
    const int64_t i0 = tm * CD_T, j0 = tn * CD_T;

    // squared norms of the tile's rows / columns (quadratic expansion only), each summed in feature
    // order from the staged chunks: thread r < 64 owns row r of the X tile, thread 64 + r row r of Y
    T nrm = T(0);

    const int tx = tid & 15, ty = tid >> 4;
    T acc[4][4];
#pragma unroll
    for (int a = 0; a < 4; ++a)
#pragma unroll
        for (int b = 0; b < 4; ++b) acc[a][b] = T(0);

    // staging role: element (row lr, feature lk) of both tiles, passes of 256 / KC rows
    constexpr int RP = 256 / KC;
    const int lk = tid & (KC - 1), lr = tid / KC;
    for (int d0 = 0; d0 < D; d0 += KC) {
        __syncthreads();
#pragma unroll
        for (int q = 0; q < CD_T / RP; ++q) {
            const int r = lr + RP * q;
            const int d = d0 + lk;
            const int64_t gi = i0 + r, gj = j0 + r;
            sX[lk][r] = (gi < M && d < D) ? X[gi * ldx + d] : T(0);
            sY[lk][r] = (gj < Nn && d < D) ? Y[gj * ldy + d] : T(0);
        }
        __syncthreads();
        if (METRIC == 0 && tid < 2 * CD_T) {
            const T(*tile)[CD_T + 4] = tid < CD_T ? sX : sY;
            const int r = tid & (CD_T - 1), lim = min(KU, D - d0);
            for (int k = 0; k < lim; ++k) nrm = cd_fma(tile[k][r], tile[k][r], nrm);
        }
        const int lim = min(KU, D - d0);
#pragma unroll
        for (int k = 0; k < KU; ++k) {
            if ((k & 1) == 0 && k >= lim) break;  // (an odd row's last pair ends in a staged zero)
            T xa[4], yb[4];
#pragma unroll
            for (int a = 0; a < 4; ++a) xa[a] = sX[k][ty * 4 + a];
#pragma unroll
            for (int b = 0; b < 4; ++b) yb[b] = sY[k][tx * 4 + b];
#pragma unroll
            for (int a = 0; a < 4; ++a)
#pragma unroll
                for (int b = 0; b < 4; ++b) {
                    if (METRIC == 0) {
                        acc[a][b] = cd_fma(xa[a], yb[b], acc[a][b]);
                    } else if (METRIC == 1) {
                        const T df = xa[a] - yb[b];
                        acc[a][b] = cd_fma(df, df, acc[a][b]);
                    } else {
                        acc[a][b] += cd_abs(xa[a] - yb[b]);
                    }
                }
        }
    }
    if (METRIC == 0) {
        if (tid < 2 * CD_T) (tid < CD_T ? sXn : sYn)[tid & (CD_T - 1)] = nrm;
        __syncthreads();
    }

    // epilogue over the lane's 4 x 4 block, in place
    if (METRIC == 0) {
        T yn[4];
#pragma unroll
        for (int b = 0; b < 4; ++b) yn[b] = sYn[tx * 4 + b];
#pragma unroll
        for (int a = 0; a < 4; ++a) {
            const T xn = sXn[ty * 4 + a];
#pragma unroll
            for (int b = 0; b < 4; ++b) {
                // the reference's order; clamp at 0 (a NaN passes: NaN < 0 is false; the value is never
                // -0 because the sum of the norms is never -0)
                const T d = cd_fma(T(-2), acc[a][b], xn + yn[b]);
                acc[a][b] = d < T(0) ? T(0) : d;
            }
        }
    }
    if (METRIC != 2) {
        if (gauss != T(0)) {
#pragma unroll
            for (int a = 0; a < 4; ++a)
#pragma unroll
                for (int b = 0; b < 4; ++b) acc[a][b] = cd_exp(-acc[a][b] * gauss);
        } else if (sqrt_flag) {
            cd_sqrt_block(acc);
        }
    }
    // 16-byte stores where the row of four lies inside the matrix and is aligned
    const int64_t gj0 = j0 + tx * 4;
    const bool vec4 = sizeof(T) == 4 && vec_out && gj0 + 3 < Nn;
#pragma unroll
    for (int a = 0; a < 4; ++a) {
        const int64_t gi = i0 + ty * 4 + a;
        if (gi >= M) continue;
        T* row = out + gi * ldo + gj0;
        if (vec4) {
            store_row4(row, acc[a]);
        } else {
#pragma unroll
            for (int b = 0; b < 4; ++b)
                if (gj0 + b < Nn) row[b] = acc[a][b];
        }
    }
    if (SYM && tm != tn && KC == 32 && sizeof(T) == 4 && vec_out && i0 + CD_T <= M && j0 + CD_T <= Nn) {
        // whole tiles: turned round in LDS, so that the transpose leaves in rows of 256 bytes too
        __syncthreads();
        T(*turned)[CD_T + 4] = stage[0];  // [64][CD_T + 4]
#pragma unroll
        for (int b = 0; b < 4; ++b) {
            const T v[4] = {acc[0][b], acc[1][b], acc[2][b], acc[3][b]};
            store_row4(&turned[tx * 4 + b][ty * 4], v);
        }
        __syncthreads();
#pragma unroll
        for (int a = 0; a < 4; ++a) {
            const int r = ty + 16 * a;
            T v[4];
#pragma unroll
            for (int b = 0; b < 4; ++b) v[b] = turned[r][tx * 4 + b];
            store_row4(out + (j0 + r) * ldo + i0 + tx * 4, v);
        }
    } else if (SYM && tm != tn) {
        const int64_t gi0 = i0 + ty * 4;
        const bool tvec4 = sizeof(T) == 4 && vec_out && gi0 + 3 < M;
#pragma unroll
        for (int b = 0; b < 4; ++b) {
            if (gj0 + b >= Nn) continue;
            T* row = out + (gj0 + b) * ldo + gi0;
            const T v[4] = {acc[0][b], acc[1][b], acc[2][b], acc[3][b]};
            if (tvec4) {
                store_row4(row, v);
            } else {
#pragma unroll
                for (int a = 0; a < 4; ++a)
                    if (gi0 + a < M) row[a] = v[a];
            }
        }
    }
}

// The direct Euclidean form of large float matrices: 128 x 64 tiles, eight rows by four columns a lane.  What bounds it is the
// vector ALU (two instructions per feature and pair, about eleven for the square root); with 4 x 4 a lane, as above, a
// fifth of the instructions were staging, addresses and the tile's turn.  The staged chunk takes the row's features only
// (18 of 18, not 32 lanes for 18), all its loads are in flight at once.  Same operations in the same order per element.
// 40 000 x 40 000 of 18 features as a triangle 1.95 -> 1.48 ms (4.3 TB/s written), 20 000 x 20 000 of 18, both halves, 0.80 -> 0.59.
static constexpr int CDB_M = 128, CDB_N = 64, CDB_LD = CDB_M + CDB_N + 4;
static constexpr int64_t CDB_LEAST = 4096;

template <int KC, bool SYM>
__global__ __launch_bounds__(256, 4) void cdist_big_kernel(const float* __restrict__ X, int64_t M, int64_t ldx,
                                                        const float* __restrict__ Y, int64_t Nn, int64_t ldy, int D,
                                                        float* __restrict__ out, int64_t ldo, int sqrt_flag, float gauss,
                                                        int64_t tiles_n, bool vec_out) {
    constexpr int NQ = (CDB_M + CDB_N) * KC / 256;
    constexpr int TURN_LD = CDB_M + 4;
    __shared__ __align__(16) float stage[!SYM || KC * CDB_LD > 64 * TURN_LD ? KC * CDB_LD : 64 * TURN_LD];
    const int tid = threadIdx.x;
    int64_t tm = blockIdx.x / tiles_n, tn = blockIdx.x % tiles_n;
    if (SYM) {
        // row tm has the column tiles 0 .. 2 tm + 1 (its diagonal block whole): tile blockIdx.x = tm (tm + 1) + tn
        int64_t t = int64_t((sqrtf(4.0f * float(blockIdx.x) + 1.0f) - 1.0f) * 0.5f);
        while (t * (t + 1) > int64_t(blockIdx.x)) --t;
        while ((t + 1) * (t + 2) <= int64_t(blockIdx.x)) ++t;
        tm = t;
        tn = int64_t(blockIdx.x) - t * (t + 1);
        if (tn >= tiles_n) return;  // (the last row's)
    }
    const int64_t i0 = tm * CDB_M, j0 = tn * CDB_N;
    const int tx = tid & 15, ty = tid >> 4;
    float acc[8][4];
#pragma unroll
    for (int a = 0; a < 8; ++a)
#pragma unroll
        for (int b = 0; b < 4; ++b) acc[a][b] = 0.f;

    for (int d0 = 0; d0 < D; d0 += KC) {
        const int lim = min(KC, D - d0), total = (CDB_M + CDB_N) * lim;
        const float inv = 1.0f / float(lim);
        float v[NQ];
        auto row_of = [&](int i) { return int((float(i) + 0.5f) * inv); };  // (exact: i < 2^13)
#pragma unroll
        for (int q = 0; q < NQ; ++q) {
            if (256 * q >= total) break;  // uniform
            const int i = tid + 256 * q, r = row_of(i), d = i - r * lim;
            const int64_t g = r < CDB_M ? i0 + r : j0 + r - CDB_M;
            const bool in = i < total && g < (r < CDB_M ? M : Nn);
            const float* p = r < CDB_M ? X + g * ldx : Y + g * ldy;
            v[q] = in ? p[d0 + d] : 0.f;
        }
        __syncthreads();
#pragma unroll
        for (int q = 0; q < NQ; ++q) {
            if (256 * q >= total) break;
            const int i = tid + 256 * q, r = row_of(i);
            if (i < total) stage[(i - r * lim) * CDB_LD + r] = v[q];
        }
        if ((lim & 1) && tid < CDB_M + CDB_N) stage[lim * CDB_LD + tid] = 0.f;  // (an odd row's last pair; KC is even)
        __syncthreads();
        const float* sX = stage + ty * 8;
        const float* sY = stage + CDB_M + tx * 4;
#pragma unroll
        for (int k = 0; k < KC; ++k) {
            if ((k & 1) == 0 && k >= lim) break;
            const floatx4 x0 = *reinterpret_cast<const floatx4*>(sX + k * CDB_LD), x1 = *reinterpret_cast<const floatx4*>(sX + k * CDB_LD + 4);
            const floatx4 y = *reinterpret_cast<const floatx4*>(sY + k * CDB_LD);
#pragma unroll
            for (int a = 0; a < 8; ++a)
#pragma unroll
                for (int b = 0; b < 4; ++b) {
                    const float df = (a < 4 ? x0[a & 3] : x1[a & 3]) - y[b];
                    acc[a][b] = fmaf(df, df, acc[a][b]);
                }
        }
    }
#pragma unroll
    for (int half = 0; half < 2; ++half) {
        float t[4][4];
#pragma unroll
        for (int a = 0; a < 4; ++a)
#pragma unroll
            for (int b = 0; b < 4; ++b) t[a][b] = acc[4 * half + a][b];
        if (gauss != 0.f) {
#pragma unroll
            for (int a = 0; a < 4; ++a)
#pragma unroll
                for (int b = 0; b < 4; ++b) t[a][b] = cd_exp(-t[a][b] * gauss);
        } else if (sqrt_flag) {
            cd_sqrt_block(t);
        }
#pragma unroll
        for (int a = 0; a < 4; ++a)
#pragma unroll
            for (int b = 0; b < 4; ++b) acc[4 * half + a][b] = t[a][b];
    }
    const int64_t gj0 = j0 + tx * 4, gi0 = i0 + ty * 8;
    const bool vec4 = vec_out && gj0 + 3 < Nn;
#pragma unroll
    for (int a = 0; a < 8; ++a) {
        if (gi0 + a >= M) continue;
        float* row = out + (gi0 + a) * ldo + gj0;
        if (vec4) {
            store_row4(row, acc[a]);
        } else {
#pragma unroll
            for (int b = 0; b < 4; ++b)
                if (gj0 + b < Nn) row[b] = acc[a][b];
        }
    }
    if (!SYM || tn >= 2 * tm) return;
    if (vec_out && i0 + CDB_M <= M && j0 + CDB_N <= Nn) {
        // whole tiles: turned round in LDS, so that the transpose leaves in rows of 512 bytes
        __syncthreads();
#pragma unroll
        for (int b = 0; b < 4; ++b)
#pragma unroll
            for (int half = 0; half < 2; ++half) {
                const float t[4] = {acc[4 * half][b], acc[4 * half + 1][b], acc[4 * half + 2][b], acc[4 * half + 3][b]};
                store_row4(stage + (tx * 4 + b) * TURN_LD + ty * 8 + 4 * half, t);
            }
        __syncthreads();
        const int c = (tid & 31) * 4;
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            const int r = (tid >> 5) + 8 * q;
            float t[4];
#pragma unroll
            for (int b = 0; b < 4; ++b) t[b] = stage[r * TURN_LD + c + b];
            store_row4(out + (j0 + r) * ldo + i0 + c, t);
        }
    } else {
#pragma unroll
        for (int b = 0; b < 4; ++b) {
            if (gj0 + b >= Nn) continue;
            float* row = out + (gj0 + b) * ldo + gi0;
#pragma unroll
            for (int a = 0; a < 8; ++a)
                if (gi0 + a < M) row[a] = acc[a][b];
        }
    }
}

template <typename T>
static int launch_cdist_t(const T* X, int64_t M, int64_t ldx, const T* Y, int64_t Nn, int64_t ldy,
                          int32_t D, T* out, int64_t ldo, int32_t metric, int32_t sqrt_flag, T gauss,
                          hipStream_t st) {
    const int64_t tiles_m = (M + CD_T - 1) / CD_T, tiles_n = (Nn + CD_T - 1) / CD_T;
    const bool vec_out = aligned16(out) && ldo % 4 == 0;
    // One triangle, stored twice, where the arithmetic outweighs the second store: in pieces of 16 bytes, or element by
    // element into rows of no whole 16-byte groups.  Least number of fp32 features, with times of 20 000 (19 999) rows, whole
    // and as a triangle: Euclidean and Gaussian 5 (9) -- 3 features 0.37, 0.37 ms, 3000 rows 19, 21 us; 6: 0.49, 0.39 (7: 0.79, 0.77;
    // 9: 0.95, 0.80) -- the expansion and absolute differences 9 (17) -- expansion of 8: 0.40, 0.41; 9: 0.47, 0.42 (7: 0.72, 0.79;
    // 15: 0.82, 0.84), differences of 8: 0.35, 0.39; 9: 0.40, 0.39 (12: 0.76, 0.81; 18: 0.97, 0.87).  float64 always: 10 000 rows of 2
    // 0.29, 0.27; of 18 0.44, 0.34.
    const int least = sizeof(T) == 8 ? 1 : metric == 1 ? (vec_out ? 5 : 9) : (vec_out ? 9 : 17);
    const bool sym = X == Y && M == Nn && ldx == ldy && D >= least;
    if constexpr (sizeof(T) == 4) {
        // Large tiles where they are enough to fill the chip several times over and the arithmetic does not hide the rest
        // anyway: 20 000 rows, triangle, of 6 features 369 -> 318 us, 9: 388 -> 300, 25: 526 -> 463, 48: 711 -> 677, 64: 802 -> 845;
        // whole, of 32: 978 -> 881, 36: 1.05 times as fast, 48: 1118 -> 1175; 5 000 of 18: 37 and 39.  Not where
        //   a triangle's transpose goes out element by element (19 999 of 18: 829 and 857), or in rows that begin in the middle of a line of
        //   128 bytes, which up to 16 features do not hide (30 000 of 8: 920 -> 1027, 39 952 of 5 to 16: 0.84 to 0.97 times as fast, of
        //   17: 1.21); begun at a quarter of one, from 20 000 rows on (30 024: 0.95 to 1.03; 16 040: 1.01 to 1.04).  Rows at the other
        //   multiples of 16 bytes pay: 9 004 1.07 to 1.22, 30 028 1.01 to 1.10, 39 948 1.07 to 1.11;
        //   few features are written element by element (24 003 x 24 003 of 5: 0.88 times as fast, of 9: 1.06);
        //   a matrix does not fill the tiles (10 x 2M of 16: 129 -> 246; 300 x 300 000 of 32: 207 -> 244; 512 x 39 000 of 18: 42 -> 54; 900 x
        //   39 000 of 16: 0.92 times as fast, 1000 x 39 000 of 6: 1.23, of 16: 0.98, of 18: 1.12; 2M x 10 of 16: 134 -> 149; 1M x 64 of 16:
        //   118 -> 103);
        //   more than 24 features meet a whole matrix of few tiles (7000 x 7000 of 32: 103 -> 107, 9000 x 9000: 1.22 times as fast; of 33:
        //   7000 x 7000 0.94, 9004 x 12 008 1.32, 12 000 x 12 000 1.09).
        const int64_t bm = (M + CDB_M - 1) / CDB_M, bn = (Nn + CDB_N - 1) / CDB_N, big = sym ? bm * (bm + 1) : bm * bn;
        const bool lines = ldo % 32 == 0 || ldo % 8 != 0 || (ldo % 16 != 0 && M < 20000);
        const bool fits = sym ? vec_out && D <= 48 && (D > 16 || lines) : D <= 36 && (vec_out || D > 8) && M >= 960 && Nn >= CDB_N;
        if (metric == 1 && D > 4 && fits && big >= (sym || D <= 24 ? 1 : D <= 32 ? 2 : 3) * CDB_LEAST && big <= 0x7fffffffLL) {
#define HKM_BIG(KC)                                                                                                          \
    do {                                                                                                                     \
        if (sym)                                                                                                             \
            hipLaunchKernelGGL((cdist_big_kernel<KC, true>), dim3((unsigned)big), dim3(256), 0, st, X, M, ldx, Y, Nn, ldy, D, out, \
                               ldo, sqrt_flag, gauss, bn, vec_out);                                                          \
        else                                                                                                                 \
            hipLaunchKernelGGL((cdist_big_kernel<KC, false>), dim3((unsigned)big), dim3(256), 0, st, X, M, ldx, Y, Nn, ldy, D, out, \
                               ldo, sqrt_flag, gauss, bn, vec_out);                                                          \
    } while (0)
            if (D <= 8) HKM_BIG(8);
            else if (D > 16) HKM_BIG(24);
            else HKM_BIG(16);
#undef HKM_BIG
            return check_launch("cdist_big_kernel");
        }
    }
    const int64_t total = sym ? tiles_m * (tiles_m + 1) / 2 : tiles_m * tiles_n;
    if (total > 0x7fffffffLL) return fail(HKM_EUNSUPPORTED, "cdist: %lld tiles exceed the grid limit", (long long)total);
#define HKM_GO2(MET, KU, SYM)                                                                                      \
    hipLaunchKernelGGL((cdist_kernel<T, MET, KU, SYM>), dim3((unsigned)total), dim3(256), 0, st, X, M, ldx, Y, Nn, \
                       ldy, D, out, ldo, sqrt_flag, gauss, tiles_n, vec_out)
#define HKM_GO1(MET, KU)              \
    do {                              \
        if (sym) HKM_GO2(MET, KU, true); \
        else HKM_GO2(MET, KU, false); \
    } while (0)
#define HKM_GO(MET)                  \
    do {                             \
        if (D <= 4) HKM_GO1(MET, 4); \
        else if (D <= 8) HKM_GO1(MET, 8); \
        else if (D <= 16) HKM_GO1(MET, 16); \
        else HKM_GO1(MET, 32);       \
    } while (0)
    if (metric == 0) HKM_GO(0);
    else if (metric == 1) HKM_GO(1);
    else HKM_GO(2);
#undef HKM_GO
#undef HKM_GO1
#undef HKM_GO2
    return check_launch("cdist_kernel");
}

int launch_cdist(const float* X, int64_t M, int64_t ldx, const float* Y, int64_t Nn, int64_t ldy,
                 int32_t D, float* out, int64_t ldo, int32_t metric, int32_t sqrt_flag, float gauss,
                 hipStream_t st) {
    // the quadratic expansion is a matrix product: matrix cores from 16 features on
    if (metric == 0 && cdist_mfma_eligible(M, Nn, D, ldx, ldy, ldo))
        return launch_cdist_mfma(X, M, ldx, Y, Nn, ldy, D, out, ldo, sqrt_flag, gauss, st);
    return launch_cdist_t<float>(X, M, ldx, Y, Nn, ldy, D, out, ldo, metric, sqrt_flag, gauss, st);
}

int launch_cdist_f64(const double* X, int64_t M, int64_t ldx, const double* Y, int64_t Nn, int64_t ldy,
                     int32_t D, double* out, int64_t ldo, int32_t metric, int32_t sqrt_flag, double gauss,
                     hipStream_t st) {
    return launch_cdist_t<double>(X, M, ldx, Y, Nn, ldy, D, out, ldo, metric, sqrt_flag, gauss, st);
}

}  // namespace hkm
