// The 2D FFTLog covariance integrals as contractions over the k grid (gfx950, FP64 MFMA).
//
// For a diagonal input d_t every node of the 2D transform (cov_kernels.hip) is
//     row_i(j) = Re sum_t d_t Ahat(i + t) Bhat(j + t),
// Ahat the inverse DFT of the first axis' array, Bhat(q) = sum_{n <= N/2} c_n B[n]
// e^{+2 pi i n q/N} with c = 1 at the two ends and 2 between (FFTW's c2r written out:
// it drops the imaginary parts of the two end terms, which the real part does here).  The
// bicubic's row and column functionals act on i and on j alone, so with
//     A_m(t) = sum_i U_m(i) / r_i^nu Ahat(i + t),   B_n(t) = sum_j V_n(j) Bhat(j + t)
// (spectrum independent, folded once per plan by k_cov_fold) an integral is
//     value(m, n) = sum_t d_t K(t; m, n),  K = Re(A_m(t) B_n(t)):
// two real products and one sum over t per (m, n), in place of two FFTs for each of the
// ~70 transform rows that a separation's bicubic touches.  Two ways to put it on the
// matrix cores (v_mfma_f64_16x16x4):
//   k_cov_many   rows = 16 diagonals (spectra x powers), columns = 16 m of one n, K formed in
//                registers as the B operand: 2 N flops per (diagonal, m, n), but diagonals
//                are padded to 16;
//   k_cov_few    rows = 16 n, columns = 16 m of one diagonal, the real and the imaginary
//                products as two instructions: 4 N flops, no padding of the diagonals.
// and their transposes k_cov_many_T / k_cov_few_T (sums over (m, n) for each t).
// The instruction reaches 76 TFLOP/s here.  Measured, against the row transforms they replace:
// 64 spectra, N = 8000, 256 separations 12.9 against 120 ms (63 TFLOP/s; the adjoint 14.0 against
// 126 ms), 8 spectra, N = 6000, 150 separations 0.68 against 10.9 ms (adjoint 0.65 against 13.5),
// one spectrum, N = 8000, 100 separations 0.12 against 1.9 ms.  What is left of the rate in
// k_cov_many goes to forming K, which shares the FP64 pipes with the MFMAs (four FP64
// operations for ST MFMAs: 55 TFLOP/s at ST = 1, 63 at 2; 62 at 4, where one wave fits a SIMD).
//
// Operand loads: an instruction reads 16 rows x 4 contracted elements, one per lane (row q =
// lane % 16, elements by g = lane / 16), and rows of an (m, t) array are far apart, which costs the
// L1 an access per lane (k_cov_few was bound by them: 214 us, 130 with fragments; k_cov_many's
// loads take 16 accesses now, the least for 1 KB).  The contracted index may run in any order, so
// the tables and the diagonals are stored as fragments: 16 x 16 blocks in the order
// [half][lane][2], lane (q, g) holding t = 4 g ... 4 g + 3 of its row in two 16-byte loads that
// read 1 KB each.  The transposes read plain rows (k_cov_unfold) with their lanes along t.
#include <hip/hip_runtime.h>

#include <utility>

#include "ce_internal.h"

namespace {

typedef double v4d __attribute__((ext_vector_type(4)));
typedef double v2d __attribute__((ext_vector_type(2)));
typedef v4d v4d_u __attribute__((aligned(8)));   // rows of odd length start on 8 bytes

// a lane's four elements of a fragment, p = the fragment + 2 lane; and of a plain row
__device__ __forceinline__ v4d ldf(const double *p)
{
    const v2d a = *(const v2d *)p, b = *(const v2d *)(p + 128);
    return (v4d){a[0], a[1], b[0], b[1]};
}
__device__ __forceinline__ v4d ld4u(const double *p) { return *(const v4d_u *)p; }

// the instruction's result: element i of a lane is row g + 4 i, column lane % 16
__device__ __forceinline__ int crow(int g, int i) { return g + 4 * i; }

__device__ __forceinline__ v4d mfma(double a, double b, v4d c)
{
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

// tab[l][part][m / 16][t / 16] fragments, part = Re A, Im A, Re B, -Im B; rows R..Rp and columns
// N..Np are zero.  A workgroup makes 16 m x 64 t of the four parts: a wave takes one m at a
// time with its lanes along t (uniform weights, contiguous grid values), LDS turns the
// values into fragments.
__global__ void __launch_bounds__(256) k_cov_fold(int N, int Np, int R, int Rp, const double2 *__restrict__ ahat,
                                                  const double2 *__restrict__ bhat, const int *__restrict__ lo,
                                                  const int *__restrict__ cnt, const int *__restrict__ off,
                                                  const double *__restrict__ uw, const double *__restrict__ fws,
                                                  const double *__restrict__ prn, double *__restrict__ tab)
{
    __shared__ double buf[4][16][65];
    const int tid = threadIdx.x, tx = tid & 63;
    const int t0 = blockIdx.x * 64, mt = blockIdx.y, l = blockIdx.z;
    const double2 *a = ahat + (int64_t)l * N, *b = bhat + (int64_t)l * N;
    for (int r = tid >> 6; r < 16; r += 4) {
        const int m = mt * 16 + r, t = t0 + tx;
        double ar = 0.0, ai = 0.0, br = 0.0, bi = 0.0;
        if (t < N && m < R) {
            const int j0 = lo[m], c = cnt[m], o = off[m];
            for (int q = 0; q < c; ++q) {
                int i = j0 + q + t;   // < 2 N
                if (i >= N) i -= N;
                const double wa = uw[o + q] / prn[j0 + q], wb = fws[o + q];
                ar += wa * a[i].x;
                ai += wa * a[i].y;
                br += wb * b[i].x;
                bi -= wb * b[i].y;
            }
        }
        buf[0][r][tx] = ar;
        buf[1][r][tx] = ai;
        buf[2][r][tx] = br;
        buf[3][r][tx] = bi;
    }
    __syncthreads();
    const int64_t S = (int64_t)Rp * Np;
    const int half = tid >> 7, g = (tid >> 5) & 3, q = (tid >> 1) & 15, sub = tid & 1;
    for (int f = 0; f < 4; ++f) {
        if (t0 + 16 * f >= Np) break;
        double *p = tab + (int64_t)l * 4 * S + ((int64_t)mt * (Np / 16) + t0 / 16 + f) * 256 + tid;
#pragma unroll
        for (int c = 0; c < 4; ++c) p[c * S] = buf[c][q][16 * f + 4 * g + 2 * half + sub];
    }
}

// the fragments as plain rows [l][part][m][t], which the adjoint reads with its lanes along t
__global__ void __launch_bounds__(256) k_cov_unfold(int Np, int64_t n, const double *__restrict__ tab,
                                                    double *__restrict__ rows)
{
    const int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;   // a row element
    if (e >= n) return;
    const int t = (int)(e % Np);
    const int64_t m = e / Np;
    rows[e] = tab[((m >> 4) * (Np / 16) + (t >> 4)) * 256 + ((t >> 1) & 1) * 128 + (((t >> 2) & 3) * 16 + (m & 15)) * 2 +
                  (t & 1)];
}

struct con_args {
    int Np, R, Rp, npair, nblk, nsplit;
    const int *pl1, *pl2;    // [npair] multipole slots
    const double *tab;
    const double *d;         // [nblk / 16][Np / 16] fragments
    const double *fac;       // [2][npair]
    int unit0, units;        // k_cov_few: the (diagonal, pair) units of this launch
    double *out;             // k_cov_many: [nsplit][nblk][npair][R][R], (m, n) at R n + m, scaled when
                             // nsplit = 1; k_cov_few: [nsplit][units][R][R]
};

// the fragments of rows 16 mt ... 16 mt + 15
__device__ __forceinline__ const double *tab_frag(const con_args &a, int l, int part, int mt)
{
    return a.tab + (((int64_t)l * 4 + part) * a.Rp + 16 * mt) * a.Np;
}

// steps of 16 t of split z: [s0, s1)
__device__ __forceinline__ void split_range(int steps, int nsplit, int z, int &s0, int &s1)
{
    const int per = (steps + nsplit - 1) / nsplit;
    s0 = min(z * per, steps);
    s1 = min(s0 + per, steps);
}

// lane J of each 16-lane row, in all of that row's lanes
template <int J>
__device__ __forceinline__ double row_bcast(double v)
{
    const long long x = __builtin_bit_cast(long long, v);
    const long long y = __builtin_amdgcn_update_dpp((long long)0, x, 0x150 + J, 0xf, 0xf, true);   // row_newbcast
    return __builtin_bit_cast(double, y);
}

// element i of the step for column n = n0 + J of k_cov_many: K from A (this lane's m) and lane
// J's B, then its MFMAs
template <int ST, int J>
__device__ __forceinline__ void many_col(int i, const v4d *A, const v4d *B, const v4d *d, v4d (*acc)[ST], int nj)
{
    if (J >= nj) return;   // wave-uniform: columns past R
    const double K = A[0][i] * row_bcast<J>(B[0][i]) + A[1][i] * row_bcast<J>(B[1][i]);
#pragma unroll
    for (int s = 0; s < ST; ++s) acc[J][s] = mfma(d[s][i], K, acc[J][s]);
}
// the columns inside, so that consecutive MFMAs add to different accumulators
template <int ST, int... J>
__device__ __forceinline__ void many_cols(std::integer_sequence<int, J...>, const v4d *A, const v4d *B, const v4d *d,
                                          v4d (*acc)[ST], int nj)
{
#pragma unroll
    for (int i = 0; i < 4; ++i) (many_col<ST, J>(i, A, B, d, acc, nj), ...);
}

// 16 ST diagonals x 16 m x Q = 16 / ST n per wave.  Per step of 16 t a lane loads its m's A and
// one n's B (row broadcasts hand the n's round) and ST diagonals, 4 + ST loads of 32 bytes,
// for 64 MFMAs; the next step's loads are issued before them.  Workgroups of one tile's
// diagonal groups, and of neighbouring tiles (which share A), go to one XCD.
template <int ST>
__global__ void __launch_bounds__(256, 2) k_cov_many(con_args a)
{
    constexpr int Q = 16 / ST;
    const int lane = threadIdx.x & 63, q16 = lane & 15, g = lane >> 4;
    const int NB = (a.R + Q - 1) / Q, NT = a.Rp / 16;
    const int ntile = a.npair * NT * NB;
    const int ng = (a.nblk + 16 * ST - 1) / (16 * ST);
    const int per = ((ntile + 3) / 4 + 7) / 8;   // workgroups of tiles per XCD
    const int xcd = blockIdx.x & 7, k = blockIdx.x >> 3;
    const int e = (xcd * per + k / ng) * 4 + (int)(threadIdx.x >> 6);
    if (e >= ntile) return;
    const int n0 = (e % NB) * Q, mt = e / NB % NT, m = mt * 16 + q16, pr = e / NB / NT;
    const int b0 = (k % ng) * ST * 16;
    const int nj = min(Q, a.R - n0);
    const double *pa[2], *pb[2], *pd[ST];
#pragma unroll
    for (int c = 0; c < 2; ++c) {
        pa[c] = tab_frag(a, a.pl1[pr], c, mt) + 2 * lane;
        // row n0 + q16 % Q in lane q16
        pb[c] = tab_frag(a, a.pl2[pr], 2 + c, n0 >> 4) + 2 * (16 * g + (n0 & 15) + q16 % Q);
    }
#pragma unroll
    for (int s = 0; s < ST; ++s)
        pd[s] = a.d + (int64_t)min(b0 / 16 + s, (a.nblk - 1) / 16) * 16 * a.Np + 2 * lane;
    v4d acc[Q][ST];
#pragma unroll
    for (int j = 0; j < Q; ++j)
#pragma unroll
        for (int s = 0; s < ST; ++s) acc[j][s] = (v4d){0.0, 0.0, 0.0, 0.0};
    int s0, s1;
    split_range(a.Np / 16, a.nsplit, blockIdx.z, s0, s1);
    v4d An[2], Bn[2], dn[ST];
    auto load = [&](int t) {
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            An[c] = ldf(pa[c] + t * 256);
            Bn[c] = ldf(pb[c] + t * 256);
        }
#pragma unroll
        for (int s = 0; s < ST; ++s) dn[s] = ldf(pd[s] + t * 256);
    };
    if (s0 < s1) load(s0);
    for (int t = s0; t < s1; ++t) {
        v4d A[2], B[2], d[ST];
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            A[c] = An[c];
            B[c] = Bn[c];
        }
#pragma unroll
        for (int s = 0; s < ST; ++s) d[s] = dn[s];
        load(min(t + 1, s1 - 1));
        many_cols<ST>(std::make_integer_sequence<int, Q>(), A, B, d, acc, nj);
    }
    if (m >= a.R) return;
    const int64_t RR = (int64_t)a.R * a.R;
#pragma unroll
    for (int s = 0; s < ST; ++s)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int b = b0 + 16 * s + crow(g, i);
            if (b >= a.nblk) continue;
            const double f = a.nsplit == 1 ? a.fac[(b & 1) * a.npair + pr] : 1.0;
            double *o = a.out + (((int64_t)blockIdx.z * a.nblk + b) * a.npair + pr) * RR + (int64_t)a.R * n0 + m;
#pragma unroll
            for (int j = 0; j < Q; ++j)
                if (j < nj) o[(int64_t)a.R * j] = acc[j][s][i] * f;
        }
}

// one diagonal and pair, a 32 x 32 tile (n, m) per wave; per step of 16 t 32 MFMAs against
// nine 32-byte loads per lane, the next step's issued before them.  nsplit is a multiple of the 8
// XCDs, each of which has its own ranges of t, so that its L2 holds the tables' part that
// all pairs and tiles of a range read (also where the tiles alone fill the chip: 4 spectra, 400
// separations, N = 8000: 5.0 ms in 8 splits, 7.2 in one).
__global__ void __launch_bounds__(256, 2) k_cov_few(con_args a)
{
    const int lane = threadIdx.x & 63, q16 = lane & 15, g = lane >> 4;
    const int E = (a.R + 31) / 32, wu = (E * E + 3) / 4;
    const int W = wu * a.units;   // workgroups per split
    const int x = (int)blockIdx.x;
    const int id = (x >> 3) % W;
    const int z = (x >> 3) / W * 8 + (x & 7);
    const int w = id % wu * 4 + (int)(threadIdx.x >> 6);
    const int unit = id / wu, bp = a.unit0 + unit;
    if (w >= E * E) return;
    const int m0 = (w % E) * 32, n0 = (w / E) * 32;
    const int pr = bp % a.npair, b = bp / a.npair;
    const bool m2 = m0 + 16 < a.R, n2 = n0 + 16 < a.R;   // wave-uniform: tiles past R
    const double *pa[2][2], *pb[2][2];
    const double *pd = a.d + (int64_t)(b >> 4) * 16 * a.Np + 2 * (16 * g + (b & 15));
    const int last = a.Rp / 16 - 1;
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            pa[h][c] = tab_frag(a, a.pl1[pr], c, min(m0 / 16 + h, last)) + 2 * lane;
            pb[h][c] = tab_frag(a, a.pl2[pr], 2 + c, min(n0 / 16 + h, last)) + 2 * lane;
        }
    v4d acc[2][2];
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[h][j] = (v4d){0.0, 0.0, 0.0, 0.0};
    int s0, s1;
    split_range(a.Np / 16, a.nsplit, z, s0, s1);
    v4d An[2][2], Bn[2][2], dn;
    auto load = [&](int t) {
        dn = ldf(pd + t * 256);
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int c = 0; c < 2; ++c) {
                An[h][c] = ldf(pa[h][c] + t * 256);
                Bn[h][c] = ldf(pb[h][c] + t * 256);
            }
    };
    if (s0 < s1) load(s0);
    for (int t = s0; t < s1; ++t) {
        v4d A[2][2], B[2][2];
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int c = 0; c < 2; ++c) {
                A[h][c] = An[h][c] * dn;
                B[h][c] = Bn[h][c];
            }
        load(min(t + 1, s1 - 1));
#pragma unroll
        for (int c = 0; c < 2; ++c)
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int h = 0; h < 2; ++h)
#pragma unroll
                    for (int j = 0; j < 2; ++j)
                        if (!((h && !n2) || (j && !m2))) acc[h][j] = mfma(B[h][c][i], A[j][c][i], acc[h][j]);
    }
    double *o = a.out + ((int64_t)z * a.units + unit) * a.R * a.R;
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int n = n0 + 16 * h + crow(g, i), m = m0 + 16 * j + q16;
                if (n < a.R && m < a.R) o[(int64_t)a.R * n + m] = acc[h][j][i];
            }
}

// out = fac sum_z part[z], the splits in order; the n values of units unit0, unit0 + 1, ...
__global__ void __launch_bounds__(256) k_cov_sum(int64_t n, int64_t RR, int npair, int nsplit, int unit0,
                                                 const double *__restrict__ part, const double *__restrict__ fac,
                                                 double *__restrict__ out)
{
    const int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (e >= n) return;
    double s = part[e];
    for (int z = 1; z < nsplit; ++z) s += part[z * n + e];
    const int64_t bp = unit0 + e / RR;
    out[unit0 * RR + e] = s * fac[((bp / npair) & 1) * npair + bp % npair];
}

#define CE_FEW_T_N 64      // n per wave of k_cov_few_T

struct conT_args {
    int Np, R, Rp, npair, nblk, nsplit;
    const int *pl1, *pl2;
    const double *tab;       // plain rows [nl][4][Rp][Np]
    const double *gint;      // [nblk][npair][R][R]
    const double *fac;
    double *part;            // [nsplit][nblk][Np]
};

// sums over (pair, m, n) for 16 ST diagonals (rows) and 64 t (columns) per wave.  A wave keeps
// the A of 16 m and its t in registers and runs over n: per n two B values per t and the
// diagonals' cotangents of the 16 m (the A operand) feed 16 ST MFMAs, K formed as the B
// operand; the next n's loads are issued before them.
template <int ST>
__global__ void __launch_bounds__(256, 2) k_cov_many_T(conT_args a)
{
    constexpr int Q = 4;
    const int lane = threadIdx.x & 63, q16 = lane & 15, g = lane >> 4;
    const int w = (int)(blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6));
    const int ntile = a.Np / 16;
    if (w * Q >= ntile) return;
    const int b0 = blockIdx.y * ST * 16;
    const int64_t S = (int64_t)a.Rp * a.Np, RR = (int64_t)a.R * a.R;
    int t[Q];
#pragma unroll
    for (int q = 0; q < Q; ++q) t[q] = min(w * Q + q, ntile - 1) * 16 + q16;
    const double *pg[ST];
#pragma unroll
    for (int s = 0; s < ST; ++s) pg[s] = a.gint + (int64_t)min(b0 + 16 * s + q16, a.nblk - 1) * a.npair * RR + 4 * g;
    const int pw = q16 & 1;   // the power of a row's diagonal (16 s is even; padded rows are not stored)
    v4d acc[ST][Q];
#pragma unroll
    for (int s = 0; s < ST; ++s)
#pragma unroll
        for (int q = 0; q < Q; ++q) acc[s][q] = (v4d){0.0, 0.0, 0.0, 0.0};
    int e, e1;   // (pair, m tile, n), n fastest
    split_range(a.npair * (a.Rp / 16) * a.R, a.nsplit, blockIdx.z, e, e1);
    while (e < e1) {
        const int u = e / a.R, m0 = u % (a.Rp / 16) * 16, pr = u / (a.Rp / 16);
        int n = e % a.R;
        const int n1 = min(a.R, n + e1 - e);
        e += n1 - n;
        const double *tA = a.tab + (int64_t)a.pl1[pr] * 4 * S + (int64_t)(m0 + 4 * g) * a.Np;
        const double *tB = a.tab + ((int64_t)a.pl2[pr] * 4 + 2) * S;
        double ar[Q][4], ai[Q][4];
#pragma unroll
        for (int q = 0; q < Q; ++q)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                ar[q][i] = tA[(int64_t)i * a.Np + t[q]];
                ai[q][i] = tA[S + (int64_t)i * a.Np + t[q]];
            }
        const double fac = a.fac[pw * a.npair + pr];
        const bool whole = m0 + 16 <= a.R;
        double brn[Q], bin[Q];
        v4d gn[ST];
        auto load = [&](int n) {
#pragma unroll
            for (int q = 0; q < Q; ++q) {
                brn[q] = tB[(int64_t)n * a.Np + t[q]];
                bin[q] = tB[S + (int64_t)n * a.Np + t[q]];
            }
#pragma unroll
            for (int s = 0; s < ST; ++s) {
                const double *G = pg[s] + pr * RR + (int64_t)n * a.R + m0;
                if (whole) {
                    gn[s] = ld4u(G);
                } else {
#pragma unroll
                    for (int i = 0; i < 4; ++i) gn[s][i] = m0 + 4 * g + i < a.R ? G[i] : 0.0;
                }
            }
        };
        load(n);
        for (; n < n1; ++n) {
            double br[Q], bi[Q];
            v4d gv[ST];
#pragma unroll
            for (int q = 0; q < Q; ++q) {
                br[q] = brn[q];
                bi[q] = bin[q];
            }
#pragma unroll
            for (int s = 0; s < ST; ++s) gv[s] = gn[s] * fac;
            load(min(n + 1, n1 - 1));
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int q = 0; q < Q; ++q) {
                    const double K = ar[q][i] * br[q] + ai[q][i] * bi[q];
#pragma unroll
                    for (int s = 0; s < ST; ++s) acc[s][q] = mfma(gv[s][i], K, acc[s][q]);
                }
        }
    }
#pragma unroll
    for (int q = 0; q < Q; ++q) {
        if (w * Q + q >= ntile) break;
#pragma unroll
        for (int s = 0; s < ST; ++s)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int b = b0 + 16 * s + crow(g, i);
                if (b < a.nblk) a.part[((int64_t)blockIdx.z * a.nblk + b) * a.Np + t[q]] = acc[s][q][i];
            }
    }
}

// one diagonal, pair and group of 64 n: X_n(t) = sum_m G(n, m) A_m(t) for the group's n (rows)
// and 32 t (columns), then sum_n Re(X_n B_n) in the lanes that hold them; per 16 m 64 MFMAs
// against four 32-byte and sixteen 8-byte loads per lane
__global__ void __launch_bounds__(256, 2) k_cov_few_T(conT_args a)
{
    constexpr int H = CE_FEW_T_N / 16;
    const int lane = threadIdx.x & 63, q16 = lane & 15, g = lane >> 4;
    const int w = (int)(blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6));
    const int ntile = a.Np / 16;
    if (w * 2 >= ntile) return;
    const int pr = blockIdx.y % a.npair, b = blockIdx.y / a.npair, n0 = blockIdx.z * CE_FEW_T_N;
    const int64_t S = (int64_t)a.Rp * a.Np, RR = (int64_t)a.R * a.R;
    int t[2];
#pragma unroll
    for (int q = 0; q < 2; ++q) t[q] = min(w * 2 + q, ntile - 1) * 16 + q16;
    const double *tA = a.tab + (int64_t)a.pl1[pr] * 4 * S + (int64_t)(4 * g) * a.Np;
    const double *tB = a.tab + ((int64_t)a.pl2[pr] * 4 + 2) * S;
    const double *G = a.gint + ((int64_t)b * a.npair + pr) * RR;
    const double *gp[H];
#pragma unroll
    for (int h = 0; h < H; ++h) gp[h] = G + (int64_t)min(n0 + 16 * h + q16, a.R - 1) * a.R + 4 * g;
    v4d X[H][2][2];
#pragma unroll
    for (int h = 0; h < H; ++h)
#pragma unroll
        for (int c = 0; c < 2; ++c)
#pragma unroll
            for (int q = 0; q < 2; ++q) X[h][c][q] = (v4d){0.0, 0.0, 0.0, 0.0};
    for (int m0 = 0; m0 < a.R; m0 += 16) {
        double v[4][2][2];
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int c = 0; c < 2; ++c)
#pragma unroll
                for (int q = 0; q < 2; ++q) v[i][c][q] = tA[c * S + (int64_t)(m0 + i) * a.Np + t[q]];
        v4d gv[H];
#pragma unroll
        for (int h = 0; h < H; ++h) {
            if (m0 + 16 <= a.R) {
                gv[h] = ld4u(gp[h] + m0);
            } else {
#pragma unroll
                for (int i = 0; i < 4; ++i) gv[h][i] = m0 + 4 * g + i < a.R ? gp[h][m0 + i] : 0.0;
            }
        }
#pragma unroll
        for (int h = 0; h < H; ++h) {
            if (n0 + 16 * h >= a.R) break;   // wave-uniform
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int c = 0; c < 2; ++c)
#pragma unroll
                    for (int q = 0; q < 2; ++q) X[h][c][q] = mfma(gv[h][i], v[i][c][q], X[h][c][q]);
        }
    }
    double sum[2] = {0.0, 0.0};
#pragma unroll
    for (int h = 0; h < H; ++h)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int n = n0 + 16 * h + crow(g, i);
            if (n < a.R)
#pragma unroll
                for (int q = 0; q < 2; ++q) {
                    const double *p = tB + (int64_t)n * a.Np + t[q];
                    sum[q] += X[h][0][q][i] * p[0] + X[h][1][q][i] * p[S];
                }
        }
    const double fac = a.fac[(b & 1) * a.npair + pr];
#pragma unroll
    for (int q = 0; q < 2; ++q) {
        double v = sum[q];
        v += __shfl_xor(v, 16);
        v += __shfl_xor(v, 32);
        if (g == 0 && w * 2 + q < ntile)
            a.part[(((int64_t)blockIdx.z * a.npair + pr) * a.nblk + b) * a.Np + t[q]] = v * fac;
    }
}

// dbar[b][t] = sum_z part[z][b][t]
__global__ void __launch_bounds__(256) k_cov_sum_T(int N, int Np, int nblk, int nsplit,
                                                   const double *__restrict__ part, double *__restrict__ dbar)
{
    const int t = blockIdx.x * blockDim.x + threadIdx.x, b = blockIdx.y;
    if (t >= N) return;
    double s = 0.0;
    for (int z = 0; z < nsplit; ++z) s += part[((int64_t)z * nblk + b) * Np + t];
    dbar[(int64_t)b * N + t] = s;
}

// 16 x ceil(nblk / 16) padded diagonals at 2 N flops each against nblk at 4 N
bool many(int nblk) { return 16 * ((nblk + 15) / 16) < 2 * nblk; }

// splits of the contracted range.  The chip holds 2048 waves of these kernels at once (2 on each
// of 1024 SIMDs); n splits take ceil(waves n / 2048) rounds of ceil(steps / n) steps, and
// each split costs about two steps more (its prologue, its sums).  From 8 on a multiple of
// the 8 XCDs.
int splits(int64_t waves, int steps, int most)
{
    int best = 1;
    double cost = 1e300;
    for (int n = 1; n <= most; n += n < 8 ? 1 : 8) {
        const double c = (double)((waves * n + 2047) / 2048) * ((steps + n - 1) / n + 2) + 2.0 * n;
        if (c < cost) {
            cost = c;
            best = n;
        }
    }
    return best;
}

// 16-row groups per wave: two, unless that pads an odd number of groups by more than forming K
// twice as often costs (35 against 31 TFLOP/s at 3 groups; 63 against 55 at 8)
int many_st(int nblk)
{
    const int S = (nblk + 15) / 16;
    return S % 2 && S < 7 ? 1 : 2;
}

int64_t many_tiles(int nblk, int npair, int R)
{
    const int Q = 16 / many_st(nblk);
    return (int64_t)npair * ((R + 15) / 16) * ((R + Q - 1) / Q);
}

int many_groups(int nblk) { return (nblk + 16 * many_st(nblk) - 1) / (16 * many_st(nblk)); }

// The forward's partial sums keep to WORK bytes (the doubles of one unit's splits, 64 R^2 bytes, at the
// least): k_cov_many takes fewer splits, k_cov_few its (diagonal, pair) units in groups.
constexpr int64_t WORK = (int64_t)512 << 20;

int many_splits(int nblk, int npair, int R, int Np)
{
    const int64_t fit = WORK / ((int64_t)8 * nblk * npair * R * R);
    return splits(many_tiles(nblk, npair, R) * many_groups(nblk), Np / 16, fit < 1 ? 1 : (fit > 32 ? 32 : (int)fit));
}

int few_splits(int nblk, int npair, int R, int Np)
{
    const int64_t E = (R + 31) / 32;
    const int64_t waves = (E * E + 3) / 4 * 4 * npair * nblk;
    int n = (int)((3072 + waves - 1) / waves);   // 1.5 waves a SIMD: 130 us at 16 splits of 192 waves, 153 at 8, 135 at 32
    n = (n + 7) / 8 * 8;
    if (n > 32) n = 32;
    while (n > 8 && n > Np / 128) n -= 8;
    return n;
}

// units per launch: as many as WORK holds, the launches alike
int few_units(int nblk, int npair, int R, int nsplit)
{
    const int64_t all = (int64_t)nblk * npair, fit = WORK / ((int64_t)8 * nsplit * R * R);
    const int64_t most = fit < 1 ? 1 : fit;
    return (int)((all + (all + most - 1) / most - 1) / ((all + most - 1) / most));
}

}  // namespace

extern "C" size_t ce_cov_contract_work(int nblk, int npair, int R, int Np)
{
    const size_t RR = (size_t)R * R;
    if (many(nblk)) {
        const int n = many_splits(nblk, npair, R, Np);
        return n > 1 ? (size_t)n * nblk * npair * RR : 0;
    }
    const int n = few_splits(nblk, npair, R, Np);
    return (size_t)n * few_units(nblk, npair, R, n) * RR;
}

extern "C" int ce_cov_contract_splits_T(int nblk, int npair, int R, int Np)
{
    if (!many(nblk)) return npair * ((R + CE_FEW_T_N - 1) / CE_FEW_T_N);
    const int64_t waves = (int64_t)((Np / 16 + 3) / 4 + 3) / 4 * 4 * many_groups(nblk);
    return splits(waves, npair * ((R + 15) / 16) * R, 64);
}

extern "C" int ce_launch_cov_fold(void *stream, int nl, int N, int Np, int R, int Rp, const double *d_ahat,
                                  const double *d_bhat, const int *d_lo, const int *d_cnt, const int *d_off,
                                  const double *d_uw, const double *d_fws, const double *d_prn, double *d_tab)
{
    hipLaunchKernelGGL(k_cov_fold, dim3((Np + 63) / 64, Rp / 16, nl), dim3(256), 0, (hipStream_t)stream, N, Np, R, Rp,
                       reinterpret_cast<const double2 *>(d_ahat), reinterpret_cast<const double2 *>(d_bhat), d_lo,
                       d_cnt, d_off, d_uw, d_fws, d_prn, d_tab);
    return (int)hipGetLastError();
}

extern "C" int ce_launch_cov_unfold(void *stream, int nl, int Np, int Rp, const double *d_tab, double *d_rows)
{
    const int64_t n = (int64_t)nl * 4 * Rp * Np;
    hipLaunchKernelGGL(k_cov_unfold, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, (hipStream_t)stream, Np, n,
                       d_tab, d_rows);
    return (int)hipGetLastError();
}

extern "C" int ce_launch_cov_contract(void *stream, int nblk, int Np, int R, int npair, const int *d_pl1,
                                      const int *d_pl2, const double *d_tab, const double *d_d, const double *d_fac,
                                      double *d_part, double *d_out)
{
    const int64_t RR = (int64_t)R * R;
    con_args a;
    a.Np = Np; a.R = R; a.Rp = (R + 15) / 16 * 16; a.npair = npair; a.nblk = nblk;
    a.pl1 = d_pl1; a.pl2 = d_pl2; a.tab = d_tab; a.d = d_d; a.fac = d_fac;
    a.unit0 = 0;
    a.units = nblk * npair;
    hipStream_t s = (hipStream_t)stream;
    auto sum = [&](int unit0, int units) {
        const int64_t n = units * RR;
        hipLaunchKernelGGL(k_cov_sum, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, n, RR, npair, a.nsplit, unit0,
                           d_part, d_fac, d_out);
    };
    if (many(nblk)) {
        a.nsplit = many_splits(nblk, npair, R, Np);
        a.out = a.nsplit == 1 ? d_out : d_part;
        const int64_t wgs = (many_tiles(nblk, npair, R) + 3) / 4;
        const dim3 grid((unsigned)((wgs + 7) / 8 * 8 * many_groups(nblk)), 1, (unsigned)a.nsplit);
        if (many_st(nblk) == 1) hipLaunchKernelGGL(k_cov_many<1>, grid, dim3(256), 0, s, a);
        else hipLaunchKernelGGL(k_cov_many<2>, grid, dim3(256), 0, s, a);
        if (a.nsplit > 1) sum(0, a.units);
        return (int)hipGetLastError();
    }
    a.nsplit = few_splits(nblk, npair, R, Np);
    a.out = d_part;
    const int E = (R + 31) / 32, all = nblk * npair, most = few_units(nblk, npair, R, a.nsplit);
    for (a.unit0 = 0; a.unit0 < all; a.unit0 += most) {
        a.units = all - a.unit0 < most ? all - a.unit0 : most;
        hipLaunchKernelGGL(k_cov_few, dim3((unsigned)((E * E + 3) / 4 * a.units * a.nsplit)), dim3(256), 0, s, a);
        sum(a.unit0, a.units);
    }
    return (int)hipGetLastError();
}

extern "C" int ce_launch_cov_contract_T(void *stream, int nblk, int N, int Np, int R, int npair, const int *d_pl1,
                                        const int *d_pl2, const double *d_tab, const double *d_gint,
                                        const double *d_fac, int nsplit, double *d_part, double *d_dbar)
{
    conT_args a;
    a.Np = Np; a.R = R; a.Rp = (R + 15) / 16 * 16; a.npair = npair; a.nblk = nblk; a.nsplit = nsplit;
    a.pl1 = d_pl1; a.pl2 = d_pl2; a.tab = d_tab; a.gint = d_gint; a.fac = d_fac; a.part = d_part;
    hipStream_t s = (hipStream_t)stream;
    if (many(nblk)) {
        const dim3 grid((unsigned)(((Np / 16 + 3) / 4 + 3) / 4), (unsigned)many_groups(nblk), (unsigned)nsplit);
        if (many_st(nblk) == 1) hipLaunchKernelGGL(k_cov_many_T<1>, grid, dim3(256), 0, s, a);
        else hipLaunchKernelGGL(k_cov_many_T<2>, grid, dim3(256), 0, s, a);
    } else {
        const int waves = (Np / 16 + 1) / 2;
        hipLaunchKernelGGL(k_cov_few_T, dim3((unsigned)((waves + 3) / 4), (unsigned)(npair * nblk),
                                             (unsigned)((R + CE_FEW_T_N - 1) / CE_FEW_T_N)),
                           dim3(256), 0, s, a);
    }
    hipLaunchKernelGGL(k_cov_sum_T, dim3((unsigned)((N + 255) / 256), (unsigned)nblk), dim3(256), 0, s, N, Np, nblk,
                       nsplit, d_part, d_dbar);
    return (int)hipGetLastError();
}
