// Integrated (lensing and potential) terms of the correlation function, full sky, on
// the GPU (gfx950, FP64).
//
// The reference evaluates them with CUBA's Cuhre or GSL Monte Carlo over [0, 1]^2
// (double-integrated, functions.c:3460-4017, signal.c:735-741) and with QAG or a
// double-exponential rule over [0, 1] (single-integrated, functions.c:1486-3458,
// signal.c:578-600).  Here both are deterministic product rules, one workgroup per
// (z_mean, mu, separation):
//   - double: x1 a composite Gauss-Legendre rule on [0, 1] (cut where lambda1 cos(theta)
//     = chi2), and for each x1 the substitution lambda2 = lambda1 c + s sinh(u),
//     s = lambda1 sin(theta), under which r = s cosh(u) and the ridge of closest
//     approach along lambda2 is smooth in u; u a composite Gauss-Legendre rule;
//   - single: the two mixed separations are closest at x = chi1 c / chi2 and chi2 c /
//     chi1; [0, 1] is cut there (and halfway between), each piece mapped by x = centre
//     +- s sinh(u) about its nearer centre (s the ridge width), u Gauss-Legendre.
// Every lookup is the Akima interpolation of the raw nodes (as ce::akima_general; the interval's
// coefficients are made once per call, k_intg_coef) and the renormalisation grid a GSL-style
// bicubic, as the reference's splines.

#include <hip/hip_runtime.h>

#include "ce_device.h"
#include "ce_internal.h"

namespace {

enum { S00, S02, S04, S11, S13, S20, S22, S31, S40, NSLOT };
// background curves with precomputed Akima coefficients: D1, a, f, conformal H against z,
// and z against chi
enum { C_D1, C_A, C_F, C_CH, C_ZOF, NBGC };

constexpr unsigned F_DEN = 1u << 0, F_RSD = 1u << 1, F_D1 = 1u << 2, F_D2 = 1u << 3, F_G1 = 1u << 4,
                   F_G2 = 1u << 5, F_G3 = 1u << 6, F_LEN = 1u << 7, F_G4 = 1u << 8, F_G5 = 1u << 9,
                   F_ONLY_CROSS = 1u << 10, F_FLAT_LL = 1u << 11, F_FLAT_DL = 1u << 12;

// A pointer into device memory that is read from device memory itself: typed, so that the
// loads through it are global ones (through a generic pointer they are flat loads,
// which occupy the LDS path as well and cannot be scalar)
struct gmem {
    const __attribute__((address_space(1))) double *p;
    __host__ __device__ operator const double *() const { return (const double *)p; }
    gmem &operator=(const double *q)
    {
        p = (const __attribute__((address_space(1))) double *)q;
        return *this;
    }
};

struct intg_args {
    int nbg;
    gmem bg_z, bg_chi, bg_D1, bg_a, bg_f, bg_cH, bg_G1, bg_G2;
    int nb;
    gmem bias_z, b1, b2;
    int nmb;
    gmem mb_z, s1, s2, fe1, fe2;
    gmem tab_x, tab_y;
    int tab_off[NSLOT], tab_len[NSLOT];
    int tab_f0[NSLOT];                 // first node of the log-uniform part (-1: bisection)
    int tab_ref;                       // a slot whose nodes every present standard table shares (-1: none)
    double tab_lx0[NSLOT], tab_lsc[NSLOT];   // its log(x[f0]) and nodes per unit of log x
    int nguess;                        // chi -> interval guesses on [0, chi_max], nguess + 1 of them
    gmem chi_guess;
    // Akima value records and node pairs (below)
    gmem tab_val[NSLOT];      // table s's records, tab_stride[s] doubles apart
    int tab_stride[NSLOT];
    gmem tab_pair;            // in the layout of tab_y
    gmem tab_wide;            // the shared-node tables' records, WIDE a node (if tab_ref >= 0)
    gmem bgc_wide, bgz_pair; // D1, a, f, conformal H: BGW a node; bg_z's node pairs
    gmem zof;                 // z against chi: {x_j, x_(j+1), y, b, c, d, 0, 0} a node
    int nren0;
    gmem ren0_x, ren0_y;
    int nren;
    gmem ren_chi;
    gmem ren_rec;   // per grid node (x fastest): {value, d/dx, d/dy, d2/dxdy}
    double Om, H0h;
    unsigned flags;
    int nz, nmu, nsep;
    gmem zmean, mu, sep;
    int p1, n1, pu, nu, ps, ns;
    gmem g1x, g1w, gux, guw, gsx, gsw;   // Gauss-Legendre rules on [-1, 1]
    double *out;                                       // [nz][nmu][nsep][2]: single, double
};

__device__ inline double ak(const double *x, const double *y, int n, double v) { return ce::akima_general(x, y, n, v); }

// An Akima lookup reads two arrays: node pairs {x_j, x_(j+1)} (16 bytes, one load: both
// ends of interval j, which also test a guessed interval), shared by the curves on one
// grid, and each curve's value records {y_j, b_j, c_j, d_j} (32 bytes, two loads).  The
// curves of one grid keep their records side by side: the eight standard tables 256 bytes
// a node (two lines), D1, a, conformal H and f 128 bytes, z(chi) 64 with its node pair, so
// a lookup of all of them moves whole lines, and k_integrated_double fetches them
// a line at a time (below).
constexpr int VAL = CE_INTG_VAL, PAIR = CE_INTG_PAIR, WIDE = CE_INTG_WIDE, BGW = CE_INTG_BGW, ZOF = CE_INTG_ZOF;
// the place of each shared-node table in the record of a node: the two halves are what
// the double integral's fetches take
constexpr int WSLOT[NSLOT - 1] = {0, 3, 5, 2, 4, 1, 7, 6};
struct nodes {
    double x0, x1;
};

__device__ __forceinline__ nodes pair_at(const double *__restrict__ p, int j)
{
    const double2 q = *reinterpret_cast<const double2 *>(p + (size_t)PAIR * j);
    return nodes{q.x, q.y};
}

// whether interval j (0 <= j <= n - 2), whose nodes g holds, is the one
// ce::interval_from returns from the guess j at once (false for a NaN v, whose callers
// then search and get j back)
__device__ __forceinline__ bool pair_hit(const nodes &g, int j, int n, double v)
{
    return g.x0 <= v && (j == n - 2 || v < g.x1);
}

// y(xq) on the segment of record r with lower node x0 (the value akima_at gives there)
__device__ __forceinline__ double cubic(double2 p, double2 q, double dx)
{
    return p.x + dx * (p.y + dx * (q.x + q.y * dx));
}
__device__ __forceinline__ double val_at(const double *__restrict__ r, double x0, double xq)
{
    return cubic(*reinterpret_cast<const double2 *>(r), *reinterpret_cast<const double2 *>(r + 2), xq - x0);
}

// The lookups: Akima of raw nodes as ce::akima_general, with the interval found from a
// guess (the background's redshift grid is uniform; chi(z) through a table of interval
// guesses; the integral tables' FFT nodes are log-uniform) and a short walk, falling
// back to bisection: the same interval, so the same value, in a few dependent loads
// where bisection over 10^4 nodes takes 14.
struct lk {
    const intg_args &a;
    __device__ lk(const intg_args &a_) : a(a_) {}
    __device__ double bg(const double *col, double z) const
    {
        const double *x = a.bg_z;
        const int n = a.nbg;
        if (!(z >= x[0] && z <= x[n - 1])) return __builtin_nan("");
        return ce::akima_at(x, col, n, ce::interval_from(x, n, z, ce::interval_guess(x, n, z)), z);
    }
    static __device__ int below_last(int g, int n) { return g > n - 2 ? n - 2 : g; }
    // the first guess of z's interval on the background's redshift grid (-1 outside it)
    __device__ int bg_guess(double z) const
    {
        const double *x = a.bg_z;
        const int n = a.nbg;
        if (!(z >= x[0] && z <= x[n - 1])) return -1;
        return below_last(ce::interval_guess(x, n, z), n);
    }
    // the interval of z on the redshift grid (-1 outside it), which the curves read at
    // one z share
    __device__ int bg_interval(double z) const
    {
        const int g = bg_guess(z);
        return g < 0 ? -1 : ce::interval_from(a.bg_z, a.nbg, z, g);
    }
    // the node pair of bg_z's interval j, and curve k's value record there
    __device__ nodes bgz(int j) const { return pair_at(a.bgz_pair, j); }
    __device__ const double *bgv(int k, int j) const { return a.bgc_wide + (size_t)BGW * j + VAL * k; }
    // D1, a, f or conformal H (curve k) in interval j (NaN for j < 0)
    __device__ double bgcj(int k, int j, double z) const
    {
        return j < 0 ? __builtin_nan("") : val_at(bgv(k, j), bgz(j).x0, z);
    }
    // curve k at z
    __device__ double bgc(int k, double z) const { return bgcj(k, bg_interval(z), z); }
    // the first guess of chi's interval on bg_chi (-1 outside it)
    __device__ int zof_guess(double chi) const
    {
        const double *x = a.bg_chi;
        const int n = a.nbg;
        if (!(chi >= x[0] && chi <= x[n - 1])) return -1;
        const int k = ce::clamp_index(chi / x[n - 1] * a.nguess, a.nguess + 1);
        return below_last(max((int)a.chi_guess[k], 0), n);
    }
    __device__ double zofj(int j, double chi) const
    {
        const double *r = a.zof + (size_t)ZOF * j;
        return val_at(r + 2, r[0], chi);
    }
    __device__ double z_of(double chi) const
    {
        const int j = zof_guess(chi);
        if (j < 0) return __builtin_nan("");
        const double *r = a.zof + (size_t)ZOF * j;
        const nodes g = pair_at(r, 0);
        if (pair_hit(g, j, a.nbg, chi)) return val_at(r + 2, g.x0, chi);
        return zofj(ce::interval_from(a.bg_chi, a.nbg, chi, j), chi);
    }
    // a first interval of r on table s's nodes (-1: r outside them): by bisection below
    // the log-uniform part (exact), from the log above it (a guess)
    __device__ int tab_guess(int s, double r) const
    {
        const double *x = a.tab_x + a.tab_off[s];
        const int n = a.tab_len[s], f0 = a.tab_f0[s];
        if (!(r >= x[0] && r <= x[n - 1])) return -1;
        if (f0 < 0) return ce::interval_bisect(x, 0, n - 1, r);
        if (r < x[f0]) return ce::interval_bisect(x, 0, f0, r);
        return below_last(f0 + ce::clamp_index((log(r) - a.tab_lx0[s]) * a.tab_lsc[s], n - f0), n);
    }
    __device__ const double *tabv(int s, int j) const { return a.tab_val[s] + (size_t)a.tab_stride[s] * j; }
    __device__ const double *tabp(int s) const { return a.tab_pair + (size_t)PAIR * a.tab_off[s]; }
    // interval j of table s settled from its guess g (-1 stays -1); *x0 its lower node
    __device__ int tab_settle(int s, int g, double r, double *x0) const
    {
        if (g < 0) return g;
        nodes nd = pair_at(tabp(s), g);
        if (!pair_hit(nd, g, a.tab_len[s], r)) {
            g = ce::interval_from(a.tab_x + a.tab_off[s], a.tab_len[s], r, g);
            nd = pair_at(tabp(s), g);
        }
        *x0 = nd.x0;
        return g;
    }
    __device__ double tab(int s, double r) const
    {
        const int g = tab_guess(s, r);
        if (g < 0) return __builtin_nan("");
        const nodes nd = pair_at(tabp(s), g);
        const double v = val_at(tabv(s, g), nd.x0, r);
        if (pair_hit(nd, g, a.tab_len[s], r)) return v;
        const int j = ce::interval_from(a.tab_x + a.tab_off[s], a.tab_len[s], r, g);
        return val_at(tabv(s, j), pair_at(tabp(s), j).x0, r);
    }
    // the interval of r on the standard tables' shared nodes (-1: none shared, or r
    // outside them) and its lower node; a standard table's value there
    __device__ int tab_interval(double r, double *x0) const
    {
        return a.tab_ref < 0 ? -1 : tab_settle(a.tab_ref, tab_guess(a.tab_ref, r), r, x0);
    }
    __device__ double tabj(int s, int j, double x0, double r) const
    {
        return j < 0 ? tab(s, r) : val_at(tabv(s, j), x0, r);
    }
    // GSL interp2d bicubic of the renormalisation grid at (x, y) (node derivatives of
    // natural cubic splines, Hermite patches; common.c:712-719)
    __device__ double bicubic(double x, double y) const
    {
        const int n = a.nren;
        const double *c = a.ren_chi;
        if (!(x >= c[0] && x <= c[n - 1] && y >= c[0] && y <= c[n - 1])) return __builtin_nan("");
        const int i = ce::interval_from(c, n, x, ce::interval_guess(c, n, x));
        const int j = ce::interval_from(c, n, y, ce::interval_guess(c, n, y));
        const double dx = c[i + 1] - c[i], dy = c[j + 1] - c[j];
        double2 q[8];
#pragma unroll
        for (int m = 0; m < 8; ++m)
            q[m] = *reinterpret_cast<const double2 *>(a.ren_rec + 4 * ((size_t)(j + m / 4) * n + i) + 2 * (m % 4));
        return patch(q, (x - c[i]) / dx, dx, (y - c[j]) / dy, dy);
    }
    // the Hermite patch at (t, u): q the records of nodes (i, j), (i + 1, j), then of j + 1
    static __device__ __forceinline__ double patch(const double2 *q, double t, double dx, double u, double dy)
    {
        const double t1 = 1 - t, u1 = 1 - u;
        const double ht[4] = {(1 + 2 * t) * t1 * t1, t * t * (3 - 2 * t), dx * t * t1 * t1, -dx * t * t * t1};
        const double hu[4] = {(1 + 2 * u) * u1 * u1, u * u * (3 - 2 * u), dy * u * u1 * u1, -dy * u * u * u1};
        double r = 0.0;
#pragma unroll
        for (int p = 0; p < 2; ++p)
#pragma unroll
            for (int m = 0; m < 2; ++m) {
                const double2 vx = q[4 * m + 2 * p], yxy = q[4 * m + 2 * p + 1];
                r += hu[m] * (vx.x * ht[p] + vx.y * ht[2 + p]) + hu[2 + m] * (yxy.x * ht[p] + yxy.y * ht[2 + p]);
            }
        return r;
    }
    // I_0^4 r^4 at r minus the grid at (x, y); the r = 0 renormalisation at `at0` where
    // `small` holds (functions.c:1524-1553, 3494-3512)
    __device__ double ren(double r2, double x, double y, bool small, double at0) const
    {
        if (small) return ak(a.ren0_x, a.ren0_y, a.nren0, at0);
        return tab(S40, sqrt(r2)) - bicubic(x, y);
    }
};

// geometry of the pair (functions.c:1498-1503, 3472-3479) and the values at the two
// end points (z(chi_i) and the biases there)
struct pt {
    double mu, chi1, chi2, c, omc, sint;
    double s1, s2, b1, b2, fe1, fe2;
    double Dc1, Dc2, fc1, fc2, cHc1, cHc2, ac1, ac2, G1c, G2c, G1c2;
};

__device__ pt make_pt(const intg_args &a, double zm, double mu, double sep)
{
    const lk L(a);
    pt p;
    p.mu = mu;
    const double cm = ak(a.bg_z, a.bg_chi, a.nbg, zm);
    p.chi1 = cm - sep * mu / 2;
    p.chi2 = cm + sep * mu / 2;
    const double den = 2 * cm * cm - mu * mu * sep * sep / 2;
    p.c = (2 * cm * cm - sep * sep + mu * mu * sep * sep / 2) / den;
    // 1 - cos(theta) without cancellation
    p.omc = sep * sep * (1 - mu * mu) / den;
    p.sint = sqrt(fmax(p.omc * (1 + p.c), 0.0));
    const double z1c = L.z_of(p.chi1), z2c = L.z_of(p.chi2);
    p.s1 = ak(a.mb_z, a.s1, a.nmb, z1c);
    p.s2 = ak(a.mb_z, a.s2, a.nmb, z2c);
    p.fe1 = ak(a.mb_z, a.fe1, a.nmb, z1c);
    p.fe2 = ak(a.mb_z, a.fe2, a.nmb, z2c);
    p.b1 = ak(a.bias_z, a.b1, a.nb, z1c);
    p.b2 = ak(a.bias_z, a.b2, a.nb, z2c);
    p.Dc1 = L.bgc(C_D1, z1c);
    p.Dc2 = L.bgc(C_D1, z2c);
    p.fc1 = L.bgc(C_F, z1c);
    p.fc2 = L.bgc(C_F, z2c);
    p.cHc1 = L.bgc(C_CH, z1c);
    p.cHc2 = L.bgc(C_CH, z2c);
    p.ac1 = L.bgc(C_A, z1c);
    p.ac2 = L.bgc(C_A, z2c);
    p.G1c = L.bg(a.bg_G1, z1c);
    p.G2c = L.bg(a.bg_G2, z2c);
    p.G1c2 = L.bg(a.bg_G1, z2c);
    return p;
}

// The double integral's constants of one (z, mu, r), and what it reads at one x1: lambda1,
// the weight times the sinh scale, the scale, the u interval's start and panel length,
// D1 / a, G1 chi1 H (f - 1), G1 chi1 H (H - 1) and (1 - x1) / x1
struct dco {
    double c, cc1, chi2, q2, a1, a2, g2chi2, k9;
    bool T, P, g4, g5, oc;
};
enum { X1_L, X1_W, X1_SC, X1_U, X1_DU, X1_DA, X1_E, X1_H, X1_IW, X1_N };

// v in scalar registers (every lane holds the same)
__device__ __forceinline__ double uniform(double v)
{
    const long long b = __double_as_longlong(v);
    const unsigned lo = __builtin_amdgcn_readfirstlane((unsigned)b), hi = __builtin_amdgcn_readfirstlane((unsigned)(b >> 32));
    return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}

// v again, which the compiler is not to take for the same in the next pass of a loop:
// what is made of it stays in the loop instead of in registers across it
template <typename V> __device__ __forceinline__ V again(V v)
{
    asm volatile("" : "+v"(v));
    return v;
}

__device__ dco double_consts(const intg_args &a, const pt &p)
{
    const unsigned f = a.flags;
    dco k;
    k.c = uniform(p.c);
    k.cc1 = uniform(p.c * p.c - 1);
    k.chi2 = uniform(p.chi2);
    k.a1 = uniform(2 - 5 * p.s1);
    k.a2 = uniform(2 - 5 * p.s2);
    k.q2 = uniform((2 - 5 * p.s1) * (2 - 5 * p.s2));
    k.g2chi2 = uniform(p.G2c * p.chi2);
    k.k9 = uniform(9 * a.Om * a.Om);
    k.g4 = f & F_G4;
    k.g5 = f & F_G5;
    k.oc = f & F_ONLY_CROSS;
    k.T = (f & F_LEN) && !k.oc && !(f & F_FLAT_LL);
    k.P = (f & F_LEN) && (k.g4 || k.g5);
    return k;
}

__device__ void x1_record(const intg_args &a, const pt &p, double x1, double w1, double *v)
{
    const lk L(a);
    const double l1 = p.chi1 * x1, centre = l1 * p.c;
    const double sc = fmax(l1 * p.sint, 1e-9 * p.chi2);
    const double lo = asinh((0.0 - centre) / sc), hi = asinh((p.chi2 - centre) / sc);
    v[X1_L] = l1;
    v[X1_W] = w1 * sc;
    v[X1_SC] = sc;
    v[X1_U] = lo;
    v[X1_DU] = (hi - lo) / a.pu;
    const double z1 = L.z_of(l1);
    const int j1 = L.bg_interval(z1);
    v[X1_DA] = L.bgcj(C_D1, j1, z1) / L.bgcj(C_A, j1, z1);
    v[X1_E] = v[X1_H] = 0.0;
    if (a.flags & F_G5) {
        const double cH = L.bgcj(C_CH, j1, z1);
        v[X1_E] = p.G1c * p.chi1 * cH * (L.bgcj(C_F, j1, z1) - 1);
        v[X1_H] = p.G1c * p.chi1 * cH * (cH - 1);
    }
    v[X1_IW] = (1 - x1) / x1;
}

// functions_double_integrated (functions.c:3460-4017) at (lambda1, lambda2) without the
// factor (H0 h)^4: v1 the x1 record, D2, a2 (and f2, cH2 with g5) at z(lambda2), ren the
// renormalised I_0^4 (g4, g5) and t the tables at r in the order of WSLOT (the first half
// where k.T, the second where k.T or k.P).  One reciprocal of r^2 serves all terms.
__device__ __forceinline__ double double_sum(const intg_args &a, const dco &k, const double *v1, double l2, double r2,
                                             double D2, double a2, double f2, double cH2, double ren, const double *t)
{
    const double c = again(k.c), cc1 = again(k.cc1), q2 = again(k.q2), l1 = v1[X1_L], iw1 = v1[X1_IW];
    const double LL = l1 * l2, m2 = k.chi2 - l2;
    double res = 0.0;
    if (k.T) {
        double T;
        if (r2 > 1e-20) {
            const double s = LL / r2;
            T = (2.0 / 5) * cc1 * LL * t[0] + (4.0 / 3) * c * t[1] + (4.0 / 15) * c * (r2 + 6 * c * LL) * t[2] +
                (2.0 / 7) * cc1 * LL * (2 + 3 * c * s) * t[3] +
                (2.0 / 15) * c * (2 * r2 + LL * (12 * c + 15 * cc1 * s)) * t[4] +
                (1.0 / 35) * cc1 * LL * (6 + s * (30 * c + 35 * cc1 * s)) * t[5];
        } else {
            T = 4 + 24 * LL * lk(a).tab(S11, 0.0) / 15;
        }
        // chi1 chi2 (1 - x1) (1 - x2) = lambda1 (1 - x1) / x1 (chi2 - lambda2)
        res += q2 / 4 * iw1 * l1 * m2 * T;
    }
    const double e1 = v1[X1_E], h1 = v1[X1_H];
    double e2 = 0.0, h2 = 0.0;
    if (k.g5) {
        e2 = k.g2chi2 * cH2 * (f2 - 1);
        h2 = k.g2chi2 * cH2 * (cH2 - 1);
    }
    if (k.g4 && !k.oc) res += q2 * ren;
    if (k.g5 && !k.oc) res += e1 * e2 * ren;
    if (k.g4 && k.g5) res += ren * (k.a1 * e2 + k.a2 * e1);
    if (k.P) {
        const double P = r2 != 0.0 ? 2 * LL * c * t[6] + LL * LL * cc1 * t[7] : 2 * LL * lk(a).tab(S31, 0.0);
        const double w2 = m2 / l2;
        if (k.g4) res += 0.5 * q2 * (w2 + iw1) * P;
        // functions.c:3927-3940: conformal_Hz (conformal_Hz - 1) as written there
        if (k.g5) res += 0.5 * P * (k.a2 * h1 * w2 + k.a1 * h2 * iw1);
    }
    return k.k9 * (v1[X1_DA] * D2 / a2) * res;
}

// Fetches by the whole wavefront.  A lookup by lanes of their own costs the L1 cache an
// access per lane and load; here eight lanes take one lane's 128-byte record (four
// a 64-byte one), 16 bytes each, straight into the wavefront's LDS buffer: an instruction
// moves 1 KB of full lines, 16 cycles of the cache where 64 gathers take 64 for 16 bytes
// a lane (measured: 8 KB of records in 229 cycles of a CU, 535 by gathers).  Instruction T
// takes the records of the lanes that are T modulo 8 (4); the 16-byte pieces of a record
// are permuted by T, so that the lanes' reads of one piece spread over the banks.  Every
// lane of the wavefront must take part.
typedef __attribute__((address_space(1))) const void *global_ptr;
typedef __attribute__((address_space(3))) void *lds_ptr;

__device__ __forceinline__ void to_lds(const char *src, char *buf)
{
    __builtin_amdgcn_global_load_lds((global_ptr)src, (lds_ptr)buf, 16, 0, 0);
}
// lanes 0-7 of each row of 16 get lane T's v, lanes 8-15 lane T + 8's
template <int T> __device__ __forceinline__ unsigned of_eight(unsigned v)
{
    const int lo = __builtin_amdgcn_update_dpp(0, (int)v, 0x150 + T, 0xf, 0x3, false);
    return (unsigned)__builtin_amdgcn_update_dpp(lo, (int)v, 0x158 + T, 0xf, 0xc, false);
}
// each quad of lanes gets its lane T's v
template <int T> __device__ __forceinline__ unsigned of_four(unsigned v)
{
    return (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, T * 0x55, 0xf, 0xf, false);
}
// piece: the lane's own 16-byte piece of a record, (lane & 7) * 16 or (lane & 3) * 16; off:
// the byte offset of its record
template <int T = 0> __device__ __forceinline__ void fetch128(const char *base, unsigned off, char *buf, unsigned piece)
{
    if constexpr (T < 8) {
        if (T == 0) piece = again(piece);
        to_lds(base + (size_t)((piece ^ (T << 4)) + of_eight<T>(off)), buf + T * 1024);
        fetch128<T + 1>(base, off, buf, piece);
    }
}
template <int T = 0> __device__ __forceinline__ void fetch64(const char *base, unsigned off, char *buf, unsigned piece)
{
    if constexpr (T < 4) {
        if (T == 0) piece = again(piece);
        to_lds(base + (size_t)((piece ^ (T << 4)) + of_four<T>(off)), buf + T * 1024);
        fetch64<T + 1>(base, off, buf, piece);
    }
}
// the lane's piece q of its record; at: its place in the buffer of the wavefront
__device__ __forceinline__ double2 piece_at(const char *smem, unsigned at, int q)
{
    return *reinterpret_cast<const double2 *>(smem + (at ^ (unsigned)(q << 4)));
}
// the buffer is filled; its reads are done and it may be filled again
__device__ __forceinline__ void fetched() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }
__device__ __forceinline__ void taken() { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); }

// The numerators of the single-integrated lensing terms that lose digits near the
// line of closest approach (functions.c:2183-2187, 2296-2303, 2638-2644; chi the local
// end point's distance, lambda the integration point's), in d = chi - lambda and
// e = 1 - cos(theta), where the squared separation is d^2 + 2 chi lambda e; each is the
// reference's polynomial identically, without its FP64 cancellation.
__device__ inline double num_rsd_i02(double ch, double lam, double d, double e)
{
    return 2 * d * d * (4 * d - ch) + 2 * e * (ch * ch * ch - 11 * ch * ch * d + 19 * ch * d * d - 12 * d * d * d) -
           3 * e * e * lam * (ch * ch - 2 * ch * d + 4 * d * d) - 6 * ch * e * e * e * lam * lam;
}

__device__ inline double num_rsd_i04(double ch, double lam, double d, double e)
{
    const double d2 = d * d, ch2 = ch * ch, e2 = e * e, lm2 = lam * lam;
    return 4 * d2 * d2 * (d - 2 * ch) + 4 * d2 * e * (12 * ch2 * ch - 23 * ch2 * d + 15 * ch * d2 - 3 * d2 * d) +
           6 * e2 * lm2 * (-2 * ch2 * ch + 6 * ch2 * d - 6 * ch * d2 + d2 * d) +
           2 * ch * e2 * e * lm2 * (2 * ch2 - 4 * ch * d + 3 * d2) + ch2 * e2 * e2 * lm2 * lam;
}

__device__ inline double num_d1_i13(double ch, double lam, double d, double e)
{
    const double d2 = d * d, ch2 = ch * ch;
    return 2 * d2 * d * (3 * ch - d) + 2 * d * e * (-9 * ch2 * ch + 14 * ch2 * d - 8 * ch * d2 + d2 * d) -
           ch * e * e * lam * (2 * ch2 - 5 * ch * d + 4 * d2) - ch2 * e * e * e * lam * lam;
}

// functions_single_integrated (functions.c:1486-3458) at x: point 1 at chi1 with the
// integrated source along line of sight 2 (lambda2 = x chi2, squared separation r21)
// and the other way round (r22); the branches where neither is exactly zero
__device__ double single_point(const intg_args &a, const pt &p, double x)
{
    const lk L(a);
    const unsigned f = a.flags;
    const double c = p.c, Om = a.Om, H2 = a.H0h * a.H0h, H4 = H2 * H2;
    const double chi1 = p.chi1, chi2 = p.chi2;
    const double l1 = chi1 * x, l2 = chi2 * x;
    const double r21 = fmax(l2 * l2 + chi1 * chi1 - 2 * chi1 * l2 * c, 0.0);
    const double r22 = fmax(l1 * l1 + chi2 * chi2 - 2 * chi2 * l1 * c, 0.0);
    const double rA = sqrt(r21), rB = sqrt(r22);
    double xA = 0.0, xB = 0.0;
    const int jA = L.tab_interval(rA, &xA), jB = L.tab_interval(rB, &xB);
    const double z1 = L.z_of(l1), z2 = L.z_of(l2);
    const int j1 = L.bg_interval(z1), j2 = L.bg_interval(z2);
    const double D1x = L.bgcj(C_D1, j1, z1), D2x = L.bgcj(C_D1, j2, z2);
    const double a1x = L.bgcj(C_A, j1, z1), a2x = L.bgcj(C_A, j2, z2);
    const double VA = D2x / a2x, VB = D1x / a1x;
    const double WA = (1 - x) * VA, WB = (1 - x) * VB;
    const double s1 = p.s1, s2 = p.s2, c2 = 2 * c * c - 1, e = p.omc;
    const bool lens = f & F_LEN, g4 = f & F_G4, g5 = f & F_G5, full_dl = !(f & F_FLAT_DL);
    double res = 0.0;
    if (lens && (f & F_DEN) && full_dl)   // functions.c:1707-1781
        res += H2 * (-3 * Om / 2) *
               (p.b1 * (2 - 5 * s2) * p.Dc1 * chi2 * WA *
                    (2 * chi1 * c * L.tabj(S11, jA, xA, rA) - chi1 * chi1 * l2 * (1 - c * c) * L.tabj(S02, jA, xA, rA) / r21) +
                p.b2 * (2 - 5 * s1) * p.Dc2 * chi1 * WB *
                    (2 * chi2 * c * L.tabj(S11, jB, xB, rB) - chi2 * chi2 * l1 * (1 - c * c) * L.tabj(S02, jB, xB, rB) / r22));
    if (lens && (f & F_RSD) && full_dl) {   // functions.c:2167-2198, then 2291-2324 or 2377-2390
        const bool wide = fabs(p.mu) < 0.999;
        auto rsd = [&](double ch, double lam, double rr, double rv, int jv, double xv) {
            (void)rr;
            const double d = ch - lam, rs = d * d + 2 * ch * lam * e;
            double v = (lam - 6 * ch * c + 3 * lam * c2) * L.tabj(S00, jv, xv, rv) / 15 -
                       num_rsd_i02(ch, lam, d, e) * L.tabj(S02, jv, xv, rv) / rs / 21;
            if (wide) v -= num_rsd_i04(ch, lam, d, e) * L.tabj(S04, jv, xv, rv) / rs / rs / 35;
            else v += 4 * (lam + ch) * L.tabj(S04, jv, xv, rv) / 35;
            return v;
        };
        res += H2 * 3 * Om / 2 *
               (chi2 * p.fc1 * (2 - 5 * s2) * p.Dc1 * WA * rsd(chi1, l2, r21, rA, jA, xA) +
                chi1 * p.fc2 * (2 - 5 * s1) * p.Dc2 * WB * rsd(chi2, l1, r22, rB, jB, xB));
    }
    if (lens && (f & F_D1) && full_dl) {   // functions.c:2624-2661 (G1 at z(chi2), 2 - 5 s2 in the second half)
        auto d1k = [&](double ch, double lam, double rr, double rv, int jv, double xv) {
            (void)rr;
            const double d = ch - lam, rs = d * d + 2 * ch * lam * e;
            return 2 * (c * (lam * lam - 2 * ch * ch) + ch * lam * (2 * c2 - 1)) * L.tabj(S11, jv, xv, rv) / 15 +
                   2 * c * L.tabj(S20, jv, xv, rv) / 3 - num_d1_i13(ch, lam, d, e) * L.tabj(S13, jv, xv, rv) / rs / 15;
        };
        res += H2 * 3 * Om / 2 *
               (chi2 * p.cHc1 * p.fc1 * p.G1c * (2 - 5 * s2) * p.Dc1 * WA * d1k(chi1, l2, r21, rA, jA, xA) +
                chi1 * p.cHc2 * p.fc2 * p.G1c2 * (2 - 5 * s2) * p.Dc2 * WB * d1k(chi2, l1, r22, rB, jB, xB));
    }
    if (lens && (f & (F_D2 | F_G1 | F_G2 | F_G3))) {
        const double PA = 2 * chi1 * c * L.tabj(S31, jA, xA, rA) - chi1 * chi1 * l2 * (1 - c * c) * L.tabj(S22, jA, xA, rA);
        const double PB = 2 * chi2 * c * L.tabj(S31, jB, xB, rB) - chi2 * chi2 * l1 * (1 - c * c) * L.tabj(S22, jB, xB, rB);
        const double A = chi2 * p.Dc1 * WA * PA, B = chi1 * p.Dc2 * WB * PB;
        const double q = 9 * Om * Om / 4 * H4;
        if (f & F_D2)   // functions.c:3000-3030
            res += H2 * (-3 * Om / 2) *
                   ((3 - p.fe1) * p.fc1 * p.cHc1 * p.cHc1 * (2 - 5 * s2) * A +
                    (3 - p.fe2) * p.fc2 * p.cHc2 * p.cHc2 * (2 - 5 * s1) * B);
        if (f & F_G1) res += q * ((1 + p.G1c) * (2 - 5 * s2) * A + (1 + p.G2c) * (2 - 5 * s1) * B);   // 3032-3060
        if (f & F_G2) res += q * ((5 * s1 - 2) * (2 - 5 * s2) * A + (5 * s2 - 2) * (2 - 5 * s1) * B);  // 3062-3090
        if (f & F_G3) res += q * ((p.fc1 - 1) * (2 - 5 * s2) * A + (p.fc2 - 1) * (2 - 5 * s1) * B);   // 3092-3120
    }
    if (g4 || g5) {
        const bool div = f & (F_D2 | F_G1 | F_G2 | F_G3 | F_G4 | F_G5);
        const double ren1 = div ? L.ren(r21, l2, chi1, r21 == 0.0, l2) : 0.0;
        const double ren2 = div ? L.ren(r22, l1, chi2, r22 == 0.0, l1) : 0.0;
        const double E1 = L.bgcj(C_CH, j1, z1) * (L.bgcj(C_F, j1, z1) - 1),
                     E2 = L.bgcj(C_CH, j2, z2) * (L.bgcj(C_F, j2, z2) - 1);
        auto rsdk = [&](double rr, double lam, double rv, int jv, double xv) {
            return (2 * rr / 3 + (c * c - 1) * lam * lam) * L.tabj(S22, jv, xv, rv) - L.tabj(S20, jv, xv, rv) / 3;
        };
        const double q = 9 * Om * Om / 2 * H4;
        const double cH2c1 = p.cHc1 * p.cHc1, cH2c2 = p.cHc2 * p.cHc2;
        if (g4) {
            if (f & F_DEN)   // functions.c:3122-3140
                res += H2 * (-3 * Om) *
                       (p.b1 * (2 - 5 * s2) * p.Dc1 * VA * L.tabj(S20, jA, xA, rA) + p.b2 * (2 - 5 * s1) * p.Dc2 * VB * L.tabj(S20, jB, xB, rB));
            if (f & F_RSD)   // functions.c:3164-3189
                res += H2 * 3 * Om *
                       (p.fc1 * (2 - 5 * s2) * p.Dc1 * VA * rsdk(r21, l2, rA, jA, xA) +
                        p.fc2 * (2 - 5 * s1) * p.Dc2 * VB * rsdk(r22, l1, rB, jB, xB));
            if (f & F_D1)    // functions.c:3220-3235
                res += H2 * 3 * Om *
                       (p.cHc1 * p.fc1 * (2 - 5 * s2) * p.Dc1 * VA * (l2 * c - chi1) * L.tabj(S31, jA, xA, rA) +
                        p.cHc2 * p.fc2 * (2 - 5 * s1) * p.Dc2 * VB * (l1 * c - chi2) * L.tabj(S31, jB, xB, rB));
            if (f & F_D2)    // functions.c:3258-3275
                res += H2 * (-3 * Om) *
                       ((3 - p.fe1) * p.fc1 * cH2c1 * (2 - 5 * s2) * p.Dc1 * VA * ren1 +
                        (3 - p.fe2) * p.fc2 * cH2c2 * (2 - 5 * s1) * p.Dc2 * VB * ren2);
            const double u1 = p.Dc1 / p.ac1 * VA * ren1, u2 = p.Dc2 / p.ac2 * VB * ren2;
            if (f & F_G1) res += q * ((1 + p.G1c) * (2 - 5 * s2) * u1 + (1 + p.G2c) * (2 - 5 * s1) * u2);   // 3298-3315
            if (f & F_G2) res += q * ((5 * s1 - 2) * (2 - 5 * s2) * u1 + (5 * s2 - 2) * (2 - 5 * s1) * u2);  // 3340-3357
            if (f & F_G3) res += q * ((p.fc1 - 1) * (2 - 5 * s2) * u1 + (p.fc2 - 1) * (2 - 5 * s1) * u2);   // 3382-3399
        }
        if (g5) {
            if (f & F_DEN)   // functions.c:3142-3162 (D1 a along the line of sight, as written there)
                res += H2 * (-3 * Om) *
                       (chi2 * p.b1 * p.G2c * p.Dc1 * E2 * D2x * a2x * L.tabj(S20, jA, xA, rA) +
                        chi1 * p.b2 * p.G1c * p.Dc2 * E1 * D1x * a1x * L.tabj(S20, jB, xB, rB));
            if (f & F_RSD)   // functions.c:3191-3218
                res += H2 * 3 * Om *
                       (chi2 * p.fc1 * p.G2c * p.Dc1 * E2 * VA * rsdk(r21, l2, rA, jA, xA) +
                        chi1 * p.fc2 * p.G1c * p.Dc2 * E1 * VB * rsdk(r22, l1, rB, jB, xB));
            if (f & F_D1)    // functions.c:3237-3256
                res += H2 * 3 * Om *
                       (chi2 * p.cHc1 * p.fc1 * p.G2c * p.Dc1 * E2 * VA * (l2 * c - chi1) * L.tabj(S31, jA, xA, rA) +
                        chi1 * p.cHc2 * p.fc2 * p.G1c * p.Dc2 * E1 * VB * (l1 * c - chi2) * L.tabj(S31, jB, xB, rB));
            if (f & F_D2)    // functions.c:3277-3296
                res += H2 * (-3 * Om) *
                       (chi2 * (3 - p.fe1) * p.fc1 * cH2c1 * p.G2c * p.Dc1 * E2 * VA * ren1 +
                        chi1 * (3 - p.fe2) * p.fc2 * cH2c2 * p.G1c * p.Dc2 * E1 * VB * ren2);
            const double u1 = chi2 * p.Dc1 / p.ac1 * E2 * VA * ren1, u2 = chi1 * p.Dc2 / p.ac2 * E1 * VB * ren2;
            if (f & F_G1) res += q * ((1 + p.G1c) * p.G2c * u1 + (1 + p.G2c) * p.G1c * u2);   // 3317-3338
            if (f & F_G2) res += q * ((5 * s1 - 2) * p.G2c * u1 + (5 * s2 - 2) * p.G1c * u2);  // 3359-3380
            if (f & F_G3) res += q * ((p.fc1 - 1) * p.G2c * u1 + (p.fc2 - 1) * p.G1c * u2);   // 3401-3422
        }
    }
    return res;
}

// node q of the composite rule on [lo, hi]: `panels` equal panels of the n-point
// Gauss-Legendre rule (gx, gw on [-1, 1]); returns the node, weight in *w
__device__ inline double composite(double lo, double hi, int panels, int n, const double *gx, const double *gw, int q,
                                   double *w)
{
    const int k = q / n, j = q - k * n;
    const double step = (hi - lo) / panels;
    const double e0 = lo + k * step, e1 = (k + 1 == panels) ? hi : lo + (k + 1) * step;
    const double h = (e1 - e0) / 2;
    *w = h * gw[j];
    return (e0 + e1) / 2 + h * gx[j];
}

// the pieces of the single-integrated rule: [a, b] mapped about centre cc with width s
struct piece {
    double a, b, cc, s;
};

__device__ int single_pieces(const pt &p, piece *pc)
{
    const double cA = p.chi1 * p.c / p.chi2, sA = fmax(p.chi1 * p.sint / p.chi2, 1e-12);
    const double cB = p.chi2 * p.c / p.chi1, sB = fmax(p.chi2 * p.sint / p.chi1, 1e-12);
    double in[2];
    int nin = 0;
    if (cA > 0.0 && cA < 1.0) in[nin++] = cA;
    if (cB > 0.0 && cB < 1.0 && !(nin == 1 && cB == cA)) in[nin++] = cB;
    if (nin == 2 && in[1] < in[0]) {
        const double t = in[0];
        in[0] = in[1];
        in[1] = t;
    }
    double cuts[5];
    int nc = 0;
    cuts[nc++] = 0.0;
    if (nin == 2) {
        cuts[nc++] = in[0];
        cuts[nc++] = (in[0] + in[1]) / 2;
        cuts[nc++] = in[1];
    } else if (nin == 1) {
        cuts[nc++] = in[0];
    }
    cuts[nc++] = 1.0;
    int np = 0;
    for (int i = 0; i + 1 < nc; ++i) {
        const double a = cuts[i], b = cuts[i + 1];
        if (b <= a) continue;
        const double m = (a + b) / 2;
        const double dA = fmin(fmin(fabs(cA - m), fabs(cA - a)), fabs(cA - b));
        const double dB = fmin(fmin(fabs(cB - m), fabs(cB - a)), fabs(cB - b));
        double cc = dA <= dB ? cA : cB;
        const double s = dA <= dB ? sA : sB;
        if (a < cc && cc < b) cc = fabs(cc - a) < fabs(cc - b) ? a : b;
        pc[np++] = piece{a, b, cc, s};
    }
    return np;
}

// the value records and node pairs of up to 16 curves, one thread per (node, curve)
struct coef_list {
    int ncurve;
    const double *x[16], *y[16];
    int n[16], stride[16], pstride[16];
    double *val[16], *pair[16];   // pair null: another curve of the grid writes it
};

__global__ void __launch_bounds__(256) k_intg_coef(coef_list L)
{
    const int t = blockIdx.y;
    const int j = blockIdx.x * blockDim.x + threadIdx.x;
    const int n = L.n[t];
    if (j >= n) return;
    const double *x = L.x[t], *y = L.y[t];
    double v[VAL] = {y[j], 0.0, 0.0, 0.0}, x1 = x[j];   // the last node's: no segment
    if (j < n - 1) {
        const ce::akima_cf<double> cf = ce::akima_coefs<double>(x, nullptr, y, nullptr, n, j);
        v[1] = cf.b;
        v[2] = cf.c;
        v[3] = cf.d;
        x1 = x[j + 1];
    }
    double *r = L.val[t] + (size_t)L.stride[t] * j;
    *reinterpret_cast<double2 *>(r) = double2{v[0], v[1]};
    *reinterpret_cast<double2 *>(r + 2) = double2{v[2], v[3]};
    if (L.pair[t]) *reinterpret_cast<double2 *>(L.pair[t] + (size_t)L.pstride[t] * j) = double2{x[j], x1};
}

// workgroup sum: wavefront shuffles, then one slot per wavefront in LDS
__device__ __forceinline__ void put_sum(double acc, double *out)
{
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) acc += __shfl_down(acc, o);
    __shared__ double red[16];
    const int wv = threadIdx.x >> 6, lane = threadIdx.x & 63;
    if (lane == 0) red[wv] = acc;
    __syncthreads();
    if (threadIdx.x == 0) {
        double ss = 0.0;
        for (int k = 0; k < (int)(blockDim.x >> 6); ++k) ss += red[k];
        *out = ss;
    }
}

// the points' end-point values, a thread each: a chain of some twenty searches, which a
// workgroup of the integrals would otherwise wait for before its first node
__global__ void __launch_bounds__(64) k_intg_points(const intg_args *__restrict__ pa, int64_t first, int count,
                                                    pt *__restrict__ pts)
{
    const intg_args &a = *pa;
    const int i = blockIdx.x * 64 + threadIdx.x;
    if (i >= count) return;
    const int64_t idx = first + i;   // (z, mu, r), r fastest
    pts[i] = make_pt(a, a.zmean[idx / ((int64_t)a.nsep * a.nmu)], a.mu[(idx / a.nsep) % a.nmu], a.sep[idx % a.nsep]);
}

// one workgroup per (z, mu, r): the single-integrated terms into out[..][0].  The
// arguments live in device memory (a pointer, not a by-value struct, whose address
// the lookups would otherwise take in private memory).
__global__ void __launch_bounds__(256) k_integrated_single(const intg_args *__restrict__ pa, const pt *__restrict__ pts,
                                                           int64_t first)
{
    const intg_args &a = *pa;
    const unsigned f = a.flags;
    double acc = 0.0;
    if ((f & (F_LEN | F_G4 | F_G5)) && (f & (F_DEN | F_RSD | F_D1 | F_D2 | F_G1 | F_G2 | F_G3))) {
        // the pieces in LDS (a private array indexed by node would live in scratch), with
        // the ends of their u intervals
        __shared__ piece pc[4];
        __shared__ double ends[4][2];
        __shared__ int npc;
        const pt &p = pts[blockIdx.x];
        if (threadIdx.x == 0) {
            piece t[4];
            npc = single_pieces(p, t);
            for (int i = 0; i < 4; ++i) pc[i] = t[i];
        }
        __syncthreads();
        const int np = npc;
        if ((int)threadIdx.x < 2 * np) {
            const int i = threadIdx.x >> 1;
            const piece &P = pc[i];
            const double sgn = P.a >= P.cc ? 1.0 : -1.0;
            // the lower end of u: that of b where the piece is mirrored
            const double e = ((threadIdx.x & 1) != 0) == (sgn > 0.0) ? P.b : P.a;
            ends[i][threadIdx.x & 1] = asinh(sgn * (e - P.cc) / P.s);
        }
        __syncthreads();
        const int per = a.ps * a.ns;
        for (int q = threadIdx.x; q < np * per; q += blockDim.x) {
            const int i = q / per;
            const piece &P = pc[i];
            const double sgn = P.a >= P.cc ? 1.0 : -1.0;
            double w;
            const double u = composite(ends[i][0], ends[i][1], a.ps, a.ns, a.gsx, a.gsw, q - i * per, &w);
            // sinh and cosh from one exponential (x's absolute error stays ~eps s)
            const double eu = exp(u), ei = 1.0 / eu;
            const double x = P.cc + sgn * P.s * (0.5 * (eu - ei));
            acc += w * P.s * (0.5 * (eu + ei)) * single_point(a, p, x);
        }
    }
    put_sum(acc, a.out + 2 * (first + blockIdx.x));
}

// The LDS of the double integral: the wavefronts' buffers and the lookup tables of the
// fetching variant (n40, nren, f0: 0 where they are not read), the x1 records.
constexpr int DWAVES = 12;   // wavefronts a workgroup of the fetching variant, at most
constexpr int N40 = 512, NREN = 512, BUCKETS = 512;
constexpr int DLDS_MAX = 160 * 1024 - 512;   // beside the static LDS of the kernel
struct dlds {
    int s40v, sx, s40x, chi, rchi, head, bucket, guess, bytes;   // byte offsets
    __host__ __device__ dlds(int waves, int n1, int n40, int nren, int f0, int nguess)
    {
        s40v = 8192 * waves;
        sx = s40v + 32 * n40;
        s40x = sx + 8 * X1_N * n1;
        chi = s40x + 8 * n40;
        rchi = chi + 8 * nren;
        head = rchi + 8 * nren;
        bucket = head + 8 * (f0 + 1);
        guess = bucket + (n40 ? 2 * (BUCKETS + 2) : 0);
        bytes = guess + 2 * nguess;
    }
};

// One workgroup per (z, mu, r): the double-integrated terms into out[..][1], 192 lambda2
// nodes for each of 128 to 192 x1 nodes by the default rule; a lane takes one node.
// FETCH: the tables that are read share their nodes, and I_0^4 and the renormalisation grid
// are small enough for LDS (the launcher's rule).  Before, 56 gathers of 64 lanes a
// node, through generic pointers, bounded it (10.3 ms for 4096 points with every term).
// Now the records come by the line (36 fetches of 1 KB a wavefront's 64 nodes, 28 cycles of
// the CU's cache path each), I_0^4 with a bucket index, the chi guesses and the
// renormalisation grid's abscissae stand in LDS, and 2 gathers are left: 5.5 ms, of it about
// 90% by those fetches and 53% by the FP64 pipes.  DWAVES: 12 wavefronts a workgroup,
// 168 registers each, whose 8 KB buffers and the tables they share fill the LDS; 16 spill
// (8.4 ms), 8 hide less (6.1 ms).  FETCH false: tables on nodes of their own, or larger ones,
// looked up lane by lane.
template <bool FETCH>
__global__ void __launch_bounds__(FETCH ? 64 * DWAVES : 256) k_integrated_double(const intg_args *__restrict__ pa, const pt *__restrict__ pts, int64_t first)
{
    const intg_args &a = *pa;
    const lk L(a);
    const pt &sp = pts[blockIdx.x];
    extern __shared__ __align__(16) char smem[];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int waves = blockDim.x >> 6;
    const bool g45 = a.flags & (F_G4 | F_G5);
    const int pB = a.p1 / 2 > 1 ? a.p1 / 2 : 1;
    const int n40 = FETCH && g45 ? a.tab_len[S40] : 0, nren = FETCH && g45 ? a.nren : 0;
    const int ref = a.tab_ref, f0 = FETCH && ref >= 0 && a.tab_f0[ref] > 0 ? a.tab_f0[ref] : 0;
    const dlds o(FETCH ? waves : 0, (a.p1 + pB) * a.n1, n40, nren, f0, FETCH ? a.nguess + 1 : 0);
    char *buf = smem + 8192 * wave;
    const unsigned p128 = (lane & 7) << 4, p64 = (lane & 3) << 4;
    const unsigned l128 = 8192 * wave + ((lane & 7) << 10) + ((lane >> 3) << 7) + p128;
    const unsigned l64 = 8192 * wave + ((lane & 3) << 10) + ((lane >> 2) << 6) + p64;
    double *sx = reinterpret_cast<double *>(smem + o.sx);
    double *x40 = reinterpret_cast<double *>(smem + o.s40x), *v40 = reinterpret_cast<double *>(smem + o.s40v);
    double *chi = reinterpret_cast<double *>(smem + o.chi), *rchi = reinterpret_cast<double *>(smem + o.rchi);
    double *head = reinterpret_cast<double *>(smem + o.head);
    unsigned short *bucket = reinterpret_cast<unsigned short *>(smem + o.bucket);
    unsigned short *guess = reinterpret_cast<unsigned short *>(smem + o.guess);
    double lx40 = 0.0, ls40 = 0.0;
    if (FETCH) {
        const double *x = a.tab_x + a.tab_off[S40];
        for (int i = threadIdx.x; i < n40; i += blockDim.x) {
            x40[i] = x[i];
            const double2 *v = reinterpret_cast<const double2 *>(L.tabv(S40, i));
            reinterpret_cast<double2 *>(v40 + 4 * i)[0] = v[0];
            reinterpret_cast<double2 *>(v40 + 4 * i)[1] = v[1];
        }
        for (int i = threadIdx.x; i < nren; i += blockDim.x) {
            chi[i] = a.ren_chi[i];
            rchi[i] = i < nren - 1 ? 1.0 / (a.ren_chi[i + 1] - a.ren_chi[i]) : 0.0;
        }
        for (int i = threadIdx.x; i <= a.nguess; i += blockDim.x) guess[i] = (unsigned short)max((int)a.chi_guess[i], 0);
        if (f0)
            for (int i = threadIdx.x; i <= f0; i += blockDim.x) head[i] = a.tab_x[a.tab_off[ref] + i];
        if (n40) {
            // uniform in log r from the second node (the first may be 0) to the last
            lx40 = uniform(log(x[1]));
            ls40 = uniform(BUCKETS / (log(x[n40 - 1]) - lx40));
            for (int i = threadIdx.x; i <= BUCKETS; i += blockDim.x)
                bucket[i] = (unsigned short)ce::interval_bisect(x, 0, n40 - 1, exp(lx40 + i / ls40));
        }
    }
    __syncthreads();
    double acc = 0.0;
    if (a.flags & (F_LEN | F_G4 | F_G5)) {
        const double xb = sp.chi1 * sp.c > sp.chi2 ? sp.chi2 / (sp.chi1 * sp.c) : 1.0;
        const int pA = a.p1, n1 = (xb < 1.0 ? pA + pB : pA) * a.n1, nu = a.nu, nuu = a.pu * nu;
        for (int i = threadIdx.x; i < n1; i += blockDim.x) {
            double w1;
            const double x1 = i < pA * a.n1 ? composite(0.0, xb, pA, a.n1, a.g1x, a.g1w, i, &w1)
                                            : composite(xb, 1.0, pB, a.n1, a.g1x, a.g1w, i - pA * a.n1, &w1);
            x1_record(a, sp, x1, w1, sx + X1_N * i);
        }
        __syncthreads();
        const dco k = double_consts(a, sp);
        const float inu = 1.0f / (float)nu;
        const int di = (int)blockDim.x / nuu, dr = (int)blockDim.x - di * nuu;
        int i1 = (int)threadIdx.x / nuu, iu = (int)threadIdx.x - i1 * nuu;
        // the lookups' uniform values
        const bool tabs = k.T || k.P;
        const int nt = ref >= 0 ? a.tab_len[ref] : 0, nbg = a.nbg, nguess = a.nguess;
        const double *tx = ref >= 0 ? a.tab_x + a.tab_off[ref] : a.tab_x;
        const double *tp = ref >= 0 ? a.tab_pair + PAIR * (size_t)a.tab_off[ref] : a.tab_pair;
        const double *gux = a.gux, *guw = a.guw, *zp = a.bgz_pair;
        const char *zof = reinterpret_cast<const char *>((const double *)a.zof);
        const char *bgw = reinterpret_cast<const char *>((const double *)a.bgc_wide);
        const char *wide = reinterpret_cast<const char *>((const double *)a.tab_wide);
        const char *rec = reinterpret_cast<const char *>((const double *)a.ren_rec);
        double t_lo = 0.0, t_hi = 0.0, t_lx0 = 0.0, t_lsc = 0.0;
        if (FETCH && tabs) {
            t_lo = tx[0];
            t_hi = tx[nt - 1];
            t_lx0 = a.tab_lx0[ref];
            t_lsc = a.tab_lsc[ref];
        }
        const double zx0 = a.bg_z[0], zx1 = a.bg_z[nbg - 1], zsc = uniform((nbg - 1) / (zx1 - zx0));
        const double cx0 = a.bg_chi[0], cx1 = a.bg_chi[nbg - 1], csc = uniform(nguess / cx1);
        const double n_lo = nren ? uniform(chi[0]) : 0.0, n_hi = nren ? uniform(chi[nren - 1]) : 0.0;
        const double nsc = nren ? uniform((nren - 1) / (n_hi - n_lo)) : 0.0;
        const double x40_lo = n40 ? uniform(x40[0]) : 0.0, x40_hi = n40 ? uniform(x40[n40 - 1]) : 0.0;
        // whole wavefronts to the end: the lanes past the last node repeat one of its row
        for (int q = wave * 64; q < n1 * nuu; q += (int)blockDim.x) {
            const bool live = i1 < n1;
            const double *v1 = sx + X1_N * (live ? i1 : n1 - 1);
            const int kp = (int)(((float)iu + 0.5f) * inu), ju = iu - kp * nu;
            const double du = v1[X1_DU];
            // sinh and cosh from one exponential (lambda2's absolute error stays ~eps sc)
            const double eu = exp(v1[X1_U] + du * (kp + 0.5 * (1.0 + gux[ju]))), ei = 1.0 / eu;
            const double wt = v1[X1_W] * (0.25 * du * guw[ju]) * (eu + ei);
            const double l1 = v1[X1_L], l2 = l1 * k.c + v1[X1_SC] * (0.5 * (eu - ei));
            const double r2 = fmax(l1 * l1 + l2 * l2 - 2 * l1 * l2 * k.c, 0.0), r = sqrt(r2);
            double D2, a2, f2 = 0.0, cH2 = 0.0, ren = 0.0, t[8];
            if (FETCH) {
                // z(lambda2) on its way
                int jc = -1;
                if (l2 >= cx0 && l2 <= cx1)
                    jc = lk::below_last(guess[ce::clamp_index(l2 * csc, nguess + 1)], nbg);
                const unsigned jz = jc < 0 ? 0u : (unsigned)jc;
                taken();
                fetch64(zof, jz * (8u * ZOF), buf, p64);
                // r's interval on the tables' nodes: exact in the head, else from the log
                const double lr = log(r);
                int jr = -1;
                double xr = 0.0;
                if (tabs && r >= t_lo && r <= t_hi) {
                    if (!f0) {
                        jr = ce::interval_bisect(tx, 0, nt - 1, r);
                    } else if (r < head[f0]) {
                        jr = ce::interval_bisect(head, 0, f0, r);
                    } else {
                        jr = lk::below_last(f0 + ce::clamp_index((lr - t_lx0) * t_lsc, nt - f0), nt);
                    }
                    nodes nd = pair_at(tp, jr);
                    if (!pair_hit(nd, jr, nt, r)) {
                        jr = ce::interval_from(tx, nt, r, jr);
                        nd = pair_at(tp, jr);
                    }
                    xr = nd.x0;
                }
                const unsigned orec = (jr < 0 ? 0u : (unsigned)jr) * (8u * WIDE);
                fetched();
                unsigned at = again(l64);
                const double2 zn = piece_at(smem, at, 0);
                double z2 = cubic(piece_at(smem, at, 1), piece_at(smem, at, 2), l2 - zn.x);
                if (jc < 0) z2 = __builtin_nan("");
                else if (!pair_hit(nodes{zn.x, zn.y}, jc, nbg, l2)) z2 = L.zofj(ce::interval_from(a.bg_chi, a.nbg, l2, jc), l2);
                // the curves at z2
                int jb = -1;
                double xz = 0.0;
                if (z2 >= zx0 && z2 <= zx1) {
                    jb = lk::below_last(ce::clamp_index((z2 - zx0) * zsc, nbg), nbg);
                    nodes nb = pair_at(zp, jb);
                    if (!pair_hit(nb, jb, nbg, z2)) {
                        jb = ce::interval_from(a.bg_z, a.nbg, z2, jb);
                        nb = pair_at(zp, jb);
                    }
                    xz = nb.x0;
                }
                const double dz = jb < 0 ? __builtin_nan("") : z2 - xz;
                taken();
                fetch128(bgw, (jb < 0 ? 0u : (unsigned)jb) * (8u * BGW), buf, p128);
                // I_0^4 r^4 from LDS
                int ix = 0, jy = 0;
                bool patched = false;
                if (n40) {
                    ren = __builtin_nan("");
                    if (r >= x40_lo && r <= x40_hi) {
                        const int b = ce::clamp_index((lr - lx40) * ls40, BUCKETS);
                        int lo = bucket[b], hi = min(bucket[b + 1] + 1, n40 - 1);
                        if (!(x40[lo] <= r && (hi == n40 - 1 || r < x40[hi]))) {
                            lo = 0;
                            hi = n40 - 1;
                        }
                        lo = ce::interval_bisect(x40, lo, hi, r);
                        ren = val_at(v40 + 4 * lo, x40[lo], r);
                    }
                    if (l1 >= n_lo && l1 <= n_hi && l2 >= n_lo && l2 <= n_hi) {
                        patched = true;
                        ix = ce::interval_from(chi, nren, l1, ce::clamp_index((l1 - n_lo) * nsc, nren));
                        jy = ce::interval_from(chi, nren, l2, ce::clamp_index((l2 - n_lo) * nsc, nren));
                    }
                }
                fetched();
                at = again(l128);
                D2 = cubic(piece_at(smem, at, 2 * C_D1), piece_at(smem, at, 2 * C_D1 + 1), dz);
                a2 = cubic(piece_at(smem, at, 2 * C_A), piece_at(smem, at, 2 * C_A + 1), dz);
                if (k.g5) {
                    f2 = cubic(piece_at(smem, at, 2 * C_F), piece_at(smem, at, 2 * C_F + 1), dz);
                    cH2 = cubic(piece_at(smem, at, 2 * C_CH), piece_at(smem, at, 2 * C_CH + 1), dz);
                }
                if (n40) {
                    const unsigned on = (unsigned)(jy * nren + ix) * 32u, row = (unsigned)nren * 32u;
                    taken();
                    fetch64(rec, on, buf, p64);
                    fetch64(rec + row, on, buf + 4096, p64);
                    fetched();
                    at = again(l64);
                    double2 p[8];
#pragma unroll
                    for (int m = 0; m < 8; ++m) p[m] = piece_at(smem, at + 4096 * (m / 4), m % 4);
                    const double bic = lk::patch(p, (l1 - chi[ix]) * rchi[ix], chi[ix + 1] - chi[ix],
                                                 (l2 - chi[jy]) * rchi[jy], chi[jy + 1] - chi[jy]);
                    ren -= patched ? bic : __builtin_nan("");
                    if (r2 <= 1e-12) ren = ak(a.ren0_x, a.ren0_y, a.nren0, l1);
                }
                at = again(l128);
                const double dr2 = jr < 0 ? __builtin_nan("") : r - xr;
                if (k.T) {
                    taken();
                    fetch128(wide, orec, buf, p128);
                    fetched();
#pragma unroll
                    for (int m = 0; m < 4; ++m) t[m] = cubic(piece_at(smem, at, 2 * m), piece_at(smem, at, 2 * m + 1), dr2);
                }
                if (tabs) {
                    taken();
                    fetch128(wide + 128, orec, buf, p128);
                    fetched();
#pragma unroll
                    for (int m = 0; m < 4; ++m)
                        t[4 + m] = cubic(piece_at(smem, at, 2 * m), piece_at(smem, at, 2 * m + 1), dr2);
                }
            } else {
                const double z2 = L.z_of(l2);
                const int j2 = L.bg_interval(z2);
                D2 = L.bgcj(C_D1, j2, z2);
                a2 = L.bgcj(C_A, j2, z2);
                if (k.g5) {
                    f2 = L.bgcj(C_F, j2, z2);
                    cH2 = L.bgcj(C_CH, j2, z2);
                }
                double xr = 0.0;
                const int jr = tabs ? L.tab_interval(r, &xr) : -1;
                if (g45) ren = L.ren(r2, l1, l2, r2 <= 1e-12, l1);
                if (k.T) {
                    t[0] = L.tabj(S00, jr, xr, r);
                    t[1] = L.tabj(S20, jr, xr, r);
                    t[2] = L.tabj(S11, jr, xr, r);
                    t[3] = L.tabj(S02, jr, xr, r);
                    t[4] = L.tabj(S13, jr, xr, r);
                    t[5] = L.tabj(S04, jr, xr, r);
                }
                if (k.P) {
                    t[6] = L.tabj(S31, jr, xr, r);
                    t[7] = L.tabj(S22, jr, xr, r);
                }
            }
            const double v = double_sum(a, k, v1, l2, r2, D2, a2, f2, cH2, ren, t);
            if (live) acc += wt * v;
            iu += dr;
            i1 += di;
            if (iu >= nuu) {
                iu -= nuu;
                ++i1;
            }
        }
        const double h2 = a.H0h * a.H0h;
        acc *= h2 * h2 / sp.chi2;
    }
    put_sum(acc, a.out + 2 * (first + blockIdx.x) + 1);
}

}  // namespace

extern "C" int ce_launch_integrated(void *stream, const ce_intg_dev *in, unsigned flags, int nz, const double *d_z,
                                    int nmu, const double *d_mu, int nsep, const double *d_sep, const int *rule,
                                    const double *d_gl, double *d_out)
{
    intg_args a;
    a.nbg = in->nbg;
    a.bg_z = in->bg_z;
    a.bg_chi = in->bg_chi;
    a.bg_D1 = in->bg_D1;
    a.bg_a = in->bg_a;
    a.bg_f = in->bg_f;
    a.bg_cH = in->bg_cH;
    a.bg_G1 = in->bg_G1;
    a.bg_G2 = in->bg_G2;
    a.nb = in->nb;
    a.bias_z = in->bias_z;
    a.b1 = in->b1;
    a.b2 = in->b2;
    a.nmb = in->nmb;
    a.mb_z = in->mb_z;
    a.s1 = in->s1;
    a.s2 = in->s2;
    a.fe1 = in->fe1;
    a.fe2 = in->fe2;
    a.tab_x = in->tab_x;
    a.tab_y = in->tab_y;
    for (int t = 0; t < NSLOT; ++t) {
        a.tab_off[t] = in->tab_off[t];
        a.tab_len[t] = in->tab_len[t];
        a.tab_f0[t] = in->tab_f0[t];
        a.tab_lx0[t] = in->tab_lx0[t];
        a.tab_lsc[t] = in->tab_lsc[t];
    }
    a.nguess = in->nguess;
    a.chi_guess = in->chi_guess;
    a.tab_ref = in->tab_ref;
    // records, then node pairs (ce_intg_coef_len): the shared nodes' tables and the
    // background curves wide, z(chi), then the other tables in tab_y's layout
    const int nsh = in->tab_ref < 0 ? 0 : in->tab_len[in->tab_ref];
    double *wide = in->coef, *bgw = wide + (size_t)WIDE * nsh, *zof = bgw + (size_t)BGW * in->nbg;
    double *own = zof + (size_t)ZOF * in->nbg, *tpair = own + (size_t)VAL * in->ntab_values;
    double *zpair = tpair + (size_t)PAIR * in->ntab_values;
    a.tab_wide = wide;
    a.tab_pair = tpair;
    a.bgc_wide = bgw;
    a.bgz_pair = zpair;
    a.zof = zof;
    coef_list cl;
    cl.ncurve = 0;
    int nmax = 0;
    for (int t = 0; t < NSLOT; ++t) {
        const bool shared = nsh && t != S40;
        double *val = shared ? wide + VAL * WSLOT[t] : own + (size_t)VAL * in->tab_off[t];
        a.tab_val[t] = val;
        a.tab_stride[t] = shared ? WIDE : VAL;
        if (in->tab_len[t] < 5) continue;
        const int q = cl.ncurve++;
        cl.x[q] = in->tab_x + in->tab_off[t];
        cl.y[q] = in->tab_y + in->tab_off[t];
        cl.n[q] = in->tab_len[t];
        cl.val[q] = val;
        cl.stride[q] = a.tab_stride[t];
        cl.pair[q] = tpair + (size_t)PAIR * in->tab_off[t];
        cl.pstride[q] = PAIR;
        nmax = cl.n[q] > nmax ? cl.n[q] : nmax;
    }
    const double *bx[NBGC] = {in->bg_z, in->bg_z, in->bg_z, in->bg_z, in->bg_chi};
    const double *by[NBGC] = {in->bg_D1, in->bg_a, in->bg_f, in->bg_cH, in->bg_z};
    for (int k = 0; k < NBGC; ++k) {
        const int q = cl.ncurve++;
        cl.x[q] = bx[k];
        cl.y[q] = by[k];
        cl.n[q] = in->nbg;
        cl.val[q] = k == C_ZOF ? zof + 2 : bgw + VAL * k;
        cl.stride[q] = k == C_ZOF ? ZOF : BGW;
        cl.pair[q] = k == C_ZOF ? zof : (k == C_D1 ? zpair : nullptr);
        cl.pstride[q] = k == C_ZOF ? ZOF : PAIR;
        nmax = in->nbg > nmax ? in->nbg : nmax;
    }
    hipLaunchKernelGGL(k_intg_coef, dim3((unsigned)((nmax + 255) / 256), (unsigned)cl.ncurve), dim3(256), 0,
                       (hipStream_t)stream, cl);
    a.nren0 = in->nren0;
    a.ren0_x = in->ren0_x;
    a.ren0_y = in->ren0_y;
    a.nren = in->nren;
    a.ren_chi = in->ren_chi;
    a.ren_rec = in->ren_rec;
    a.Om = in->Om;
    a.H0h = in->H0h;
    a.flags = flags;
    a.nz = nz;
    a.nmu = nmu;
    a.nsep = nsep;
    a.zmean = d_z;
    a.mu = d_mu;
    a.sep = d_sep;
    a.p1 = rule[0];
    a.n1 = rule[1];
    a.pu = rule[2];
    a.nu = rule[3];
    a.ps = rule[4];
    a.ns = rule[5];
    a.g1x = d_gl;
    a.g1w = d_gl + a.n1;
    a.gux = d_gl + 2 * a.n1;
    a.guw = a.gux + a.nu;
    a.gsx = a.guw + a.nu;
    a.gsw = a.gsx + a.ns;
    a.out = d_out;
    const int64_t blocks = (int64_t)nz * nmu * nsep;
    if (blocks <= 0 || blocks > 0x7fffffff) return (int)hipErrorInvalidValue;
    static_assert(sizeof(intg_args) <= CE_INTG_ARGS_BYTES, "intg_args outgrew its device slot");
    static_assert(NBGC == CE_INTG_NBGC, "background curves with segment records");
    hipError_t e = hipMemcpyAsync(in->args_dev, &a, sizeof(a), hipMemcpyHostToDevice, (hipStream_t)stream);
    if (e == hipSuccess) e = hipStreamSynchronize((hipStream_t)stream);   /* `a` is on this stack */
    if (e != hipSuccess) return (int)e;
    // the fetching variant where the tables that are read share their nodes, what it keeps in
    // LDS is small and its 16- and 32-bit indices hold; with the most wavefronts whose
    // buffers fit beside it
    const bool g45 = flags & (F_G4 | F_G5);
    const bool tabs = (flags & F_LEN) && (g45 || (!(flags & F_ONLY_CROSS) && !(flags & F_FLAT_LL)));
    const int n1 = (a.p1 + (a.p1 / 2 > 1 ? a.p1 / 2 : 1)) * a.n1;
    const int n40 = g45 ? a.tab_len[S40] : 0, nren = g45 ? a.nren : 0;
    const int f0 = nsh && a.tab_f0[a.tab_ref] > 0 ? a.tab_f0[a.tab_ref] : 0;
    const bool fetch = (!tabs || nsh) && n40 <= N40 && nren <= NREN && nsh <= (1 << 23) && a.nbg <= (1 << 16);
    int waves = fetch ? DWAVES : 0;
    while (waves > 4 && dlds(waves, n1, n40, nren, f0, a.nguess + 1).bytes > DLDS_MAX) --waves;
    const size_t lds = (size_t)(fetch ? dlds(waves, n1, n40, nren, f0, a.nguess + 1) : dlds(0, n1, 0, 0, 0, 0)).bytes;
    if (fetch) {
        // the most of any call: threads whose calls differ in size don't lower each other's limit
        e = hipFuncSetAttribute((const void *)k_integrated_double<true>, hipFuncAttributeMaxDynamicSharedMemorySize, DLDS_MAX);
        if (e != hipSuccess) return (int)e;
    }
    const intg_args *d_args = (const intg_args *)in->args_dev;
    pt *pts = (pt *)in->points;
    static_assert(sizeof(pt) <= CE_INTG_POINT * sizeof(double), "a point outgrew its record");
    for (int64_t first = 0; first < blocks; first += CE_INTG_POINTS) {
        const int count = (int)(blocks - first < CE_INTG_POINTS ? blocks - first : CE_INTG_POINTS);
        hipLaunchKernelGGL(k_intg_points, dim3((unsigned)(count + 63) / 64), dim3(64), 0, (hipStream_t)stream, d_args, first,
                           count, pts);
        hipLaunchKernelGGL(k_integrated_single, dim3((unsigned)count), dim3(256), 0, (hipStream_t)stream, d_args,
                           (const pt *)pts, first);
        if (fetch)
            hipLaunchKernelGGL(k_integrated_double<true>, dim3((unsigned)count), dim3(64 * waves), lds, (hipStream_t)stream,
                               d_args, (const pt *)pts, first);
        else
            hipLaunchKernelGGL(k_integrated_double<false>, dim3((unsigned)count), dim3(256), lds, (hipStream_t)stream, d_args,
                               (const pt *)pts, first);
    }
    return (int)hipGetLastError();
}
