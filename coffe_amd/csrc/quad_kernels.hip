// Small-separation nodes of the I_l^n tables (gfx950, FP64).
//
// Below the FFTLog grid the reference fills each table with 43 direct integrals
// (integrals.c:520-557, min_sep of integrals.c:111-126):
//   node 0:      r = 0, (1/2pi^2) int dk k^(2+l-n) P(k) / (2l+1)!!   if n >= l, else 0
//                (integrals.c:238-269, coefficient 215-231)
//   node i > 0:  r = min_sep[i-1], (1/2pi^2) int dk k^2 P(k) j_l(kr)/(kr)^n, times r^(n-l)
//                if n >= l (integrals.c:280-325)
// over [kmin, kmax], P(k) the Akima spline of the input samples, by QUADPACK QAG
// with the 61-point Gauss-Kronrod rule, epsabs 0, epsrel 1e-5 (common.c:1004-1040).
//
// One wavefront runs one adaptive integration: lane j evaluates Kronrod node j of both
// halves of the interval being refined, the Gauss / Kronrod / |f| / |f - mean| sums are
// reduced with DPP adds, and lane i holds interval i of the list (a, b, result, error)
// in registers.  Every lane holds the same reduced values, so the control flow of the
// bisection loop is uniform across the wavefront.  The few integrals that need more than
// 64 intervals (the r = 0 renormalisation below 0.01 Mpc, of the divergent tables) are left to
// a second kernel with the list in LDS (cap CE_QAG_CAP).
//
// What bounds it: the bisections are serial, and a step was a chain of a ten-step search of
// the samples in L2, nine divisions for the Akima coefficients, series loops and shuffles,
// twice, with five wavefronts a CU (32 KB of LDS list each).  The spline's coefficients
// and an index of its nodes by their leading bits now sit in LDS, shared by a workgroup's
// wavefronts, and sixteen wavefronts fit a CU: the FP64 units now bound it (two sines and a
// division a node).  40,995 integrals of about 20 intervals, 600
// samples: 1.12 against 8.2 ms.
#include <float.h>
#include <hip/hip_runtime.h>

#include "ce_device.h"
#include "ce_internal.h"
#include "gk61_nodes.h"

namespace {

__constant__ double c_min_sep[CE_MIN_SEP_LEN];
__constant__ double c_xgk[31], c_wgk[31], c_wg[15];

// lane i (uniform) of v
__device__ __forceinline__ double read_lane(double v, int i)
{
    return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), i),
                            __builtin_amdgcn_readlane(__double2loint(v), i));
}

// v of the lane that DPP control C names; lanes without one keep `own`
template <int C, int ROWS = 0xf>
__device__ __forceinline__ double dpp(double own, double v)
{
    return __hiloint2double(
        __builtin_amdgcn_update_dpp(__double2hiint(own), __double2hiint(v), C, ROWS, 0xf, false),
        __builtin_amdgcn_update_dpp(__double2loint(own), __double2loint(v), C, ROWS, 0xf, false));
}

// sum and maximum over the wavefront, in every lane: shifts by 1, 2, 4, 8 inside the rows of
// 16, then the rows' last lanes broadcast on (0x142, 0x143), the total in lane 63
__device__ __forceinline__ double wave_sum(double v)
{
    v += dpp<0x111>(0.0, v);
    v += dpp<0x112>(0.0, v);
    v += dpp<0x114>(0.0, v);
    v += dpp<0x118>(0.0, v);
    v += dpp<0x142, 0xa>(0.0, v);
    v += dpp<0x143, 0xc>(0.0, v);
    return read_lane(v, 63);
}
__device__ __forceinline__ double wave_max(double v)
{
    v = fmax(v, dpp<0x111>(v, v));
    v = fmax(v, dpp<0x112>(v, v));
    v = fmax(v, dpp<0x114>(v, v));
    v = fmax(v, dpp<0x118>(v, v));
    v = fmax(v, dpp<0x142, 0xa>(v, v));
    v = fmax(v, dpp<0x143, 0xc>(v, v));
    return read_lane(v, 63);
}

// x^n, integer n (a few products: pow() costs more than the rest of an integrand)
__device__ __forceinline__ double ipow(double x, int n)
{
    const int m = n < 0 ? -n : n;
    double p = 1.0;
    for (int i = 0; i < m; ++i) p *= x;
    return n < 0 ? 1.0 / p : p;
}

// j_0: sin(x) / x has no cancellation
__device__ __forceinline__ double sph_j0(double x) { return x == 0.0 ? 1.0 : sin(x) / x; }

// spherical Bessel j_l(x), integer 0 <= l <= 4, x >= 0 (GSL sf_bessel_jl is called at
// integrals.c:309-316): upward recurrence from j_0, j_1 for x > l, else the power series, whose
// alternating terms fall from the first on there (x^2 <= 2 (2 l + 3) for l <= 5).  rc: lane k
// holds 1 / (k (2 l + 2 k + 1)).
__device__ double sph_jl(int l, double x, double rc)
{
    if (l == 0) return sph_j0(x);
    const bool ser = x <= (double)l;
    double res = 0.0;
    if (!ser) {
        double s, c;
        sincos(x, &s, &c);
        const double ix = 1.0 / x;
        double jm = s * ix, jc = (jm - c) * ix;
        for (int k = 1; k < l; ++k) {
            const double jn = (2.0 * k + 1.0) * ix * jc - jm;
            jm = jc;
            jc = jn;
        }
        res = jc;
    }
    if (__ballot(ser) != 0) {   // every lane of the wavefront is here: read_lane's rc
        double pre = 1.0;
        for (int k = 1; k <= l; ++k) pre *= x / (2.0 * k + 1.0);
        const double y = ser ? -0.5 * x * x : 0.0;
        double term = 1.0, sum = 1.0;
        for (int k = 1; k < 40; ++k) {
            term *= y * read_lane(rc, k);
            sum += term;
            if (__ballot(fabs(term) >= 1e-18 * fabs(sum)) == 0) break;
        }
        if (ser) res = pre * sum;
    }
    return res;
}

// cylindrical Bessel J_m(x), integer m >= 0, x >= 0 (the half-integer tables' small-r
// integrand calls GSL's sf_bessel_Jn, integrals.c:296-306): power series below 2,
// Hankel's asymptotic expansion from 25 on (the terms of P and Q fall below 1e-17
// there for the orders used), otherwise Miller's downward recurrence normalised with
// J_0 + 2 sum_k J_2k = 1, started 30 orders above max(m, x)
__device__ double cyl_jn(int m, double x)
{
    if (x == 0.0) return m == 0 ? 1.0 : 0.0;
    if (x < 2.0) {
        double pre = 1.0;
        for (int i = 1; i <= m; ++i) pre *= 0.5 * x / i;
        const double y = -0.25 * x * x;
        double term = 1.0, sum = 1.0;
        for (int k = 1; k < 40; ++k) {
            term *= y / (k * (double)(k + m));
            sum += term;
            if (fabs(term) < 1e-18 * fabs(sum)) break;
        }
        return pre * sum;
    }
    const double pi = 3.14159265358979323846;
    if (x >= 25.0) {
        const double mu = 4.0 * m * m;
        double P = 1.0, Q = 0.0, ak = 1.0;
        for (int k = 1; k < 60; ++k) {
            ak *= (mu - (2.0 * k - 1.0) * (2.0 * k - 1.0)) / (k * 8.0 * x);
            if (k & 1)
                Q += (((k - 1) / 2) & 1) ? -ak : ak;
            else
                P += ((k / 2) & 1) ? -ak : ak;
            if (fabs(ak) < 1e-17) break;
        }
        double sn, cs;
        sincos(x - (0.5 * m + 0.25) * pi, &sn, &cs);
        return sqrt(2.0 / (pi * x)) * (P * cs - Q * sn);
    }
    const int top = m > (int)x ? m : (int)x;
    const int N = 2 * ((top + 30) / 2 + 1);
    double fp = 0.0, fc = 1e-30, fm = 0.0, norm = 0.0;
    for (int k = N; k > 0; --k) {
        if (k == m) fm = fc;
        if ((k & 1) == 0) norm += 2.0 * fc;
        const double fn = 2.0 * k / x * fc - fp;
        fp = fc;
        fc = fn;
        if (fabs(fc) > 1e250) {
            fc *= 1e-250;
            fp *= 1e-250;
            fm *= 1e-250;
            norm *= 1e-250;
        }
    }
    if (m == 0) fm = fc;
    norm += fc;
    return fm / norm;
}

// integrands over k of the Akima spline P(k) of the input samples
enum {
    SR_BESSEL = 0,    // k^2 P j_l(k r) / (k r)^n              (integrals.c:280-325)
    SR_PREFACTOR = 1, // k^(2+l-n) P                            (integrals.c:238-269)
    SR_RENORM0 = 2,   // P (1 - j_0(k r)^2) / k^2                (integrals.c:389-398)
    SR_RENORM = 3     // P j_0(k r) j_0(k r2) / k^2              (integrals.c:405-417)
};

struct sr_unit {
    int n, l;
    double r, r2;
    int kind;
    // half-integer table (n, l both half-integers, integrals.c:186-207): nd, ld are
    // n and l, and the kernel is sqrt(pi/2) J_{l+1/2}(kr) / (kr)^(n+1/2) = j_l(kr)/(kr)^n
    int half;
    double nd, ld;
};

// The Akima spline of the samples as a workgroup's wavefronts read it: coefficients and an index
// of the intervals in LDS (LDS = true), or the samples themselves where they do not fit
// (LDS = false: a bisection in L2 and the coefficients anew at every value).
#define CE_SPL_BUCKETS 1024
// samples in LDS: 40 bytes each of the CU's 160 KB, which beside them hold the second kernel's list.
// At 2999 samples, LDS against L2: 4194 divergent integrals 539 and 499 us, 40995 2588 and 2556, 2000
// 317 and 360; small-r nodes 83 and 90 (344), 283 and 343 (13760): even there, far ahead below
// (1293 against 2324 us for 40995 integrals at 600)
#define CE_SPL_MAX 3000
struct lds_spline {
    const double *x;        // [n]
    const double2 *yb, *cd; // [n]: value and coefficients of the interval from node j
    const unsigned short *idx;   // [CE_SPL_BUCKETS + 1]: interval of each bucket's lower edge
    int base, shift, nb;
};
template <bool LDS>
struct spline {
    const double *k, *p;
    int n;
    double x0, x1;
    lds_spline s;
};

// a bucket is a step of the leading bits of a (positive) double: 2^-s octave
__device__ __forceinline__ int key_of(double v, int shift) { return __double2hiint(v) >> shift; }

__host__ __device__ inline size_t spline_bytes(int n)
{
    return (size_t)n * 40 + (CE_SPL_BUCKETS + 8) * sizeof(unsigned short);
}

// the workgroup fills sp.s for values in [lo, hi], lo > 0; ends with a barrier
template <bool LDS>
__device__ void spline_load(spline<LDS> &sp, const double *k, const double *p, int n, double lo, double hi, char *mem)
{
    sp.k = k;
    sp.p = p;
    sp.n = n;
    sp.x0 = k[0];
    sp.x1 = k[n - 1];
    if (!LDS) return;
    double2 *yb = (double2 *)mem, *cd = yb + n;
    double *x = (double *)(cd + n);
    unsigned short *idx = (unsigned short *)(x + n);
    int shift = 14;   // 64 buckets an octave, or as many as there is room for
    while (key_of(hi, shift) - key_of(lo, shift) + 1 > CE_SPL_BUCKETS) ++shift;
    sp.s.shift = shift;
    sp.s.base = key_of(lo, shift);
    sp.s.nb = key_of(hi, shift) - sp.s.base + 1;
    sp.s.x = x;
    sp.s.yb = yb;
    sp.s.cd = cd;
    sp.s.idx = idx;
    for (int j = threadIdx.x; j < n; j += blockDim.x) {
        x[j] = k[j];
        const ce::akima_cf<double> c = ce::akima_coefs<double>(k, nullptr, p, nullptr, n, j < n - 1 ? j : n - 2);
        yb[j] = make_double2(c.y0, c.b);
        cd[j] = make_double2(c.c, c.d);
    }
    for (int b = threadIdx.x; b <= sp.s.nb; b += blockDim.x) {
        const double edge = __hiloint2double((sp.s.base + b) << shift, 0);
        int j = 0;
        if (edge >= k[n - 1]) j = n - 2;
        else if (edge > k[0]) j = ce::interval_bisect(k, 0, n - 1, edge);
        idx[b] = (unsigned short)j;
    }
    __syncthreads();
}

// the spline at v; NaN outside the samples (as ce::akima_general)
template <bool LDS>
__device__ __forceinline__ double spline_at(const spline<LDS> &sp, double v)
{
    if (!LDS) return ce::akima_general(sp.k, sp.p, sp.n, v);
    const int b = min(max(key_of(v, sp.s.shift) - sp.s.base, 0), sp.s.nb - 1);
    int lo = sp.s.idx[b], hi = min((int)sp.s.idx[b + 1] + 1, sp.n - 1);
    while (hi > lo + 1) {
        const int m = (lo + hi) >> 1;
        if (sp.s.x[m] > v) hi = m;
        else lo = m;
    }
    const double t = v - sp.s.x[lo];
    const double2 yb = sp.s.yb[lo], cd = sp.s.cd[lo];
    const double r = yb.x + t * (yb.y + t * (cd.x + cd.y * t));
    return v >= sp.x0 && v <= sp.x1 ? r : __builtin_nan("");
}

template <bool LDS>
__device__ __forceinline__ double integrand(const sr_unit &u, const spline<LDS> &sp, double k, double rc)
{
    const double pk = spline_at(sp, k);
    const double sqrt_pi_2 = 1.25331413731550025121;
    if (u.half && u.kind == SR_PREFACTOR) return sqrt_pi_2 * pow(k, 2.0 + u.ld - u.nd) * pk;
    if (u.half && u.kind == SR_BESSEL) {
        const double x = k * u.r;
        return k * k * pk * sqrt_pi_2 * cyl_jn((int)(u.ld + 0.5), x) / pow(x, u.nd + 0.5);
    }
    switch (u.kind) {
    case SR_PREFACTOR: return ipow(k, 2 + u.l - u.n) * pk;
    case SR_RENORM0: {
        const double x = fabs(k * u.r);
        // 1 - j0^2 ~ x^2 / 3 keeps what the rounding of j0 leaves: the series is the closer
        // one below 0.5 (at most half a unit off)
        double j0 = sph_j0(x), term = 1.0, sum = 1.0;
        const double y = x < 0.5 ? -0.5 * x * x : 0.0;
        for (int i = 1; i < 20 && __ballot(term != 0.0 && fabs(term) >= 1e-18 * fabs(sum)) != 0; ++i) {
            term *= y * read_lane(rc, i);
            sum += term;
        }
        if (x < 0.5) j0 = sum;
        return pk * (1. - j0 * j0) / (k * k);
    }
    case SR_RENORM: {
        // the product of the two Bessel factors first: symmetric in (r, r2) bit for bit
        // (j_0 is 1 below 1e-8; from 1e-100 down, so that the product below does not underflow)
        const double xa = k * u.r, xb = k * u.r2;
        const bool za = fabs(xa) < 1e-100, zb = fabs(xb) < 1e-100;
        const double ss = (za ? 1.0 : sin(xa)) * (zb ? 1.0 : sin(xb));
        return pk * ss / ((za ? 1.0 : xa) * (zb ? 1.0 : xb) * (k * k));
    }
    default: {
        const double x = k * u.r;
        return k * k * pk * sph_jl(u.l, x, rc) * ipow(x, -u.n);
    }
    }
}

struct qk_out {
    double result, abserr, resabs, resasc;
};

// a lane's node of the 61-point rule: lane j < 61 evaluates node j (j < 30: the left half,
// j = 30: the centre, j > 30: the right half) at centre + half x; the other lanes repeat the
// last one with weight 0
struct qk_lane {
    double x, wk, wg, rc;
};
__device__ __forceinline__ qk_lane qk_node(int lane, int l)
{
    qk_lane q;
    const int i = min(lane, 60), j = i <= 30 ? i : 60 - i;   // QUADPACK index of the node
    q.x = i < 30 ? -c_xgk[j] : (i == 30 ? 0.0 : c_xgk[j]);
    q.wk = lane < 61 ? c_wgk[j] : 0.0;
    q.wg = lane < 61 && (j & 1) ? c_wg[j >> 1] : 0.0;
    q.rc = lane ? 1.0 / (lane * (2.0 * l + 2.0 * lane + 1.0)) : 0.0;
    return q;
}

__device__ __forceinline__ qk_out qk_finish(double rk, double rg, double rabs, double rasc, double half)
{
    qk_out o;
    double err = fabs((rk - rg) * half);
    o.result = rk * half;
    o.resabs = rabs * fabs(half);
    o.resasc = rasc * fabs(half);
    if (o.resasc != 0.0 && err != 0.0) {
        const double t = 200.0 * err / o.resasc, scale = t * sqrt(t);
        err = scale < 1.0 ? o.resasc * scale : o.resasc;
    }
    if (o.resabs > DBL_MIN / (50.0 * DBL_EPSILON)) {
        const double min_err = 50.0 * DBL_EPSILON * o.resabs;
        if (min_err > err) err = min_err;
    }
    o.abserr = err;
    return o;
}

// QUADPACK qk61 on [a, b]
template <bool LDS>
__device__ __forceinline__ qk_out qk61(const sr_unit &u, const spline<LDS> &sp, const qk_lane &q, double a, double b)
{
    const double half = 0.5 * (b - a);
    const double f = integrand(u, sp, 0.5 * (a + b) + half * q.x, q.rc);
    // a node with weight 0 adds 0, not a NaN
    const double fw = q.wk != 0.0 ? f : 0.0;
    const double rk = wave_sum(q.wk * fw), rg = wave_sum(q.wg * fw), rabs = wave_sum(q.wk * fabs(fw));
    const double rasc = wave_sum(q.wk * fabs(fw - 0.5 * rk));
    return qk_finish(rk, rg, rabs, rasc, half);
}

// the two halves of an interval, their sums side by side
template <bool LDS>
__device__ __forceinline__ void qk61_pair(const sr_unit &u, const spline<LDS> &sp, const qk_lane &q, double a, double m,
                                          double b, qk_out &o1, qk_out &o2)
{
    const double h1 = 0.5 * (m - a), h2 = 0.5 * (b - m);
    const double e1 = integrand(u, sp, 0.5 * (a + m) + h1 * q.x, q.rc);
    const double e2 = integrand(u, sp, 0.5 * (m + b) + h2 * q.x, q.rc);
    const double f1 = q.wk != 0.0 ? e1 : 0.0, f2 = q.wk != 0.0 ? e2 : 0.0;
    const double k1 = wave_sum(q.wk * f1), k2 = wave_sum(q.wk * f2);
    const double g1 = wave_sum(q.wg * f1), g2 = wave_sum(q.wg * f2);
    const double a1 = wave_sum(q.wk * fabs(f1)), a2 = wave_sum(q.wk * fabs(f2));
    const double s1 = wave_sum(q.wk * fabs(f1 - 0.5 * k1)), s2 = wave_sum(q.wk * fabs(f2 - 0.5 * k2));
    o1 = qk_finish(k1, g1, a1, s1, h1);
    o2 = qk_finish(k2, g2, a2, s2, h2);
}

// the interval list of one integral: lane i's registers hold interval i (up to 64), or LDS holds
// them (up to CE_QAG_CAP).  largest(): the interval with the largest error, the first on ties.
struct list_regs {
    static constexpr int cap = 64;
    int lane;
    double a, b, r, e;
    __device__ void init(int l, double *)
    {
        lane = l;
        a = b = r = 0.0;
        e = -1.0;
    }
    __device__ void get(int i, double &ia, double &ib, double &ir, double &ie) const
    {
        ia = read_lane(a, i);
        ib = read_lane(b, i);
        ir = read_lane(r, i);
        ie = read_lane(e, i);
    }
    __device__ void put(int i, double ia, double ib, double ir, double ie)
    {
        if (lane == i) {
            a = ia;
            b = ib;
            r = ir;
            e = ie;
        }
    }
    __device__ int largest(int size) const
    {
        const double m = wave_max(lane < size ? e : -1.0);
        const unsigned long long hit = __ballot(lane < size && e == m);
        return hit ? __builtin_ctzll(hit) : 0;
    }
    __device__ double sum(int) const { return wave_sum(r); }
};
struct list_lds {
    static constexpr int cap = CE_QAG_CAP;
    int lane;
    double *ia, *ib, *ir, *ie;
    __device__ void init(int l, double *mem)
    {
        lane = l;
        ia = mem;
        ib = ia + cap;
        ir = ib + cap;
        ie = ir + cap;
    }
    __device__ void get(int i, double &a, double &b, double &r, double &e) const
    {
        a = ia[i];
        b = ib[i];
        r = ir[i];
        e = ie[i];
    }
    __device__ void put(int i, double a, double b, double r, double e)
    {
        __syncthreads();   // one wavefront per workgroup: the list's earlier reads are done
        if (lane == 0) {
            ia[i] = a;
            ib[i] = b;
            ir[i] = r;
            ie[i] = e;
        }
        __syncthreads();
    }
    __device__ int largest(int size) const
    {
        double be = -1.0;
        int bi = 0x7fffffff;
        for (int k = lane; k < size; k += 64)
            if (ie[k] > be) { be = ie[k]; bi = k; }
        const double m = wave_max(be);
        int best = be == m ? bi : 0x7fffffff;   // the first of the lanes' firsts
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) best = min(best, __shfl_xor(best, off, 64));
        return best < size ? best : 0;
    }
    __device__ double sum(int size) const
    {
        double part = 0.0;
        for (int k = lane; k < size; k += 64) part += ir[k];
        return wave_sum(part);
    }
};

#define QAG_MORE (-1)   // more intervals than the list holds: the integral is left to the next kernel

// QUADPACK QAG (epsabs 0, the 61-point rule) of u over [lo, hi] by one wavefront; every lane
// returns the same sum.  Status: 0 converged, 1 interval limit (CE_QAG_CAP), 2 roundoff,
// 3 bad integrand behaviour, QAG_MORE.
template <class List, bool LDS>
__device__ int qag_wave(const sr_unit &u, const spline<LDS> &sp, double lo, double hi, double epsrel, int lane,
                        double *mem, double &result, int &nint)
{
    const qk_lane q = qk_node(lane, u.l);
    nint = 1;
    const qk_out q0 = qk61(u, sp, q, lo, hi);
    int st = 0;
    result = q0.result;
    double tol = epsrel * fabs(q0.result);
    const double round_off = 50.0 * DBL_EPSILON * q0.resabs;
    const bool done0 = (q0.abserr <= round_off && q0.abserr > tol) ||
                       (q0.abserr <= tol && q0.abserr != q0.resasc) || q0.abserr == 0.0;
    if (q0.abserr <= round_off && q0.abserr > tol) st = 2;
    if (done0) return st;
    List list;
    list.init(lane, mem);
    list.put(0, lo, hi, q0.result, q0.abserr);
    int size = 1, imax = 0, iter = 1, rt1 = 0, rt2 = 0;
    double area = q0.result, errsum = q0.abserr;
    do {
        double a1, b2, ri, ei;
        list.get(imax, a1, b2, ri, ei);
        const double b1 = 0.5 * (a1 + b2), a2 = b1;
        qk_out q1, q2;
        qk61_pair(u, sp, q, a1, b1, b2, q1, q2);
        const double area12 = q1.result + q2.result, err12 = q1.abserr + q2.abserr;
        errsum += err12 - ei;
        area += area12 - ri;
        if (q1.resasc != q1.abserr && q2.resasc != q2.abserr) {
            const double delta = ri - area12;
            if (fabs(delta) <= 1.0e-5 * fabs(area12) && err12 >= 0.99 * ei) rt1++;
            if (iter >= 10 && err12 > ei) rt2++;
        }
        tol = epsrel * fabs(area);
        if (errsum > tol) {
            if (rt1 >= 6 || rt2 >= 20) st = 2;
            const double tmp = (1 + 100 * DBL_EPSILON) * (fabs(a2) + 1000 * DBL_MIN);
            if (fabs(a1) <= tmp && fabs(b2) <= tmp) st = 3;
        }
        // the refined interval keeps the half with the larger error
        const bool right = q2.abserr > q1.abserr;
        list.put(imax, right ? a2 : a1, right ? b2 : b1, right ? q2.result : q1.result, right ? q2.abserr : q1.abserr);
        list.put(size, right ? a1 : a2, right ? b1 : b2, right ? q1.result : q2.result, right ? q1.abserr : q2.abserr);
        size++;
        iter++;
        if (iter >= CE_QAG_CAP && errsum > tol && !st) st = 1;
        if (iter >= CE_QAG_CAP || st || !(errsum > tol)) break;
        if (size >= List::cap) return QAG_MORE;
        imax = list.largest(size);
    } while (true);
    result = list.sum(size);
    nint = size;
    return st;
}

struct sr_args {
    int nspec, ntab;
    const ce_spec_dev *spec;
    const ce_grid_dev *grids;
    const ce_table_desc *tabs;
    const double *k, *p;
    double epsrel;
    double *out;      // [nspec][ntab][1 + CE_MIN_SEP_LEN]
    int *status;      // same layout: 0 converged, 1 interval limit, 2 roundoff, 3 bad integrand
};

// the integral of `unit` = (spectrum, table, node); false: its value is 0
__device__ __forceinline__ bool small_r_unit(const sr_args &a, int unit, sr_unit &u)
{
    constexpr int NODES = 1 + CE_MIN_SEP_LEN;
    const int node = unit % NODES;
    const int t = (unit / NODES) % a.ntab;
    u.n = (int)a.tabs[t].n;
    u.l = (int)a.tabs[t].l;
    u.nd = a.tabs[t].n;
    u.ld = a.tabs[t].l;
    u.half = u.ld != floor(u.ld);
    u.kind = node == 0 ? SR_PREFACTOR : SR_BESSEL;
    u.r = node == 0 ? 0.0 : c_min_sep[node - 1];
    u.r2 = 0.0;
    return !(node == 0 && (u.half ? u.nd < u.ld : u.n < u.l));   // I_l^n(0) = 0 for n < l
}

__device__ void small_r_store(const sr_args &a, int unit, const sr_unit &u, double result, int st)
{
    const double pi = 3.14159265358979323846;
    double v = result / 2. / pi / pi;
    if (u.kind == SR_PREFACTOR && u.half) {
        // 2^(l+1/2) Gamma(l+3/2) = 2^m m!, m = l + 1/2 (integrals.c:215-231)
        const int m = (int)(u.ld + 0.5);
        double c = 1.0;
        for (int i = 1; i <= m; ++i) c *= 2.0 * i;
        v /= c;
    } else if (u.kind == SR_PREFACTOR) {
        double df = 1.0;   // (2l+1)!! = 2^(l+1/2) Gamma(l+3/2) / sqrt(pi/2)
        for (int i = 3; i <= 2 * u.l + 1; i += 2) df *= i;
        v /= df;
    } else if (u.half ? u.nd >= u.ld : u.n >= u.l) {
        v *= u.half ? pow(u.r, u.nd - u.ld) : pow(u.r, (double)(u.n - u.l));
    }
    if (!isfinite(v) && st == 0) st = 3;
    a.out[unit] = v;
    a.status[unit] = st;
}

// one wavefront per (spectrum, table, node); a workgroup's wavefronts share a spectrum
// (blockIdx.y) and its spline
template <class List, bool LDS>
__global__ void __launch_bounds__(512) k_small_r(sr_args a, size_t list_bytes)
{
    extern __shared__ double2 quad_lds[];
    const int lane = threadIdx.x & 63, nw = blockDim.x >> 6;
    const int per = a.ntab * (1 + CE_MIN_SEP_LEN);
    const int s = blockIdx.y;
    const ce_spec_dev spec = a.spec[s];
    const ce_grid_dev &g = a.grids[spec.grid];
    const bool again = List::cap != 64;   // only what the first kernel left
    spline<LDS> sp;
    if (again) {
        int any = 0;
        for (int e = lane; e * (int)gridDim.x + (int)blockIdx.x < per; e += 64)
            any |= a.status[(int64_t)s * per + e * (int)gridDim.x + (int)blockIdx.x] == QAG_MORE;
        if (!__ballot(any)) return;
    }
    spline_load(sp, a.k + spec.in_off, a.p + spec.in_off, spec.n_in, g.kmin, g.kmax, (char *)quad_lds + list_bytes);
    for (int e = blockIdx.x * nw + (threadIdx.x >> 6); e < per; e += gridDim.x * nw) {
        const int unit = s * per + e;
        if (again && a.status[unit] != QAG_MORE) continue;
        sr_unit u;
        if (!small_r_unit(a, unit, u)) {
            if (lane == 0) {
                a.out[unit] = 0.0;
                a.status[unit] = 0;
            }
            continue;
        }
        double result;
        int nint;
        const int st = qag_wave<List>(u, sp, g.kmin, g.kmax, a.epsrel, lane, (double *)quad_lds, result, nint);
        if (lane == 0) {
            if (st == QAG_MORE) a.status[unit] = st;
            else small_r_store(a, unit, u, result, st);
        }
    }
}

struct div_args {
    const double *k, *p;   // input samples of the spectrum
    int n_in;
    double kmin, kmax, epsrel;
    const double *sep;     // [nsep]
    int nsep;
    const double *chi;     // [nchi]
    int nchi;
    double *i40, *r0;      // [nsep] each
    double *ren;           // [nchi][nchi]: (chi[j], chi[i]) at i nchi + j
    int *status;           // [2 nsep + nchi^2]: the QAG status, 4 for a non-finite value
    int *nint;             // same layout: final interval count, or null
};

// the divergent table I_0^4 and its renormalisations (integrals.c:772-909), one
// wavefront per integral: units [0, nsep) I_0^4(sep) sep^4, [nsep, 2 nsep) the r = 0
// renormalisation at sep (times sep^4 as well, integrals.c:351-356, n = 4, l = 0), then
// the nchi^2 grid of int P j_0 j_0 / k^2; all divided by 2 pi^2.  The wavefronts stride over
// the units, so that neighbours (which cost alike) go to different workgroups.
template <class List, bool LDS>
__global__ void __launch_bounds__(256, 4) k_divergent(div_args a, size_t list_bytes)
{
    extern __shared__ double2 quad_lds[];
    const int lane = threadIdx.x & 63, nw = blockDim.x >> 6;
    const int units = 2 * a.nsep + a.nchi * a.nchi;
    const int stride = gridDim.x * nw;
    const bool again = List::cap != 64;   // only what the first kernel left
    if (again) {
        int any = 0;
        for (int64_t e = (int64_t)lane * stride + blockIdx.x; e < units; e += (int64_t)64 * stride)
            any |= a.status[e] == QAG_MORE;
        if (!__ballot(any)) return;
    }
    spline<LDS> sp;
    spline_load(sp, a.k, a.p, a.n_in, a.kmin, a.kmax, (char *)quad_lds + list_bytes);
    sr_unit u;
    u.n = 4;
    u.l = 0;
    u.half = 0;
    u.nd = 4.0;
    u.ld = 0.0;
    for (int unit = (threadIdx.x >> 6) * gridDim.x + blockIdx.x; unit < units; unit += stride) {
        if (again && a.status[unit] != QAG_MORE) continue;
        u.r2 = 0.0;
        if (unit < 2 * a.nsep) {
            u.kind = unit < a.nsep ? SR_BESSEL : SR_RENORM0;
            u.r = a.sep[unit < a.nsep ? unit : unit - a.nsep];
        } else {
            const int q = unit - 2 * a.nsep;
            u.kind = SR_RENORM;
            u.r = a.chi[q % a.nchi];
            u.r2 = a.chi[q / a.nchi];
        }
        double result;
        int nint;
        int st = qag_wave<List>(u, sp, a.kmin, a.kmax, a.epsrel, lane, (double *)quad_lds, result, nint);
        if (lane != 0) continue;
        if (st == QAG_MORE) {
            a.status[unit] = st;
            continue;
        }
        const double pi = 3.14159265358979323846;
        if (a.nint) a.nint[unit] = nint;
        double v = result;
        if (u.kind != SR_RENORM && u.r > 0) v *= pow(u.r, 4.0);
        v = v / 2. / pi / pi;
        if (!isfinite(v)) st = 4;
        if (unit < a.nsep) a.i40[unit] = v;
        else if (unit < 2 * a.nsep) a.r0[unit - a.nsep] = v;
        else a.ren[unit - 2 * a.nsep] = v;
        a.status[unit] = st;
    }
}

constexpr size_t LIST_BYTES = 4 * CE_QAG_CAP * sizeof(double);

// always a kernel's own most: threads whose launches differ in size don't lower each other's limit
template <class F>
hipError_t lds_limit(F *fn, size_t bytes)
{
    return hipFuncSetAttribute((const void *)fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes);
}

// first the kernel with the list in registers, then the one with the list in LDS for what it left
template <bool LDS>
hipError_t launch_small_r(const sr_args &all, size_t sbytes, hipStream_t s)
{
    const int per = all.ntab * (1 + CE_MIN_SEP_LEN);
    // eight wavefronts share a spline, also where the integrals do not fill the chip: making it
    // takes eight times as long in one wavefront, and above 2000 samples (more than half a CU's
    // LDS) a CU then runs one wavefront.  1720 integrals: 77 us at 600 samples and 86 at 2999,
    // against 123 and 629 with one wavefront, 80 and 126 with four; 43 integrals of 600: 69, 83, 68.
    const int nw = 8;
    const size_t smost = LDS ? spline_bytes(CE_SPL_MAX) : 0;
    hipError_t e = lds_limit(k_small_r<list_regs, LDS>, smost);
    if (e == hipSuccess) e = lds_limit(k_small_r<list_lds, LDS>, LIST_BYTES + smost);
    for (int s0 = 0; s0 < all.nspec && e == hipSuccess; s0 += 32768) {   // the grid's y range
        sr_args a = all;
        a.nspec = all.nspec - s0 < 32768 ? all.nspec - s0 : 32768;
        a.spec += s0;
        a.out += (int64_t)s0 * per;
        a.status += (int64_t)s0 * per;
        hipLaunchKernelGGL((k_small_r<list_regs, LDS>), dim3((per + nw - 1) / nw, a.nspec), dim3(64 * nw), sbytes, s, a,
                           (size_t)0);
        hipLaunchKernelGGL((k_small_r<list_lds, LDS>), dim3(per < 64 ? per : 64, a.nspec), dim3(64),
                           LIST_BYTES + sbytes, s, a, LIST_BYTES);
        e = hipGetLastError();
    }
    return e;
}

template <bool LDS>
hipError_t launch_divergent(const div_args &a, int units, size_t sbytes, hipStream_t s)
{
    const size_t smost = LDS ? spline_bytes(CE_SPL_MAX) : 0;
    hipError_t e = lds_limit(k_divergent<list_regs, LDS>, smost);
    if (e == hipSuccess) e = lds_limit(k_divergent<list_lds, LDS>, LIST_BYTES + smost);
    if (e != hipSuccess) return e;
    // four wavefronts share a spline, whatever the number of integrals (2000 of them: 214 us at 600
    // samples and 317 at 2999, against 306 and 1216 with a spline a wavefront, 218 and 557 with
    // two); two rounds of the workgroups that are resident at once (40995 integrals, 600 samples, 128
    // VGPRs: 1116 us, against 1186 with one round, 1195 with eight wavefronts, 1296 at 168 VGPRs
    // and 1379 at 256)
    const int nw = 4;
    const int wg = (units + nw - 1) / nw, most = 2048;
    hipLaunchKernelGGL((k_divergent<list_regs, LDS>), dim3(wg < most ? wg : most), dim3(64 * nw), sbytes, s, a,
                       (size_t)0);
    hipLaunchKernelGGL((k_divergent<list_lds, LDS>), dim3(units < 512 ? units : 512), dim3(64), LIST_BYTES + sbytes, s, a,
                       LIST_BYTES);
    return hipGetLastError();
}

}  // namespace

extern "C" int ce_launch_small_r(void *stream, int nspec, int ntab, const ce_spec_dev *d_spec,
                                 const ce_grid_dev *d_grids, const ce_table_desc *d_tabs, const double *d_k,
                                 const double *d_pk, int max_n, double epsrel, double *d_out, int *d_status)
{
    static const double min_sep[CE_MIN_SEP_LEN] = {
        1E-6, 1E-5, 1E-4, 1E-3, 2E-3, 5E-3, 7E-3, 8E-3, 9E-3, 1E-2, 1.1E-2, 1.2E-2, 1.25E-2, 1.3E-2,
        1.35E-2, 1.5E-2, 2E-2, 2.5E-2, 3E-2, 3.5E-2, 5E-2, 7E-2, 8E-2, 9E-2, 1E-1, 1.1E-1, 1.2E-1,
        1.25E-1, 1.3E-1, 1.35E-1, 1.5E-1, 1.75E-1, 2E-1, 2.5E-1, 3E-1, 3.5E-1, 4E-1, 5E-1, 6E-1,
        7E-1, 8E-1, 9E-1};
    hipStream_t s = (hipStream_t)stream;
    hipError_t e = hipMemcpyToSymbolAsync(HIP_SYMBOL(c_min_sep), min_sep, sizeof(min_sep), 0,
                                          hipMemcpyHostToDevice, s);
    if (e == hipSuccess)
        e = hipMemcpyToSymbolAsync(HIP_SYMBOL(c_xgk), GK61K_X, sizeof(GK61K_X), 0, hipMemcpyHostToDevice, s);
    if (e == hipSuccess)
        e = hipMemcpyToSymbolAsync(HIP_SYMBOL(c_wgk), GK61K_W, sizeof(GK61K_W), 0, hipMemcpyHostToDevice, s);
    if (e == hipSuccess)
        e = hipMemcpyToSymbolAsync(HIP_SYMBOL(c_wg), GK61G_W, sizeof(GK61G_W), 0, hipMemcpyHostToDevice, s);
    if (e != hipSuccess) return (int)e;
    sr_args a;
    a.nspec = nspec; a.ntab = ntab; a.spec = d_spec; a.grids = d_grids; a.tabs = d_tabs;
    a.k = d_k; a.p = d_pk; a.epsrel = epsrel; a.out = d_out; a.status = d_status;
    return (int)(max_n <= CE_SPL_MAX ? launch_small_r<true>(a, spline_bytes(max_n), s) : launch_small_r<false>(a, 0, s));
}

extern "C" int ce_launch_divergent(void *stream, const double *d_k, const double *d_pk, int n_in, double kmin,
                                   double kmax, const double *d_sep, int nsep, const double *d_chi, int nchi,
                                   double epsrel, double *d_i40, double *d_r0, double *d_ren, int *d_status,
                                   int *d_nint)
{
    hipStream_t s = (hipStream_t)stream;
    hipError_t e = hipMemcpyToSymbolAsync(HIP_SYMBOL(c_xgk), GK61K_X, sizeof(GK61K_X), 0, hipMemcpyHostToDevice, s);
    if (e == hipSuccess)
        e = hipMemcpyToSymbolAsync(HIP_SYMBOL(c_wgk), GK61K_W, sizeof(GK61K_W), 0, hipMemcpyHostToDevice, s);
    if (e == hipSuccess)
        e = hipMemcpyToSymbolAsync(HIP_SYMBOL(c_wg), GK61G_W, sizeof(GK61G_W), 0, hipMemcpyHostToDevice, s);
    if (e != hipSuccess) return (int)e;
    div_args a;
    a.k = d_k; a.p = d_pk; a.n_in = n_in; a.kmin = kmin; a.kmax = kmax; a.epsrel = epsrel;
    a.sep = d_sep; a.nsep = nsep; a.chi = d_chi; a.nchi = nchi;
    a.i40 = d_i40; a.r0 = d_r0; a.ren = d_ren; a.status = d_status; a.nint = d_nint;
    const int units = 2 * nsep + nchi * nchi;
    if (units <= 0) return 0;
    return (int)(n_in <= CE_SPL_MAX ? launch_divergent<true>(a, units, spline_bytes(n_in), s)
                                    : launch_divergent<false>(a, units, 0, s));
}
