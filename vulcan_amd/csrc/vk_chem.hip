// Rate constants, chemistry + diffusion right-hand side, Jacobian and Ros2
// left-hand-side assembly.  One workgroup per layer for the per-layer
// kernels: the layer's y row and its reaction rates live in LDS, species
// rows are gathered from per-species CSR lists (no atomics, fixed order).
#include <algorithm>

#include "vk_internal.h"
#include "vk_device.h"

using namespace vk;

// Bounds-checked build (compiled with VK_CHECKED, libvulcan_amd_checked.so):
// every index the gather/scatter kernels read from their tables is checked
// against the length of the array it indexes; the first index out of range
// records its site in vk_check_word and the access uses index 0 instead,
// so nothing is read or written outside its array.  The normal build
// compiles the checks away.
enum VkCheckSite {
    VK_SITE_SPECIES = 1,   // species of a reaction side (rates of pairs, slot derivatives)
    VK_SITE_PAIR = 2,      // pair of a production/loss entry of a species
    VK_SITE_CHEM = 3,      // production/loss entry of a species
    VK_SITE_SLOTPAIR = 4,  // pair of a derivative slot
    VK_SITE_TERM = 5,      // Jacobian term of an entry
    VK_SITE_SLOT = 6,      // derivative slot of a Jacobian term
    VK_SITE_DENSE = 7,     // dense index of a long Jacobian entry
};
#ifdef VK_CHECKED
static __device__ int vk_check_word;
__device__ __forceinline__ int vk_ix(int i, int n, int site) {
    if ((unsigned)i < (unsigned)n) return i;
    atomicCAS(&vk_check_word, 0, site);
    return 0;
}
#define VK_IX(i, n, site) vk_ix((i), (n), (site))
#else
#define VK_IX(i, n, site) (i)
#endif

namespace {

constexpr int BLK = 256;
constexpr int RATE_LAYERS = 8;   // layers of a workgroup of k_rates, at most

// ---------------------------------------------------------------------------
// rates (op.py:145-207, 287-309; photolysis op.py:2786)
// ---------------------------------------------------------------------------

// One workgroup per LG layers: what depends on a layer alone (log T in two
// doubles, powers of T, g/RT of every species) is formed once and kept in LDS,
// and a thread keeps a pair's parameters and species for all its layers.
// T^n exp(-E/T) and the reverse constant's exp(dG/RT) take one exponential
// each, of an argument held in two doubles, instead of a pow, an exp and a
// division; arguments or results near the ends of the range (and NaN) take
// the library functions.  256 columns (36 000 layers), 93 species, 620 pairs:
// 493 us in two kernels, with g/RT written and read back, -> 255 us (bound by
// FP64 arithmetic; the 360 MB of rates take 75 us); the largest error against
// 64 bits is the same 2.4e-15.

struct LayerRate {
    double T, rT, lh, ll;              // 1/T, log T = lh + ll (NaN: no fast path)
    double M, emtau, x, rx;            // exp(-tau), CORR T and its inverse
    double logT, T2, T3, T4;
};

// g/RT = h/RT - s/R of the NASA9 polynomials (thermo/gibbs_text.txt:13-18),
// low set below 1000 K, high set at and above (chem_funs.py:2789-2792)
__device__ inline double g_layer(const LayerRate &y, const double *a20) {
    const double *a = a20 + (y.T < 1000.0 ? 0 : 10);
    const double h = -a[0] / y.T2 + a[1] * y.logT / y.T + a[2] + a[3] * y.T / 2. + a[4] * y.T2 / 3. + a[5] * y.T3 / 4. +
                     a[6] * y.T4 / 5. + a[8] / y.T;
    const double r = -a[0] / y.T2 / 2. - a[1] / y.T + a[2] * y.logT + a[3] * y.T + a[4] * y.T2 / 2. + a[5] * y.T3 / 3. +
                     a[6] * y.T4 / 4. + a[9];
    return h - r;
}

constexpr double LN2_HI = 0x1.62e42fefa39efp-1, LN2_LO = 0x1.abc9e3b39803fp-56;   // ln 2 in two doubles

// log x for normal x > 0 as h + l, from log m = 2 atanh((m - 1) / (m + 1)) with
// the series in two-double arithmetic (|m - 1| / (m + 1) < 0.172: 16 terms
// leave 1e-25); once per layer
__device__ inline void log2d(double x, double &h, double &l) {
    int e;
    double m = frexp(x, &e);
    if (m < 0.70710678118654752) {
        m *= 2.0;
        e--;
    }
    const double num = m - 1.0, dh = m + 1.0, dl = (1.0 - dh) + m;
    const double sh = num / dh, sl = (fma(-sh, dh, num) - sh * dl) / dh;
    const double zh = sh * sh, zl = fma(sh, sh, -zh) + 2.0 * sh * sl;
    double ph = 0.0, pl = 0.0;
    for (int j = 15; j >= 0; j--) {
        const double d = 2 * j + 1, ch = 1.0 / d, cl = fma(-ch, d, 1.0) / d;
        const double t = ph * zh, tl = fma(ph, zh, -t) + (ph * zl + pl * zh);
        ph = ch + t;
        pl = ((ch - ph) + t) + (tl + cl);
    }
    const double uh = 2.0 * sh * ph, ul = fma(2.0 * sh, ph, -uh) + 2.0 * (sh * pl + sl * ph);
    const double eh = e * LN2_HI, el = fma((double)e, LN2_HI, -eh) + e * LN2_LO;
    const double t = eh + uh, bb = t - eh, tl = ((eh - (t - bb)) + (uh - bb)) + (el + ul);
    h = t + tl;
    l = (t - h) + tl;
}

// c exp(t + lo) for |t| < 700, |lo| << 1: t = k ln 2 + r, the exponential's
// series to r^13 / 13! (|r| < 0.35: 4e-18 left out)
__device__ inline double mul_exp(double c, double t, double lo) {
    const double k = rint(t * 1.4426950408889634);
    const double r = fma(-k, LN2_HI, t) + fma(-k, LN2_LO, lo);
    double q = 1. / 6227020800.;
    q = fma(q, r, 1. / 479001600.);
    q = fma(q, r, 1. / 39916800.);
    q = fma(q, r, 1. / 3628800.);
    q = fma(q, r, 1. / 362880.);
    q = fma(q, r, 1. / 40320.);
    q = fma(q, r, 1. / 5040.);
    q = fma(q, r, 1. / 720.);
    q = fma(q, r, 1. / 120.);
    q = fma(q, r, 1. / 24.);
    q = fma(q, r, 1. / 6.);
    q = fma(q, r, 0.5);
    const double e = fma(q, r * r, r);
    return ldexp(fma(c, e, c), (int)k);
}

constexpr double EXP_FAST = 650.0;                    // |exponents| of the fast paths
__device__ inline bool rate_normal(double k) { return fabs(k) > 1e-280 && fabs(k) < 1e280; }

// A T^n exp(-E/T)
__device__ inline double arrh(double A, double n, double E, const LayerRate &y) {
    const double q = E * y.rT, ql = fma(-q, y.T, E) * y.rT;              // E/T = q + ql
    const double h = n * y.lh, hl = fma(n, y.lh, -h) + n * y.ll;         // n log T = h + hl
    const double t = h - q, bb = t - h, tl = (h - (t - bb)) - (q + bb);  // h - q = t + tl
    const bool in = fabs(h) < EXP_FAST && fabs(q) < EXP_FAST && fabs(t) < EXP_FAST;   // false for NaN
    const double k = in ? mul_exp(A, t, tl + (hl - ql)) : 0.0;
    if (rate_normal(k)) return k;
    return A * pow(y.T, n) * exp(-E / y.T);
}

__global__ void __launch_bounds__(BLK, 4) k_rates(int L, int LG, int npairs, int ni, const int *__restrict__ kind,
                                               const double *__restrict__ par, const int *__restrict__ rev,
                                               const int *__restrict__ reac, const int *__restrict__ prod,
                                               const double *__restrict__ nasa9, const double *__restrict__ Tco,
                                               const double *__restrict__ M, const double *__restrict__ tau,
                                               double *__restrict__ k) {
    __shared__ LayerRate lay[RATE_LAYERS];
    __shared__ double gl[RATE_LAYERS][VK_NI_MAX + 1];    // the last entry: no species, 0
    const int l0 = blockIdx.x * LG, nl = min(LG, L - l0);
    if ((int)threadIdx.x < nl) {
        LayerRate y;
        const int l = l0 + threadIdx.x;
        y.T = Tco[l];
        y.rT = 1.0 / y.T;
        y.lh = y.ll = nan("");
        if (y.T > 1e-300 && y.T < 1e300) log2d(y.T, y.lh, y.ll);
        y.M = M[l];
        y.emtau = exp(-(tau ? tau[l] : 0.0));
        y.x = CORR * y.T;
        y.rx = 1.0 / y.x;
        y.logT = log(y.T);
        y.T2 = y.T * y.T;
        y.T3 = pow(y.T, 3.0);
        y.T4 = pow(y.T, 4.0);
        lay[threadIdx.x] = y;
        gl[threadIdx.x][ni] = 0.0;
    }
    __syncthreads();
    for (int q = threadIdx.x; q < nl * ni; q += BLK) {
        const int a = q / ni, s = q - a * ni;
        gl[a][s] = g_layer(lay[a], nasa9 + 20 * s);
    }
    __syncthreads();
    for (int p = blockIdx.y * BLK + threadIdx.x; p < npairs; p += BLK * gridDim.y) {
        double pa[8];
#pragma unroll
        for (int q = 0; q < 8; q++) pa[q] = par[8 * p + q];
        const int kd = kind[p], rv = rev[p];
        const int narrh = kd == VK_KIND_ARRH || kd == VK_KIND_K0 ? 1 : (kd == VK_KIND_LIND || kd == VK_KIND_TROE ? 2 : 0);
        int sr[4], sp[4], dn = 0;
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const int r = reac[4 * p + q], o = prod[4 * p + q];
            sr[q] = r >= 0 ? VK_IX(r, ni, VK_SITE_SPECIES) : ni;
            sp[q] = o >= 0 ? VK_IX(o, ni, VK_SITE_SPECIES) : ni;
            dn += (r >= 0) - (o >= 0);
        }
        for (int a = 0; a < nl; a++) {
            const LayerRate &y = lay[a];
            const double T = y.T, m = y.M;
            // the one or two Arrhenius expressions of the pair, in a loop: one
            // copy of the code
            double k0 = 0.0, kinf = 0.0;
#pragma unroll 1
            for (int h = 0; h < narrh; h++) {
                const double v = arrh(h ? pa[3] : pa[0], h ? pa[4] : pa[1], h ? pa[5] : pa[2], y);
                k0 = h ? k0 : v;
                kinf = h ? v : kinf;
            }
            double kf;
            switch (kd) {
            case VK_KIND_ARRH:
            case VK_KIND_K0:
                kf = k0;
                break;
            case VK_KIND_LIND:
                kf = k0 / (1 + k0 * m / kinf);
                break;
            case VK_KIND_CH3OH:
                k0 = 1.932E3 * pow(T, -9.88) * exp(-7544. / T) + 5.109E-11 * pow(T, -6.25) * exp(-1433. / T);
                kinf = 1.031E-10 * pow(T, -0.018) * exp(16.74 / T);
                [[fallthrough]];
            case VK_KIND_TROE: {
                const double Fc = kd == VK_KIND_TROE
                                      ? pa[6]
                                      : 0.1855 * exp(-T / 155.8) + 0.8145 * exp(-T / 1675.) + exp(-4531. / T);
                double nn = 0.75 - 1.27 * log(Fc);
                double q = log(k0 * m / kinf) / nn;
                double ff = exp(log(Fc) / (1. + q * q));
                kf = k0 / (1 + k0 * m / kinf) * ff;
                break;
            }
            case VK_KIND_PHOTO:
                kf = pa[7] * y.emtau;
                break;
            default:
                kf = 0.0;
            }
            double kr = 0.0;
            if (rv) {
                // K = exp(-(-g_r1 - g_r2 + g_p1 + g_p2)) * (corr T)^(n_r - n_p)  (make_chem_funs.py:568-580)
                double acc = 0.0;
#pragma unroll
                for (int q = 0; q < 4; q++) acc -= gl[a][sr[q]];
#pragma unroll
                for (int q = 0; q < 4; q++) acc += gl[a][sp[q]];
                if (fabs(acc) < EXP_FAST && dn >= -1 && dn <= 1)
                    kr = mul_exp(kf, acc, 0.0) * (dn == 0 ? 1.0 : (dn == 1 ? y.rx : y.x));
                if (!rate_normal(kr)) {
                    double K = exp(-acc);
                    if (dn != 0) {
                        double f;
                        if (dn == 1) f = y.x;
                        else if (dn == -1) f = 1.0 / y.x;
                        else if (dn == 2) f = y.x * y.x;
                        else f = pow(y.x, (double)dn);
                        K = K * f;
                    }
                    kr = kf / K;
                }
            }
            double *out = k + 2 * ((size_t)(l0 + a) * npairs + p);
            out[0] = kf;
            out[1] = kr;
        }
    }
}

// ---------------------------------------------------------------------------
// per-layer helpers
// ---------------------------------------------------------------------------

struct LayerCtx {
    int l, c, off, nz, j;
};

__device__ inline LayerCtx layer_ctx(const int *off, const int *layer_col, int l) {
    LayerCtx x;
    x.l = l;
    x.c = layer_col[l];
    x.off = off[x.c];
    x.nz = off[x.c + 1] - x.off;
    x.j = l - x.off;
    return x;
}

// v_p = k_f * prod(reac) - k_r * prod(prod), left to right (make_chem_funs.py:293-315);
// the four terms of a side are one 16-byte load
__device__ inline double side_product(int4 t4, double kcol, const double *yl, double m, int ni) {
    const int t[4] = {t4.x, t4.y, t4.z, t4.w};
    double a = kcol;
#pragma unroll
    for (int q = 0; q < 4; q++) {
        if (t[q] == -2) continue;
        a = a * (t[q] == -1 ? m : yl[VK_IX(t[q], ni, VK_SITE_SPECIES)]);
    }
    return a;
}

__device__ inline double pair_rate(const int4 *reac, const int4 *prod, const double *kl, const double *yl,
                                   double m, int p, int ni) {
    const double a = side_product(reac[p], kl[2 * p], yl, m, ni);
    const double b = side_product(prod[p], kl[2 * p + 1], yl, m, ni);
    return a - b;
}

// d/dy_sp of kcol * prod(terms)
__device__ inline double dside(int4 t4, double kcol, const double *yl, double m, int sp, bool &any, int ni) {
    const int t[4] = {t4.x, t4.y, t4.z, t4.w};
    double tot = 0.0;
    any = false;
#pragma unroll
    for (int q = 0; q < 4; q++) {
        if (t[q] != sp) continue;
        double acc = kcol;
#pragma unroll
        for (int q2 = 0; q2 < 4; q2++) {
            if (q2 == q || t[q2] == -2) continue;
            acc = acc * (t[q2] == -1 ? m : yl[VK_IX(t[q2], ni, VK_SITE_SPECIES)]);
        }
        tot = any ? tot + acc : acc;
        any = true;
    }
    return tot;
}

// ysum[l] = sum_i y[l][i] in numpy's pairwise order, one thread per layer
__global__ void k_ysum(int L, int ni, const double *__restrict__ y, double *__restrict__ ysum) {
    const int l = blockIdx.x * blockDim.x + threadIdx.x;
    if (l < L) ysum[l] = pw_sum(y + (size_t)l * ni, ni);
}

// the three layer totals a layer's diffusion terms use (0 outside the column)
__device__ inline void ysum_around(const double *ysum, const LayerCtx &x, double &ym, double &y0, double &yp) {
    const double *ys = ysum + x.off;
    ym = x.j > 0 ? ys[x.j - 1] : 0.0;
    y0 = ys[x.j];
    yp = x.j < x.nz - 1 ? ys[x.j + 1] : 0.0;
}

// ---------------------------------------------------------------------------
// chemdf + diffdf (+ stage-2 term), one workgroup per layer
// mode bit 0: include chemistry, bit 1: include diffusion
// ---------------------------------------------------------------------------

__global__ void __launch_bounds__(BLK) k_rhs(
    int ni, int npairs, int nchem, const int *__restrict__ off, const int *__restrict__ layer_col,
    const int *__restrict__ reac, const int *__restrict__ prod, const int *__restrict__ chem_ptr,
    const int2 *__restrict__ chem_ent, const double *__restrict__ ms,
    const double *__restrict__ alpha, vk_atm atm, const double *__restrict__ y, const double *__restrict__ k,
    const double *__restrict__ M, int mode, int mol, const double *__restrict__ k1,
    const double *__restrict__ dtc, const double *__restrict__ ysum, const vk_colstate *__restrict__ st,
    double *__restrict__ out) {
    extern __shared__ double smem[];
    double *yl = smem;              // ni
    double *v = smem + VK_NI_MAX;   // npairs
    const int l = blockIdx.x;
    LayerCtx x = layer_ctx(off, layer_col, l);
    if (st && st[x.c].done) return;
    const double *yrow = y + (size_t)l * ni;
    for (int i = threadIdx.x; i < ni; i += blockDim.x) yl[i] = yrow[i];
    double ysm = 0.0, ys0 = 0.0, ysp = 0.0;
    if (mode & 2) ysum_around(ysum, x, ysm, ys0, ysp);
    __syncthreads();
    if (mode & 1) {
        const double *kl = k + (size_t)l * 2 * npairs;
        double m = M[l];
        for (int p = threadIdx.x; p < npairs; p += blockDim.x)
            v[p] = pair_rate((const int4 *)reac, (const int4 *)prod, kl, yl, m, p, ni);
        __syncthreads();
    }
    ColAtm ca = col_atm(atm, x.c, x.off, x.nz, ni);
    double c2 = 0.0;
    if (k1) c2 = 2. / (R_ROS * dtc[x.c]);
    for (int i = threadIdx.x; i < ni; i += blockDim.x) {
        double chem = 0.0;
        if (mode & 1) {
            const int lo = chem_ptr[i], hi = chem_ptr[i + 1];
            if (lo < hi) {
                int2 t = chem_ent[VK_IX(lo, nchem, VK_SITE_CHEM)];   // (pair, sign)
                chem = t.y * v[VK_IX(t.x, npairs, VK_SITE_PAIR)];
                // the terms in order, eight entries loaded ahead of their sums
                int e = lo + 1;
                for (; e + 8 <= hi; e += 8) {
                    int2 tt[8];
#pragma unroll
                    for (int u = 0; u < 8; u++) tt[u] = chem_ent[VK_IX(e + u, nchem, VK_SITE_CHEM)];
#pragma unroll
                    for (int u = 0; u < 8; u++) chem = chem + tt[u].y * v[VK_IX(tt[u].x, npairs, VK_SITE_PAIR)];
                }
                for (; e < hi; e++) {
                    t = chem_ent[VK_IX(e, nchem, VK_SITE_CHEM)];
                    chem = chem + t.y * v[VK_IX(t.x, npairs, VK_SITE_PAIR)];
                }
            }
        }
        double val = chem;
        if (mode & 2) {
            double ym = x.j > 0 ? y[(size_t)(l - 1) * ni + i] : 0.0;
            double yp = x.j < x.nz - 1 ? y[(size_t)(l + 1) * ni + i] : 0.0;
            double d = diff_value(ca, x.j, i, ysm, ys0, ysp, ym, yl[i], yp, ms[i], alpha[i], mol != 0);
            val = (mode & 1) ? chem + d : d;
        }
        if (k1) val = val - c2 * k1[(size_t)l * ni + i];
        out[(size_t)l * ni + i] = val;
    }
}

// ---------------------------------------------------------------------------
// Jacobian blocks (mode 0: J = d chemdf/dy) or Ros2 lhs blocks (mode 1:
// D = c0 I - J - J_diff, Lsub, Usup), one workgroup per layer
// ---------------------------------------------------------------------------

// The diagonal of a layer's lhs block after c0 - J: the diffusion terms in
// the reference's order.  xmode 1: the escape term first (top layer, _vm
// operators, op.py:2101-2107); xmode 2: the deposition velocity last (bottom
// layer, op.py:2029).
__device__ __forceinline__ double lhs_diag(double val, int i, int mol, const double *dg0, const double *dg1,
                                           const double *dgx, int xmode) {
    if (xmode == 1) val = val - dgx[i];
    val = val - dg0[i];
    if (mol) val = val - dg1[i];
    if (xmode == 2) val = val - dgx[i];
    return val;
}

// one entry of the lhs (mode 1) or of the Jacobian (mode 0): its terms in order
__device__ __forceinline__ void jac_entry(int q, const int4 *__restrict__ jac_ent, const int *__restrict__ jac_tp,
                                          const double *dv, int ni, int njac, int nslot, int mode, int mol, double c0,
                                          const double *dg0, const double *dg1, const double *dgx, int xmode,
                                          double *__restrict__ Dl) {
    const int4 en = jac_ent[q];           // (dense index, first term, end of terms, row)
    double J = 0.0;
    if (en.z > en.y) {
        const int t = jac_tp[VK_IX(en.y, njac, VK_SITE_TERM)];
        J = vk_jac_coef(t) * dv[VK_IX(vk_jac_slot(t), nslot, VK_SITE_SLOT)];
        // terms in order; four loads in flight per round
        for (int u = en.y + 1; u < en.z; u += 4) {
            const int t0 = jac_tp[VK_IX(u, njac, VK_SITE_TERM)];
            const int t1 = u + 1 < en.z ? jac_tp[VK_IX(u + 1, njac, VK_SITE_TERM)] : t0;
            const int t2 = u + 2 < en.z ? jac_tp[VK_IX(u + 2, njac, VK_SITE_TERM)] : t0;
            const int t3 = u + 3 < en.z ? jac_tp[VK_IX(u + 3, njac, VK_SITE_TERM)] : t0;
            J = J + vk_jac_coef(t0) * dv[VK_IX(vk_jac_slot(t0), nslot, VK_SITE_SLOT)];
            if (u + 1 < en.z) J = J + vk_jac_coef(t1) * dv[VK_IX(vk_jac_slot(t1), nslot, VK_SITE_SLOT)];
            if (u + 2 < en.z) J = J + vk_jac_coef(t2) * dv[VK_IX(vk_jac_slot(t2), nslot, VK_SITE_SLOT)];
            if (u + 3 < en.z) J = J + vk_jac_coef(t3) * dv[VK_IX(vk_jac_slot(t3), nslot, VK_SITE_SLOT)];
        }
    }
    const int ex = VK_IX(en.x, ni * ni, VK_SITE_DENSE);
    if (mode == 0) {
        Dl[ex] = J;
        return;
    }
    const int i = en.w;
    double val = -J;
    if (ex == i * ni + i) val = lhs_diag(c0 + val, i, mol, dg0, dg1, dgx, xmode);
    Dl[ex] = val;
}

__global__ void __launch_bounds__(BLK) k_jac_lhs(
    int ni, int npairs, int nslot, int nent, int njac, const int *__restrict__ off, const int *__restrict__ layer_col,
    const int *__restrict__ reac, const int *__restrict__ prod, const int *__restrict__ slot_pair,
    const int *__restrict__ slot_sp, const int4 *__restrict__ jac_ent, const int *__restrict__ jac_emap, int nheavy,
    const int *__restrict__ jac_tp,
    const double *__restrict__ ms, const double *__restrict__ alpha, vk_atm atm, const double *__restrict__ y,
    const double *__restrict__ k, const double *__restrict__ M, int mode, int mol, const double *__restrict__ dtc,
    const double *__restrict__ ysum, const vk_colstate *__restrict__ st, double *__restrict__ D,
    double *__restrict__ Lsub, double *__restrict__ Usup, int write_zeros) {
    extern __shared__ double smem[];
    double *yl = smem;                       // ni
    double *dg0 = smem + VK_NI_MAX;          // diffusion terms of the diagonal, per species
    double *dg1 = smem + 2 * VK_NI_MAX;
    double *dgx = smem + 3 * VK_NI_MAX;      // escape (top) or deposition (bottom) term
    double *dv = smem + 4 * VK_NI_MAX;       // nslot
    const int l = blockIdx.x;
    LayerCtx x = layer_ctx(off, layer_col, l);
    if (st && st[x.c].done) return;
    const double *yrow = y + (size_t)l * ni;
    for (int i = threadIdx.x; i < ni; i += blockDim.x) yl[i] = yrow[i];
    __syncthreads();   // the slot derivatives read yl
    const int nn = ni * ni;
    double *Dl = D + (size_t)l * nn;
    const double *kl = k + (size_t)l * 2 * npairs;
    const double m = M[l];
    // slot derivatives: JS slots per thread per round, every load of a round
    // (slot -> pair -> the pair's sides and rates, three loads deep) issued
    // before its arithmetic
    constexpr int JS = 4;
    for (int s0 = threadIdx.x; s0 < nslot; s0 += JS * blockDim.x) {
        int p[JS], sp[JS];
#pragma unroll
        for (int u = 0; u < JS; u++) {
            const int s = s0 + u * blockDim.x;
            p[u] = s < nslot ? VK_IX(slot_pair[s], npairs, VK_SITE_SLOTPAIR) : 0;
            sp[u] = s < nslot ? slot_sp[s] : 0;
        }
        int4 rt[JS], pt[JS];
        double kf[JS], kb[JS];
#pragma unroll
        for (int u = 0; u < JS; u++) {
            rt[u] = ((const int4 *)reac)[p[u]];
            pt[u] = ((const int4 *)prod)[p[u]];
            kf[u] = kl[2 * p[u]];
            kb[u] = kl[2 * p[u] + 1];
        }
#pragma unroll
        for (int u = 0; u < JS; u++) {
            const int s = s0 + u * blockDim.x;
            if (s < nslot) {
                bool a1, a2;
                const double dr = dside(rt[u], kf[u], yl, m, sp[u], a1, ni);
                const double dp = dside(pt[u], kb[u], yl, m, sp[u], a2, ni);
                dv[s] = (a1 ? dr : 0.0) - (a2 ? dp : 0.0);
            }
        }
    }
    double c0 = 0.0;
    int xmode = 0;
    if (mode == 1) {
        // diffusion part of the lhs (op.py:2012-2040): once per species
        c0 = 1. / (R_ROS * dtc[x.c]);
        double ysm, ys0, ysp;
        ysum_around(ysum, x, ysm, ys0, ysp);
        ColAtm ca = col_atm(atm, x.c, x.off, x.nz, ni);
        if (x.j == 0 && ca.use_bot) xmode = 2;
        else if (x.j == x.nz - 1 && ca.vm && mol && atm.top_flux && esc_any(atm)) xmode = 1;
        for (int i = threadIdx.x; i < ni; i += blockDim.x) {
            LhsDiff r = lhs_diff(ca, x.j, i, ysm, ys0, ysp, ms[i], alpha[i], mol != 0);
            dg0[i] = r.d0;
            dg1[i] = r.d1;
            if (xmode == 2) {
                dgx[i] = -1. * ca.bot_vdep[i] / ca.dzi[0];
            } else if (xmode == 1) {
                // diff_lim = top_flux / y for escaping species with y > 0 (no 1/dzi, as there)
                double e = 0.0;
                if (((atm.esc[i >> 5] >> (i & 31)) & 1u) && yrow[i] > 0)
                    e = 0.0 + atm.top_flux[(size_t)x.c * ni + i] / yrow[i];
                dgx[i] = e;
            }
            double u = 0.0, lo = 0.0;
            if (r.has_u) { u = 0.0 - r.u0; if (r.has_mol) u = u - r.u1; }
            if (r.has_l) { lo = 0.0 - r.l0; if (r.has_mol) lo = lo - r.l1; }
            if (blockIdx.y == 0) {
                Usup[(size_t)l * ni + i] = u;
                Lsub[(size_t)l * ni + i] = lo;
            }
        }
    }
    __syncthreads();
    // Every dense entry is written once (the structural zeros only with
    // write_zeros: the integrator clears its blocks once and skips them).
    // Entries with at most JAC_LIGHT
    // terms (and the structural zeros) in one coalesced pass over the dense
    // index; the few long term lists (jac_ent[0, nheavy): the list is sorted
    // by term count) by their own threads alongside.  With few layers the
    // entries of a layer are split over the grid's y dimension (each
    // workgroup forms the layer's shared terms itself).
    const int e0 = threadIdx.x + blockIdx.y * blockDim.x, es = blockDim.x * gridDim.y;
    for (int q = e0; q < nheavy; q += es)
        jac_entry(q, jac_ent, jac_tp, dv, ni, njac, nslot, mode, mol, c0, dg0, dg1, dgx, xmode, Dl);
#pragma unroll 4
    for (int e = e0; e < nn; e += es) {
        // (first term << 4 | term count), -1: structural zero, -2: long term list
        const int code = jac_emap[e];
        if (code == -2 || (code == -1 && !write_zeros)) continue;
        double val = 0.0;
        if (code >= 0) {
            const int u0 = code >> 4, nt = code & 15;
            double J = 0.0;
            if (nt > 0) {
                // only the entry's own terms are loaded (all issued before the sums)
                int t[VK_JAC_LIGHT];
#pragma unroll
                for (int m = 0; m < VK_JAC_LIGHT; m++) t[m] = m < nt ? jac_tp[VK_IX(u0 + m, njac, VK_SITE_TERM)] : 0;
                J = vk_jac_coef(t[0]) * dv[VK_IX(vk_jac_slot(t[0]), nslot, VK_SITE_SLOT)];
#pragma unroll
                for (int m = 1; m < VK_JAC_LIGHT; m++)
                    if (m < nt) J = J + vk_jac_coef(t[m]) * dv[VK_IX(vk_jac_slot(t[m]), nslot, VK_SITE_SLOT)];
            }
            if (mode == 0) {
                val = J;
            } else {
                const int i = e / ni;
                val = -J;
                if (e == i * ni + i) val = lhs_diag(c0 + val, i, mol, dg0, dg1, dgx, xmode);
            }
        }
        Dl[e] = val;
    }
}

}  // namespace

// ---------------------------------------------------------------------------
// host entry points
// ---------------------------------------------------------------------------

static inline hipStream_t S(void *s) { return (hipStream_t)s; }

static size_t rhs_smem(const vk_plan *p) { return sizeof(double) * (VK_NI_MAX + (size_t)p->npairs); }
static size_t jac_smem(const vk_plan *p) { return sizeof(double) * (4 * VK_NI_MAX + (size_t)p->nslot); }

extern "C" int vk_rates(const vk_plan *plan, const vk_columns *cols, const vk_atm *atm, double *d_k, void *stream) {
    if (!plan || !cols || !atm || !d_k) return VK_EINVAL;
    const int L = cols->L, cu = vk_device_cus();
    // layers per workgroup: the most (their pairs' parameters are read once)
    // that still leave eight workgroups per CU; below that one layer each, and
    // its pairs over several workgroups
    int LG = RATE_LAYERS;
    while (LG > 1 && L < 8 * cu * LG) LG /= 2;
    const int split = LG > 1 ? 1 : (plan->npairs + BLK - 1) / BLK;
    hipLaunchKernelGGL(k_rates, dim3((L + LG - 1) / LG, split), dim3(BLK), 0, S(stream), L, LG, plan->npairs, plan->ni,
                       plan->kind, plan->par, plan->rev, plan->reac, plan->prod, plan->nasa9, atm->Tco, atm->M,
                       atm->tau, d_k);
    VK_CHECK(hipGetLastError());
    return 0;
}

static int launch_ysum(const vk_columns *cols, int ni, const double *y, double *ysum, hipStream_t s) {
    hipLaunchKernelGGL(k_ysum, dim3((cols->L + 127) / 128), dim3(128), 0, s, cols->L, ni, y, ysum);
    VK_CHECK(hipGetLastError());
    return 0;
}

// ysum: scratch of L doubles (needed when the diffusion terms are evaluated)
int vk_launch_rhs(const vk_plan *plan, const vk_columns *cols, const vk_atm *atm, const double *y,
                  const double *k, int mode, int mol, const double *k1, const double *dtc,
                  const vk_colstate *st, double *ysum, double *out, hipStream_t s) {
    vk_atm a = *atm;
    if (mode & 2) {
        if (!ysum) return VK_EINVAL;
        int r = launch_ysum(cols, plan->ni, y, ysum, s);
        if (r) return r;
    }
    hipLaunchKernelGGL(k_rhs, dim3(cols->L), dim3(BLK), rhs_smem(plan), s, plan->ni, plan->npairs, plan->nchem,
                       cols->d_off,
                       cols->d_layer_col, plan->reac, plan->prod, plan->chem_ptr, plan->chem_ent, plan->ms,
                       plan->alpha, a, y, k, atm->M, mode, mol, k1, dtc, ysum, st, out);
    VK_CHECK(hipGetLastError());
    return 0;
}

// ysum_ready: the caller's earlier launch on s has left the layer sums of y in ysum
int vk_launch_jac_lhs(const vk_plan *plan, const vk_columns *cols, const vk_atm *atm, const double *y,
                      const double *k, const double *M, int mode, int mol, const double *dtc,
                      const vk_colstate *st, double *ysum, double *D, double *Lsub, double *Usup, hipStream_t s,
                      bool ysum_ready = false, bool write_zeros = true) {
    vk_atm a{};
    if (atm) a = *atm;
    if (mode == 1) {
        if (!ysum) return VK_EINVAL;
        if (!ysum_ready) {
            int r = launch_ysum(cols, plan->ni, y, ysum, s);
            if (r) return r;
        }
    }
    // fewer layers than twice the CUs: split each layer's entries over up to 4 workgroups
    static const int ncu = [] {
        int dev = 0, n = 0;
        if (hipGetDevice(&dev) != hipSuccess ||
            hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
            return 0;
        return n;
    }();
    const int gy = ncu > 0 ? std::max(1, std::min(4, 2 * ncu / std::max(cols->L, 1))) : 1;
    hipLaunchKernelGGL(k_jac_lhs, dim3(cols->L, gy), dim3(BLK), jac_smem(plan), s, plan->ni, plan->npairs, plan->nslot,
                       plan->njent, plan->njac, cols->d_off, cols->d_layer_col, plan->reac, plan->prod, plan->slot_pair,
                       plan->slot_sp, plan->jac_ent, plan->jac_emap, plan->njheavy, plan->jac_tp, plan->ms, plan->alpha, a, y, k, M, mode, mol,
                       dtc, ysum, st, D, Lsub, Usup, (int)write_zeros);
    VK_CHECK(hipGetLastError());
    return 0;
}

// temporary layer totals for the one-shot entry points
struct YsumTmp {
    double *p = nullptr;
    hipStream_t s;
    explicit YsumTmp(hipStream_t st) : s(st) {}
    int alloc(int L) { return hipMallocAsync((void **)&p, sizeof(double) * (size_t)L, s) == hipSuccess ? 0 : VK_ENOMEM; }
    ~YsumTmp() { if (p) (void)hipFreeAsync(p, s); }
};

extern "C" int vk_chemdf(const vk_plan *plan, const vk_columns *cols, const double *d_y, const double *d_M,
                         const double *d_k, double *d_dydt, void *stream) {
    if (!plan || !cols || !d_y || !d_M || !d_k || !d_dydt) return VK_EINVAL;
    vk_atm a{};
    a.M = d_M;
    return vk_launch_rhs(plan, cols, &a, d_y, d_k, 1, 0, nullptr, nullptr, nullptr, nullptr, d_dydt, S(stream));
}

extern "C" int vk_diffdf(const vk_plan *plan, const vk_columns *cols, const vk_atm *atm, const double *d_y,
                         int use_moldiff, double *d_out, void *stream) {
    if (!plan || !cols || !atm || !d_y || !d_out) return VK_EINVAL;
    YsumTmp ys(S(stream));
    if (ys.alloc(cols->L)) return VK_ENOMEM;
    return vk_launch_rhs(plan, cols, atm, d_y, nullptr, 2, use_moldiff, nullptr, nullptr, nullptr, ys.p, d_out,
                         S(stream));
}

extern "C" int vk_rhs(const vk_plan *plan, const vk_columns *cols, const vk_atm *atm, const double *d_y,
                      const double *d_k, int use_moldiff, const double *d_k1, const double *d_dt, double *d_out,
                      void *stream) {
    if (!plan || !cols || !atm || !d_y || !d_k || !d_out || (d_k1 && !d_dt)) return VK_EINVAL;
    YsumTmp ys(S(stream));
    if (ys.alloc(cols->L)) return VK_ENOMEM;
    return vk_launch_rhs(plan, cols, atm, d_y, d_k, 3, use_moldiff, d_k1, d_dt, nullptr, ys.p, d_out, S(stream));
}

extern "C" int vk_jac(const vk_plan *plan, const vk_columns *cols, const double *d_y, const double *d_M,
                      const double *d_k, double *d_J, void *stream) {
    if (!plan || !cols || !d_y || !d_M || !d_k || !d_J) return VK_EINVAL;
    return vk_launch_jac_lhs(plan, cols, nullptr, d_y, d_k, d_M, 0, 0, nullptr, nullptr, nullptr, d_J, nullptr, nullptr,
                             S(stream));
}

extern "C" int vk_lhs(const vk_plan *plan, const vk_columns *cols, const vk_atm *atm, const double *d_y,
                      const double *d_k, int use_moldiff, const double *d_dt, double *d_D, double *d_Lsub,
                      double *d_Usup, void *stream) {
    if (!plan || !cols || !atm || !d_y || !d_k || !d_dt || !d_D || !d_Lsub || !d_Usup) return VK_EINVAL;
    YsumTmp ys(S(stream));
    if (ys.alloc(cols->L)) return VK_ENOMEM;
    return vk_launch_jac_lhs(plan, cols, atm, d_y, d_k, atm->M, 1, use_moldiff, d_dt, nullptr, ys.p, d_D, d_Lsub, d_Usup,
                             S(stream));
}

extern "C" int vk_debug_checks(int *site_out, int reset) {
    if (!site_out) return VK_EINVAL;
#ifdef VK_CHECKED
    int v = 0;
    VK_CHECK(hipMemcpyFromSymbol(&v, HIP_SYMBOL(vk_check_word), sizeof(int)));
    if (reset) {
        const int z = 0;
        VK_CHECK(hipMemcpyToSymbol(HIP_SYMBOL(vk_check_word), &z, sizeof(int)));
    }
    *site_out = v;
    return 0;
#else
    (void)reset;
    return VK_ENOTCHECKED;
#endif
}
