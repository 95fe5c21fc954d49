// Rate constants, chemistry + diffusion right-hand side, Jacobian and Ros2
// left-hand-side assembly.  One workgroup per layer or few layers for the
// per-layer kernels: a layer's y row and its reaction rates live in LDS, species
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
// 440 us in two kernels, with g/RT written and read back, -> 230 us (bound by
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
// series to r^13 / 13! (|r| < 0.35: 4e-18 left out).  The power of two comes
// first: a factor below 2e-308 would round to its own coarse grid in the sum.
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
    const double e = fma(q, r * r, r), s = ldexp(c, (int)k);
    return fma(s, e, s);
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

// d/dy_sp of kcol * prod(terms), yl[LG s] the amount of species s
template <int LG>
__device__ inline double dside(int4 t4, double kcol, const double *yl, double m, int sp, int ni) {
    const int t[4] = {t4.x, t4.y, t4.z, t4.w};
    double tot = 0.0;
    bool any = false;
#pragma unroll
    for (int q = 0; q < 4; q++) {
        if (t[q] != sp) continue;
        double acc = kcol;
#pragma unroll
        for (int q2 = 0; q2 < 4; q2++) {
            if (q2 == q || t[q2] == -2) continue;
            acc = acc * (t[q2] == -1 ? m : yl[LG * VK_IX(t[q2], ni, VK_SITE_SPECIES)]);
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
// chemdf + diffdf (+ stage-2 term), one workgroup per LG layers
// mode bit 0: include chemistry, bit 1: include diffusion
//
// Bound by the table reads: a pair is eight bytes (its amounts' indices), the
// species' terms lie term by term over the species, so that the lanes of a
// wave read neighbouring ones, and with two layers a workgroup reads a pair
// once for both.  36 000 layers of 93 species, 620 pairs: 320 -> 263 us; 150
// layers: 13.5 -> 12.4 us.
// ---------------------------------------------------------------------------

template <int LG>
__global__ void __launch_bounds__(BLK) k_rhs(
    int L, int ni, int npairs, int nchem, const int *__restrict__ off, const int *__restrict__ layer_col,
    const uint2 *__restrict__ pair_tab, const int *__restrict__ chem_ptr, const int2 *__restrict__ chem_ent,
    const double *__restrict__ ms, const double *__restrict__ alpha, vk_atm atm, const double *__restrict__ y,
    const double *__restrict__ k, const double *__restrict__ M, int mode, int mol, const double *__restrict__ k1,
    const double *__restrict__ dtc, const double *__restrict__ ysum, const vk_colstate *__restrict__ st,
    double *__restrict__ out) {
    extern __shared__ __align__(16) double smem[];
    double *v = smem;                  // npairs x LG: rates of the pairs
    double *yl = smem + LG * npairs;   // (ni + 2) x LG: amounts, then M and one
    const int l0 = blockIdx.x * LG;
    LayerCtx xs[LG];
    bool on[LG], any = false;
#pragma unroll
    for (int a = 0; a < LG; a++) {
        xs[a] = layer_ctx(off, layer_col, min(l0 + a, L - 1));
        on[a] = l0 + a < L && !(st && st[xs[a].c].done);
        any = any || on[a];
    }
    if (!any) return;
    for (int q = threadIdx.x; q < ni + 2; q += BLK)
#pragma unroll
        for (int a = 0; a < LG; a++)
            yl[LG * q + a] = q < ni ? y[(size_t)xs[a].l * ni + q] : (q > ni ? 1.0 : (mode & 1 ? M[xs[a].l] : 0.0));
    __syncthreads();
    if (mode & 1) {
        // v_p = k_f * prod(reac) - k_r * prod(prod), left to right (make_chem_funs.py:293-315)
        for (int p = threadIdx.x; p < npairs; p += BLK) {
            const uint2 t = pair_tab[p];
            double f[LG], r[LG];
#pragma unroll
            for (int a = 0; a < LG; a++) {
                const double *kl = k + ((size_t)xs[a].l * npairs + p) * 2;
                f[a] = kl[0];
                r[a] = kl[1];
            }
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const double *yf = yl + LG * VK_IX(t.x >> 8 * q & 255, ni + 2, VK_SITE_SPECIES);
                const double *yr = yl + LG * VK_IX(t.y >> 8 * q & 255, ni + 2, VK_SITE_SPECIES);
#pragma unroll
                for (int a = 0; a < LG; a++) {
                    f[a] = f[a] * yf[a];
                    r[a] = r[a] * yr[a];
                }
            }
#pragma unroll
            for (int a = 0; a < LG; a++) v[LG * p + a] = f[a] - r[a];
        }
        __syncthreads();
    }
    for (int q = threadIdx.x; q < LG * ni; q += BLK) {
        const int a = q / ni, i = q - a * ni;
        LayerCtx x = xs[0];
        bool go = on[0];
        if (LG > 1 && a > 0) {
            x = xs[LG - 1];
            go = on[LG - 1];
        }
        if (!go) continue;
        const int l = x.l;
        double ysm = 0.0, ys0 = 0.0, ysp = 0.0;
        if (mode & 2) ysum_around(ysum, x, ysm, ys0, ysp);
        double chem = 0.0;
        if (mode & 1) {
            const int n = chem_ptr[i + 1] - chem_ptr[i];
            if (n > 0) {
                int2 t = chem_ent[VK_IX(i, nchem, VK_SITE_CHEM)];   // (pair, sign)
                chem = t.y * v[LG * VK_IX(t.x, npairs, VK_SITE_PAIR) + a];
                // the terms in order, eight entries loaded ahead of their sums
                int e = 1;
                for (; e + 8 <= n; e += 8) {
                    int2 tt[8];
#pragma unroll
                    for (int u = 0; u < 8; u++) tt[u] = chem_ent[VK_IX((e + u) * ni + i, nchem, VK_SITE_CHEM)];
#pragma unroll
                    for (int u = 0; u < 8; u++) chem = chem + tt[u].y * v[LG * VK_IX(tt[u].x, npairs, VK_SITE_PAIR) + a];
                }
                for (; e < n; e++) {
                    t = chem_ent[VK_IX(e * ni + i, nchem, VK_SITE_CHEM)];
                    chem = chem + t.y * v[LG * VK_IX(t.x, npairs, VK_SITE_PAIR) + a];
                }
            }
        }
        const ColAtm ca = col_atm(atm, x.c, x.off, x.nz, ni);
        double val = chem;
        if (mode & 2) {
            double ym = x.j > 0 ? y[(size_t)(l - 1) * ni + i] : 0.0;
            double yp = x.j < x.nz - 1 ? y[(size_t)(l + 1) * ni + i] : 0.0;
            double d = diff_value(ca, x.j, i, ysm, ys0, ysp, ym, yl[LG * i + a], yp, ms[i], alpha[i], mol != 0);
            val = (mode & 1) ? chem + d : d;
        }
        if (k1) val = val - 2. / (R_ROS * dtc[x.c]) * k1[(size_t)l * ni + i];
        out[(size_t)l * ni + i] = val;
    }
}

// ---------------------------------------------------------------------------
// Jacobian blocks (mode 0: J = d chemdf/dy) or Ros2 lhs blocks (mode 1:
// D = c0 I - J - J_diff, Lsub, Usup), one workgroup per LG layers.
//
// Bound by instructions and the table reads, not by the block it writes: the
// tables (38 KB of slots, 70 KB of entries for 93 species and 620 pairs) are
// laid out so that a slot is two products of three looked-up amounts and an
// entry's first two terms come with it, and with two layers a workgroup reads
// them once for both (a slot's values of the layers side by side in LDS).
// 93 species, 620 pairs: 36 000 layers 1695 -> 1310 us (1435 with one layer a
// workgroup; the vector cache waits on L2 for four fifths of it, the 2.7 GB of
// sectors it touches take 0.4 ms), 2048 layers 139 -> 76 us, 150 layers
// 39 -> 22 us.
// ---------------------------------------------------------------------------

// The diagonal of a layer's lhs block after c0 - J: the diffusion terms in
// the reference's order.  xmode 1: the escape term first (top layer, _vm
// operators, op.py:2101-2107); xmode 2: the deposition velocity last (bottom
// layer, op.py:2029).
struct LhsDiag {
    double c0;
    int xmode, mol;
    const double *dg0, *dg1, *dgx;       // per species
    __device__ __forceinline__ double operator()(double val, int i) const {
        val = c0 + val;
        if (xmode == 1) val = val - dgx[i];
        val = val - dg0[i];
        if (mol) val = val - dg1[i];
        if (xmode == 2) val = val - dgx[i];
        return val;
    }
};

// J += (or =) a packed term, for each layer
template <int LG>
__device__ __forceinline__ void add_term(double (&J)[LG], bool first, int t, const double *dv, int nslot) {
    const double c = vk_jac_coef(t);
    const double *d = dv + LG * VK_IX(vk_jac_slot(t), nslot, VK_SITE_SLOT);
#pragma unroll
    for (int a = 0; a < LG; a++) J[a] = first ? c * d[a] : J[a] + c * d[a];
}

// NTH threads for the LG layers, WAVES a SIMD
template <int LG, int NTH, int WAVES>
__global__ void __launch_bounds__(NTH, WAVES) k_jac_lhs(
    int L, int ni, int npairs, int nslot, int nlight, int nheavy, int njac, const int *__restrict__ off,
    const int *__restrict__ layer_col, const int *__restrict__ reac, const int *__restrict__ prod,
    const int4 *__restrict__ slot_tab, const int4 *__restrict__ jac_ent, const int4 *__restrict__ jac_light,
    const int *__restrict__ jac_emap, const int *__restrict__ jac_tp, const double *__restrict__ ms,
    const double *__restrict__ alpha, vk_atm atm, const double *__restrict__ y, const double *__restrict__ k,
    const double *__restrict__ M, int mode, int mol, const double *__restrict__ dtc, const double *__restrict__ ysum,
    const vk_colstate *__restrict__ st, double *__restrict__ D, double *__restrict__ Lsub, double *__restrict__ Usup,
    int write_zeros) {
    extern __shared__ __align__(16) double smem[];
    double *dv = smem;                                 // nslot x LG
    double *yl = dv + LG * nslot;                      // (ni + 2) x LG: amounts, then M and one
    double *dg = yl + LG * (VK_NI_MAX + 2);            // LG x 3 VK_NI_MAX: terms of the diagonal, per species
    const int l0 = blockIdx.x * LG, nn = ni * ni;
    LayerCtx x[LG];
    bool on[LG], any = false;
#pragma unroll
    for (int a = 0; a < LG; a++) {
        x[a] = layer_ctx(off, layer_col, min(l0 + a, L - 1));
        on[a] = l0 + a < L && !(st && st[x[a].c].done);
        any = any || on[a];
    }
    if (!any) return;
    for (int q = threadIdx.x; q < ni + 2; q += NTH)
#pragma unroll
        for (int a = 0; a < LG; a++)
            yl[LG * q + a] = q < ni ? y[(size_t)x[a].l * ni + q] : (q == ni ? M[x[a].l] : 1.0);
    __syncthreads();   // the slot derivatives read yl
    for (int s = threadIdx.x; s < nslot; s += NTH) {
        const int4 e = slot_tab[s];
        const int p = VK_IX(e.x, npairs, VK_SITE_SLOTPAIR);
        double kf[LG], kb[LG], d[LG];
#pragma unroll
        for (int a = 0; a < LG; a++) {
            const double *kl = k + ((size_t)x[a].l * npairs + p) * 2;
            kf[a] = kl[0];
            kb[a] = kl[1];
        }
        auto product = [&](int side, const double (&kc)[LG], double sign) {
            const double *f0 = yl + LG * VK_IX(side & 255, ni + 2, VK_SITE_SPECIES);
            const double *f1 = yl + LG * VK_IX(side >> 8 & 255, ni + 2, VK_SITE_SPECIES);
            const double *f2 = yl + LG * VK_IX(side >> 16 & 255, ni + 2, VK_SITE_SPECIES);
#pragma unroll
            for (int a = 0; a < LG; a++) {
                const double v = kc[a] * f0[a] * f1[a] * f2[a];
                d[a] = sign > 0 ? (side >> 24 ? v : 0.0) : d[a] - (side >> 24 ? v : 0.0);
            }
        };
        product(e.y, kf, 1.0);
        product(e.z, kb, -1.0);
        if (((e.y | e.z) >> 24) & 2) {
            const int4 rt = ((const int4 *)reac)[p], pt = ((const int4 *)prod)[p];
#pragma unroll
            for (int a = 0; a < LG; a++) {
                const double m = yl[LG * ni + a];
                d[a] = dside<LG>(rt, kf[a], yl + a, m, e.w, ni) - dside<LG>(pt, kb[a], yl + a, m, e.w, ni);
            }
        }
#pragma unroll
        for (int a = 0; a < LG; a++) dv[LG * s + a] = d[a];
    }
    LhsDiag diag[LG];
#pragma unroll
    for (int a = 0; a < LG; a++) {
        double *dg0 = dg + 3 * VK_NI_MAX * a, *dg1 = dg0 + VK_NI_MAX, *dgx = dg1 + VK_NI_MAX;
        diag[a] = {0.0, 0, mol, dg0, dg1, dgx};
        if (mode != 1) continue;
        // diffusion part of the lhs (op.py:2012-2040): once per species
        const LayerCtx &xa = x[a];
        diag[a].c0 = 1. / (R_ROS * dtc[xa.c]);
        double ysm, ys0, ysp;
        ysum_around(ysum, xa, ysm, ys0, ysp);
        ColAtm ca = col_atm(atm, xa.c, xa.off, xa.nz, ni);
        int xmode = 0;
        if (xa.j == 0 && ca.use_bot) xmode = 2;
        else if (xa.j == xa.nz - 1 && ca.vm && mol && atm.top_flux && esc_any(atm)) xmode = 1;
        diag[a].xmode = xmode;
        // each layer's species on threads of their own
        for (int i = (int)threadIdx.x - NTH / LG * a; i < ni; i += NTH) {
            if (i < 0) continue;
            LhsDiff r = lhs_diff(ca, xa.j, i, ysm, ys0, ysp, ms[i], alpha[i], mol != 0);
            dg0[i] = r.d0;
            dg1[i] = r.d1;
            if (xmode == 2) {
                dgx[i] = -1. * ca.bot_vdep[i] / ca.dzi[0];
            } else if (xmode == 1) {
                // diff_lim = top_flux / y for escaping species with y > 0 (no 1/dzi, as there)
                double e = 0.0;
                if (((atm.esc[i >> 5] >> (i & 31)) & 1u) && yl[LG * i + a] > 0)
                    e = 0.0 + atm.top_flux[(size_t)xa.c * ni + i] / yl[LG * i + a];
                dgx[i] = e;
            }
            double u = 0.0, lo = 0.0;
            if (r.has_u) { u = 0.0 - r.u0; if (r.has_mol) u = u - r.u1; }
            if (r.has_l) { lo = 0.0 - r.l0; if (r.has_mol) lo = lo - r.l1; }
            if (blockIdx.y == 0 && on[a]) {
                Usup[(size_t)xa.l * ni + i] = u;
                Lsub[(size_t)xa.l * ni + i] = lo;
            }
        }
    }
    __syncthreads();
    // Every dense entry is written once (the structural zeros only with
    // write_zeros: the integrator clears its blocks once and skips them): the
    // few long term lists (jac_ent[0, nheavy): the list is sorted by term
    // count) by threads of their own, the others in one nearly coalesced pass
    // in the order of the dense index.  With the zeros that pass runs over the
    // dense index itself and writes whole lines where there are many layers
    // (the zeros in a pass behind the entries: 32 768 layers of 150 species 4.11
    // ms for 3.15); the lanes on zeros then wait for the others, so few layers
    // keep the pass behind (64 layers 38 us for 46).  With few layers the entries
    // of a layer are split over the grid's y dimension (each workgroup forms the
    // layer's shared terms itself).
    auto store = [&](int e, const double (&J)[LG], bool dg) {
        e = VK_IX(e, nn, VK_SITE_DENSE);
#pragma unroll
        for (int a = 0; a < LG; a++) {
            double val = J[a];
            if (mode) {
                val = -val;
                if (dg) val = diag[a](val, e / (ni + 1));
            }
            if (on[a]) D[(size_t)x[a].l * nn + e] = val;
        }
    };
    const int e0 = threadIdx.x + blockIdx.y * NTH, es = NTH * gridDim.y;
    for (int q = e0; q < nheavy; q += es) {
        const int4 en = jac_ent[q];       // (dense index, first term, end of terms, row)
        double J[LG];
        add_term<LG>(J, true, jac_tp[VK_IX(en.y, njac, VK_SITE_TERM)], dv, nslot);
        // terms in order; eight loads in flight per round
        int u = en.y + 1;
        for (; u + 8 <= en.z; u += 8) {
            int t[8];
#pragma unroll
            for (int m = 0; m < 8; m++) t[m] = jac_tp[VK_IX(u + m, njac, VK_SITE_TERM)];
#pragma unroll
            for (int m = 0; m < 8; m++) add_term<LG>(J, false, t[m], dv, nslot);
        }
        for (; u < en.z; u++) add_term<LG>(J, false, jac_tp[VK_IX(u, njac, VK_SITE_TERM)], dv, nslot);
        store(en.x, J, en.x == en.w * (ni + 1));
    }
    auto light = [&](int q) {
        const int4 en = jac_light[q];
        const int nt = en.x >> 16 & 15;
        int t[VK_JAC_LIGHT];
#pragma unroll
        for (int m = 2; m < VK_JAC_LIGHT; m++) t[m] = m < nt ? jac_tp[VK_IX(en.y + m, njac, VK_SITE_TERM)] : 0;
        double J[LG] = {};
        if (nt > 0) add_term<LG>(J, true, en.z, dv, nslot);
        if (nt > 1) add_term<LG>(J, false, en.w, dv, nslot);
#pragma unroll
        for (int m = 2; m < VK_JAC_LIGHT; m++)
            if (m < nt) add_term<LG>(J, false, t[m], dv, nslot);
        store(en.x & 0xffff, J, en.x >> 20);
    };
    auto zero = [&](int e) {
        if (jac_emap[e] == VK_JAC_ZERO)
#pragma unroll
            for (int a = 0; a < LG; a++)
                if (on[a]) D[(size_t)x[a].l * nn + e] = 0.0;
    };
    if (LG > 1 && write_zeros) {
#pragma unroll 2
        for (int e = e0; e < nn; e += es) {
            const int q = jac_emap[e];
            if (q >= 0) light(q);
            else zero(e);
        }
        return;
    }
#pragma unroll 2
    for (int q = e0; q < nlight; q += es) light(q);
    if (write_zeros)
        for (int e = e0; e < nn; e += es) zero(e);
}

}  // namespace

// ---------------------------------------------------------------------------
// host entry points
// ---------------------------------------------------------------------------

static inline hipStream_t S(void *s) { return (hipStream_t)s; }

static size_t rhs_smem(const vk_plan *p, int layers) {
    return sizeof(double) * layers * (p->ni + 2 + (size_t)p->npairs);
}
static size_t jac_smem(const vk_plan *p, int layers) {
    return sizeof(double) * layers * (4 * VK_NI_MAX + 2 + (size_t)p->nslot);
}

extern "C" int vk_rates(const vk_plan *plan, const vk_columns *cols, const vk_atm *atm, double *d_k, void *stream) {
    if (!plan || !cols || !atm || !d_k) return VK_EINVAL;
    const int L = cols->L, cu = vk_device_cus();
    // layers per workgroup: the most (their pairs' parameters are read once)
    // that leave about three workgroups per CU (93 species, 620 pairs, one, two,
    // four, eight layers: 1 536 layers 26, 21, 28, 38 us, 3 008 layers 42, 36, 32,
    // 46, 6 144 layers 76, 60, 54, 51); below that one layer each, and its pairs
    // over several workgroups, each of which forms what the layer's pairs share,
    // only to give every CU two (1 024 layers over three 27 us, over one 18)
    int LG = RATE_LAYERS;
    while (LG > 1 && 4L * L < 11L * cu * LG) LG /= 2;
    const int split = LG > 1 ? 1 : std::max(1, std::min((plan->npairs + BLK - 1) / BLK, 2 * cu / std::max(L, 1)));
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
    auto launch = [&](auto kernel, int layers) {
        hipLaunchKernelGGL(kernel, dim3((cols->L + layers - 1) / layers), dim3(BLK), rhs_smem(plan, layers), s, cols->L,
                           plan->ni, plan->npairs, plan->nchem_ent, cols->d_off, cols->d_layer_col, plan->pair_tab,
                           plan->chem_ptr, plan->chem_ent, plan->ms, plan->alpha, a, y, k, atm->M, mode, mol, k1, dtc,
                           ysum, st, out);
    };
    // two layers a workgroup where a CU holds eight such workgroups and still gets
    // several (30 and 93 species: 3 008 layers, one each, 11.8 and 21.1 us, 3 072
    // layers, two, 9.8 and 19.9)
    if (rhs_smem(plan, 2) <= 20 * 1024 && cols->L >= 12 * vk_device_cus())
        launch(k_rhs<2>, 2);
    else
        launch(k_rhs<1>, 1);
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
    const int ncu = vk_device_cus();
    auto launch = [&](auto kernel, int layers, int threads, int gy) {
        hipLaunchKernelGGL(kernel, dim3((cols->L + layers - 1) / layers, gy), dim3(threads), jac_smem(plan, layers), s,
                           cols->L, plan->ni, plan->npairs, plan->nslot, plan->njlight, plan->njheavy, plan->njac,
                           cols->d_off, cols->d_layer_col, plan->reac, plan->prod, plan->slot_tab, plan->jac_ent,
                           plan->jac_light, plan->jac_emap, plan->jac_tp, plan->ms, plan->alpha, a, y, k, M, mode, mol,
                           dtc, ysum, st, D, Lsub, Usup, (int)write_zeros);
    };
    // Up to one layer a CU: one layer a workgroup, its entries over up to 4 of
    // them.  Beyond, two layers a workgroup (448 layers of 150 species 53
    // against 65 us, 93 species 40 against 43) where two such workgroups fit a
    // CU's 160 KB.  What a small network's layer takes is latency, so with six
    // layers a CU and more its two layers run on 256 threads where the LDS then
    // holds as many waves as with 512 (four workgroups) or more (six), for the
    // layers in flight: 32 768 layers, 512 threads against 256 of four and of six
    // workgroups: 30 species 445, 308, 267 us, 40 species 566, 417, 351, 61
    // species 808, 714, 751, 93 species (three workgroups) 1217, 1325, 1368; 61
    // species, 1024 layers 37 against 44 and 2048 layers 57 against 51.
    const size_t two = jac_smem(plan, 2);
    if (two > 80 * 1024 || cols->L <= ncu)
        launch(k_jac_lhs<1, BLK, 4>, 1, BLK, ncu > 0 ? std::max(1, std::min(4, 2 * ncu / std::max(cols->L, 1))) : 1);
    else if (two > 160 * 1024 / 4 || cols->L < 6 * ncu)
        launch(k_jac_lhs<2, 2 * BLK, 4>, 2, 2 * BLK, 1);
    else if (two > 160 * 1024 / 6)
        launch(k_jac_lhs<2, BLK, 4>, 2, BLK, 1);
    else
        launch(k_jac_lhs<2, BLK, 6>, 2, BLK, 1);
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
