// Photochemical radiative transfer on the device: optical depth, two-stream
// diffuse flux and photolysis rates (ODESolver.compute_tau / compute_flux /
// compute_J, op.py:2580-2787), refreshed every update_photo_frq steps of the
// integration loop (op.py:818-830).
//
// Layout per column c with nz layers (layers off[c] .. off[c+1]-1 of the
// stack): the staggered level arrays (tau, direct beam, diffuse up / down
// fluxes; nz + 1 levels) occupy rows off[c] + c .. off[c] + c + nz of
// [L + ncols][nbin]; the layer arrays (single-scattering albedo, actinic
// flux) rows off[c] .. of [L][nbin].  One thread per (column, wavelength
// bin) sweeps the layers: every bin is independent, and consecutive threads
// read consecutive bins of a row (coalesced).
#include <algorithm>

#include "vk_internal.h"
#include "vk_device.h"

namespace {

// the tables and state the kernels read (plain data, passed by value)
struct PhotoDev {
    int nbin, nabs, nscat, nbranch, nT, nTJ, din12;
    double dbin1, dbin2, cos_sl, edd, f_diurnal, flux_atol;
    int ncols, L;
    int *abs_sp, *abs_T, *scat_sp, *br_col, *br_T;
    double *bins, *sflux_top, *cross, *cross_T, *cross_scat, *cross_J, *cross_J_T, *hc_bin;
    double *tau, *sflux, *dflux_u, *dflux_d, *w0, *aflux;
    unsigned long long *change;   // per column: max relative change (bits of a positive double)
    int *last, *switched, *due;   // per column: count of the last update, final frequency on, update now
};

}  // namespace

struct vk_photo {
    PhotoDev d;
    std::vector<void *> allocs;
};

namespace {

constexpr int PT = 256;

// per column: is an update due at this attempt (force, or the first attempt
// of a step whose count is a multiple of the frequency in force, op.py:818-827)
__global__ void k_photo_due(int ncols, const vk_colstate *__restrict__ st, int force, int ini_frq, int final_frq,
                            double yconv_min, int *__restrict__ last, int *__restrict__ switched,
                            int *__restrict__ due, unsigned long long *__restrict__ change) {
    const int c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= ncols) return;
    change[c] = 0ull;
    // a forced update (the set-up call before the loop, vulcan.py:172-174)
    // leaves the loop's own schedule alone: its first step updates again
    if (force) { due[c] = 1; return; }
    const vk_colstate s = st[c];
    if (s.done) { due[c] = 0; return; }
    if (!switched[c] && s.longdy < yconv_min * 10. && s.longdydt < 1.e-6) switched[c] = 1;
    const int frq = switched[c] ? final_frq : ini_frq;
    const int d = (s.count % frq == 0) && last[c] != s.count;
    if (d) last[c] = s.count;
    due[c] = d;
}

// optical depth (op.py:2580-2601) and single-scattering albedo (op.py:2627-2639)
__global__ void __launch_bounds__(PT) k_photo_tau(PhotoDev ph, int ni, const int *__restrict__ off,
                                                  const double *__restrict__ y, const double *__restrict__ ymix,
                                                  const double *__restrict__ dz) {
    const int c = blockIdx.y, b = blockIdx.x * PT + threadIdx.x;
    if (!ph.due[c] || b >= ph.nbin) return;
    const int o = off[c], nz = off[c + 1] - o, nb = ph.nbin;
    const size_t top = (size_t)(o + c + nz) * nb + b;
    ph.tau[top] = 0.0;
    double above = 0.0;
    for (int j = nz - 1; j >= 0; j--) {
        const int l = o + j;
        const double *yl = y + (size_t)l * ni, *ml = ymix + (size_t)l * ni;
        const double dzl = dz[l];
        double t = 0.0, tabs = 0.0, tscat = 0.0;
        for (int a = 0; a < ph.nabs; a++) {
            const int sp = ph.abs_sp[a], tt = ph.abs_T[a];
            const double cr = ph.cross[(size_t)a * nb + b];
            const double crt = tt >= 0 ? ph.cross_T[((size_t)tt * ph.L + l) * nb + b] : cr;
            t += yl[sp] * dzl * crt;
            tabs += ml[sp] * cr;
        }
        for (int q = 0; q < ph.nscat; q++) {
            const int sp = ph.scat_sp[q];
            const double cr = ph.cross_scat[(size_t)q * nb + b];
            t += yl[sp] * dzl * cr;
            tscat += ml[sp] * cr;
        }
        above = t + above;
        ph.tau[(size_t)(o + c + j) * nb + b] = above;
        double w = tscat / (tabs + tscat);
        if (w != w) w = 0.0;                       // nan_to_num: 0/0
        w = fmin(w, 1. - 1.E-8);
        ph.w0[(size_t)l * nb + b] = w;
    }
}

// two-stream coefficients of layer l (op.py:2648-2677, isotropic scattering)
struct TwoStream {
    double chi, xi, phi, i_u, i_d;
};

__device__ inline TwoStream two_stream(const PhotoDev &ph, double mu, double w, double dtau, double dir_lo,
                                       double dir_hi) {
    const double edd = ph.edd;
    const double s1 = sqrt(1. - w);
    const double tran = exp(-1. / edd * s1 * dtau);
    const double zp = 0.5 * (1. + s1), zm = 0.5 * (1. - s1);
    const double ll = -1. * w / (1. / (mu * mu) - 1. / (edd * edd) * (1. - w));
    const double gp = 0.5 * (ll * (1. / edd + 1. / mu)), gm = 0.5 * (ll * (1. / edd - 1. / mu));
    TwoStream r;
    r.chi = zm * zm * (tran * tran) - zp * zp;
    r.xi = zp * zm * (1. - tran * tran);
    r.phi = (zm * zm - zp * zp) * tran;
    r.i_u = r.phi * gp * dir_lo - (r.xi * gm + r.chi * gp) * dir_hi;
    r.i_d = r.phi * gm * dir_hi - (r.chi * gm + r.xi * gp) * dir_lo;
    return r;
}

// direct beam, diffuse fluxes by a downward then an upward sweep, actinic
// flux and its relative change (op.py:2603-2738)
__global__ void __launch_bounds__(PT) k_photo_flux(PhotoDev ph, const int *__restrict__ off) {
    const int c = blockIdx.y;
    if (!ph.due[c]) return;                          // uniform over the workgroup
    // threads past the last bin take part in the reduction below only
    const int b = min(blockIdx.x * PT + threadIdx.x, ph.nbin - 1);
    const bool mine = blockIdx.x * PT + threadIdx.x < ph.nbin;
    double mx = 0.0;
    if (mine) {
        const int o = off[c], nz = off[c + 1] - o, nb = ph.nbin;
        const double mu = -1. * ph.cos_sl, top = ph.sflux_top[b];
        const size_t base = (size_t)(o + c) * nb + b;   // level 0 of the column
        double *tau = ph.tau + base, *sf = ph.sflux + base, *du = ph.dflux_u + base, *dd = ph.dflux_d + base;
        for (int j = 0; j <= nz; j++) sf[(size_t)j * nb] = top * exp(-1. * tau[(size_t)j * nb] / ph.cos_sl);
        // downward: dflux_d[j] from dflux_d[j+1] and the previous update's dflux_u[j]
        for (int j = nz - 1; j >= 0; j--) {
            const size_t lj = (size_t)j * nb;
            const TwoStream t = two_stream(ph, mu, ph.w0[(size_t)(o + j) * nb + b], tau[lj] - tau[lj + nb],
                                           sf[lj] * ph.cos_sl, sf[lj + nb] * ph.cos_sl);
            dd[lj] = 1. / t.chi * (t.phi * dd[lj + nb] - t.xi * du[lj] + t.i_d / mu);
        }
        // upward
        for (int j = 1; j <= nz; j++) {
            const size_t lj = (size_t)(j - 1) * nb;
            const TwoStream t = two_stream(ph, mu, ph.w0[(size_t)(o + j - 1) * nb + b], tau[lj] - tau[lj + nb],
                                           sf[lj] * ph.cos_sl, sf[lj + nb] * ph.cos_sl);
            du[lj + nb] = 1. / t.chi * (t.phi * du[lj] - t.xi * dd[lj + nb] + t.i_u / mu);
        }
        // actinic flux and the largest relative change over the bins above flux_atol
        for (int j = 0; j < nz; j++) {
            const size_t lj = (size_t)j * nb;
            const double ave = 0.5 * (sf[lj] + sf[lj + nb]);
            const double tot = ave + 0.5 * (du[lj] + du[lj + nb] + dd[lj + nb] + dd[lj]) / ph.edd;
            const double af = tot / ph.hc_bin[b];
            double *ap = ph.aflux + (size_t)(o + j) * nb + b;
            const double prev = *ap;
            *ap = af;
            if (af > ph.flux_atol) {
                const double ch = fabs(af - prev) / af;
                if (ch == ch) mx = fmax(mx, ch);
            }
        }
    }
    // positive doubles order as their bit patterns
    __shared__ double red[PT];
    red[threadIdx.x] = mx;
    __syncthreads();
    for (int w = PT / 2; w > 0; w >>= 1) {
        if (threadIdx.x < w) red[threadIdx.x] = fmax(red[threadIdx.x], red[threadIdx.x + w]);
        __syncthreads();
    }
    if (threadIdx.x == 0 && red[0] > 0.0)
        atomicMax(&ph.change[c], (unsigned long long)__double_as_longlong(red[0]));
}

// ---------------------------------------------------------------------------
// The same optical depth and fluxes by two kernels that do what a layer
// contributes on its own for many layers at once, and leave to one thread
// per bin the running sum of the optical depth and the sweeps' few serial
// operations.  Every value is formed by the operations of k_photo_tau and
// k_photo_flux in their order.  A thread per bin doing all of it (k_photo_tau, k_photo_flux)
// keeps 10 workgroups busy for one column, each waiting on memory and on the
// coefficients' latency layer after layer.  150 layers of 2 588 bins: 583 us
// each before, 15 us (k_photo_layers, bound by reading the cross sections
// from L2) and 37 us (k_photo_rt, a third of it the serial parts) now; 48
// columns: 1 125 us each before, 170 and 777 us now (three workgroups per CU
// by LDS).  photo_per_bin says where a thread per bin is the better choice.
// ---------------------------------------------------------------------------

// every layer's own optical depth (left in the tau row of its lower level)
// and single-scattering albedo (op.py:2580-2601, 2627-2639); PT bins and
// TAU_LAYERS layers per workgroup, so that a cross section is read once per
// TAU_LAYERS layers
constexpr int TAU_LAYERS = 8, TAU_SPECIES = 32;   // species per round through LDS

__global__ void __launch_bounds__(PT, 4) k_photo_layers(PhotoDev ph, int ni, const int *__restrict__ layer_col,
                                                     const double *__restrict__ y, const double *__restrict__ ymix,
                                                     const double *__restrict__ dz) {
    __shared__ double ny[TAU_SPECIES][TAU_LAYERS], mx[TAU_SPECIES][TAU_LAYERS];   // y dz and ymix
    // one dimension: a grid's y is 65 535 long, half a million layers
    const int nb = ph.nbin, groups = (nb + PT - 1) / PT;
    const int l0 = TAU_LAYERS * (blockIdx.x / groups), nl = min(TAU_LAYERS, ph.L - l0);
    const int bt = PT * (blockIdx.x % groups) + threadIdx.x, b = min(bt, nb - 1);
    const bool mine = bt < nb;
    // the layers' columns, seldom more than two: asked layer by layer this was most
    // of an attempt that updates nothing (256 columns, 2 588 bins: 57 us, 26 now)
    bool any = false;
    for (int c = layer_col[l0], last = layer_col[l0 + nl - 1]; c <= last; c++) any = any || ph.due[c];
    if (!any) return;
    double t[TAU_LAYERS], tabs[TAU_LAYERS], tscat[TAU_LAYERS];
#pragma unroll
    for (int q = 0; q < TAU_LAYERS; q++) t[q] = tabs[q] = tscat[q] = 0.0;
    // the species of a round: absorbers, then scatterers
    auto stage = [&](const int *list, int a0, int n) {
        __syncthreads();
        for (int e = threadIdx.x; e < n * TAU_LAYERS; e += PT) {
            const int a = e / TAU_LAYERS, q = e % TAU_LAYERS, l = l0 + min(q, nl - 1), sp = list[a0 + a];
            ny[a][q] = y[(size_t)l * ni + sp] * dz[l];
            mx[a][q] = ymix[(size_t)l * ni + sp];
        }
        __syncthreads();
    };
    for (int a0 = 0; a0 < ph.nabs; a0 += TAU_SPECIES) {
        const int n = min(TAU_SPECIES, ph.nabs - a0);
        stage(ph.abs_sp, a0, n);
#pragma unroll 2
        for (int a = 0; a < n; a++) {
            const int tt = ph.abs_T[a0 + a];
            const double cr = ph.cross[(size_t)(a0 + a) * nb + b];
            if (tt >= 0) {
                const double *ct = ph.cross_T + ((size_t)tt * ph.L + l0) * nb + b;
                double crt[TAU_LAYERS];
#pragma unroll
                for (int q = 0; q < TAU_LAYERS; q++) crt[q] = ct[(size_t)min(q, nl - 1) * nb];
#pragma unroll
                for (int q = 0; q < TAU_LAYERS; q++) t[q] += ny[a][q] * crt[q];
            } else {
#pragma unroll
                for (int q = 0; q < TAU_LAYERS; q++) t[q] += ny[a][q] * cr;
            }
#pragma unroll
            for (int q = 0; q < TAU_LAYERS; q++) tabs[q] += mx[a][q] * cr;
        }
    }
    for (int a0 = 0; a0 < ph.nscat; a0 += TAU_SPECIES) {
        const int n = min(TAU_SPECIES, ph.nscat - a0);
        stage(ph.scat_sp, a0, n);
        for (int a = 0; a < n; a++) {
            const double cr = ph.cross_scat[(size_t)(a0 + a) * nb + b];
#pragma unroll
            for (int q = 0; q < TAU_LAYERS; q++) {
                t[q] += ny[a][q] * cr;
                tscat[q] += mx[a][q] * cr;
            }
        }
    }
    if (!mine) return;
#pragma unroll
    for (int q = 0; q < TAU_LAYERS; q++) {
        if (q >= nl) break;
        const int l = l0 + q, c = layer_col[l];
        if (!ph.due[c]) continue;
        double w = tscat[q] / (tabs[q] + tscat[q]);
        if (w != w) w = 0.0;                       // nan_to_num: 0/0
        ph.tau[(size_t)(l + c) * nb + b] = t[q];
        ph.w0[(size_t)l * nb + b] = fmin(w, 1. - 1.E-8);
    }
}

// optical depth of the levels, direct beam, both sweeps, actinic flux
// (op.py:2603-2738): RT_BINS bins of a column per workgroup, 32 threads per
// bin.  A sweep's step is
//     F[j] = 1/chi (phi F[j'] - xi G + i / mu)
// with G the other flux at the layer's far level, known ahead of the
// downward sweep from the previous update, and of the upward one from the
// downward: xi G is formed ahead too, and four operations a layer stay
// serial, in the reference's order (as one multiply-add with 1/chi taken
// into the constants they lose six digits where xi G and i / mu cancel).
// RT_ARRAYS doubles per bin and level in LDS: the serial parts' latency is
// hidden by the other workgroups of a CU, so what a thread alone uses later
// (xi and i / mu of its up to RT_LANES-spaced R layers) waits in its
// registers, and the downward flux in global memory.  Columns of up to 416
// layers run here; longer ones keep k_photo_tau and k_photo_flux.
constexpr int RT_BINS = 8, RT_LANES = PT / RT_BINS, RT_ARRAYS = 4, RT_RUN = 8, RT_ROUNDS = 13;

constexpr size_t rt_lds(int nz) { return sizeof(double) * RT_ARRAYS * RT_BINS * (size_t)(nz + 1); }

// f = inv (phi f - xg + F) over n layers from j in steps of dj, f into F;
// RT_RUN layers are read ahead of the chain and written behind it (a store
// between two layers' loads would put an LDS round trip into every step)
__device__ __forceinline__ void rt_sweep(const double *inv, const double *phi, const double *xg, double *F, int j, int dj,
                                         int n, double f) {
    for (int q0 = 0; q0 < n; q0 += RT_RUN) {
        double i[RT_RUN], p[RT_RUN], x[RT_RUN], v[RT_RUN];
#pragma unroll
        for (int q = 0; q < RT_RUN; q++) {
            const int e = RT_BINS * (j + dj * min(q0 + q, n - 1));
            i[q] = inv[e]; p[q] = phi[e]; x[q] = xg[e]; v[q] = F[e];
        }
#pragma unroll
        for (int q = 0; q < RT_RUN; q++) v[q] = f = i[q] * (p[q] * f - x[q] + v[q]);
#pragma unroll
        for (int q = 0; q < RT_RUN; q++)
            if (q0 + q < n) F[RT_BINS * (j + dj * (q0 + q))] = v[q];
    }
}

// R: rounds of RT_LANES layers that cover the longest column
template <int R>
__global__ void __launch_bounds__(PT) k_photo_rt(PhotoDev ph, const int *__restrict__ off) {
    extern __shared__ double rt[];
    const int c = blockIdx.y;
    if (!ph.due[c]) return;
    const int o = off[c], nz = off[c + 1] - o, nb = ph.nbin, span = RT_BINS * (nz + 1);
    const int bl = threadIdx.x % RT_BINS, j0 = threadIdx.x / RT_BINS;
    const bool mine = blockIdx.x * RT_BINS + bl < nb;
    const int b = min((int)blockIdx.x * RT_BINS + bl, nb - 1);
    // [level][bin] each; F holds i / mu until the fluxes replace it
    double *inv = rt + bl, *phi = inv + span, *xg = phi + span, *F = xg + span;
    const size_t base = (size_t)(o + c) * nb + b;           // level 0 of the column
    auto at = [](int j) { return j * RT_BINS; };
    double *tau = inv;
#pragma unroll
    for (int r = 0; r < R; r++) {
        const int j = j0 + RT_LANES * r;
        if (j < nz) tau[at(j)] = ph.tau[base + (size_t)j * nb];
    }
    __syncthreads();
    if (j0 == 0) {
        double above = 0.0;
        tau[at(nz)] = 0.0;
        for (int j = nz - 1; j >= 0; j -= RT_RUN) {
            double v[RT_RUN];
#pragma unroll
            for (int u = 0; u < RT_RUN; u++) v[u] = tau[at(max(j - u, 0))];
#pragma unroll
            for (int u = 0; u < RT_RUN; u++) v[u] = above = v[u] + above;
#pragma unroll
            for (int u = 0; u < RT_RUN; u++)
                if (j - u >= 0) tau[at(j - u)] = v[u];
        }
    }
    __syncthreads();
    const double mu = -1. * ph.cos_sl, top = ph.sflux_top[b];
    double *sf = xg;
    for (int j = j0; j <= nz; j += RT_LANES) {
        const double t = tau[at(j)], f = top * exp(-1. * t / ph.cos_sl);
        sf[at(j)] = f;
        F[at(j)] = t;                    // tau again, for the layers' differences
        if (mine) {
            ph.tau[base + (size_t)j * nb] = t;
            ph.sflux[base + (size_t)j * nb] = f;
        }
    }
    __syncthreads();
    // the coefficients take tau's and the beam's places a round of layers
    // behind their reads
    double xi[R], iu[R];
#pragma unroll
    for (int r = 0; r < R; r++) {
        const int j = j0 + RT_LANES * r;
        TwoStream t = {};
        double prev = 0.0;
        if (j < nz) {
            t = two_stream(ph, mu, ph.w0[(size_t)(o + j) * nb + b], F[at(j)] - F[at(j + 1)], sf[at(j)] * ph.cos_sl,
                           sf[at(j + 1)] * ph.cos_sl);
            prev = ph.dflux_u[base + (size_t)j * nb];
        }
        __syncthreads();
        if (j < nz) {
            inv[at(j)] = 1. / t.chi;
            phi[at(j)] = t.phi;
            xg[at(j)] = t.xi * prev;
            F[at(j)] = t.i_d / mu;
        }
        xi[r] = t.xi;
        iu[r] = t.i_u / mu;
    }
    __syncthreads();
    if (j0 == 0) {
        const double d = ph.dflux_d[base + (size_t)nz * nb];
        F[at(nz)] = d;
        rt_sweep(inv, phi, xg, F, nz - 1, -1, nz, d);
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < R; r++) {
        const int j = j0 + RT_LANES * r;
        if (j < nz) {
            xg[at(j)] = xi[r] * F[at(j + 1)];
            if (mine) ph.dflux_d[base + (size_t)j * nb] = F[at(j)];
        }
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < R; r++) {
        const int j = j0 + RT_LANES * r;
        if (j < nz) F[at(j)] = iu[r];
    }
    __syncthreads();
    // the upward flux of level j + 1 in layer j's place
    if (j0 == 0) rt_sweep(inv, phi, xg, F, 0, 1, nz, ph.dflux_u[base]);
    __syncthreads();
    // actinic flux and the largest relative change over the bins above flux_atol
    double mx = 0.0;
    if (mine) {
        const double hc = ph.hc_bin[b];
        for (int j = j0; j < nz; j += RT_LANES) {
            const size_t lj = base + (size_t)j * nb;
            const double ulo = j > 0 ? F[at(j - 1)] : ph.dflux_u[base], uhi = F[at(j)];
            const double ave = 0.5 * (ph.sflux[lj] + ph.sflux[lj + nb]);
            const double tot = ave + 0.5 * (ulo + uhi + ph.dflux_d[lj + nb] + ph.dflux_d[lj]) / ph.edd;
            const double af = tot / hc;
            ph.dflux_u[lj + nb] = uhi;
            double *ap = ph.aflux + (size_t)(o + j) * nb + b;
            const double prev = *ap;
            *ap = af;
            if (af > ph.flux_atol) {
                const double ch = fabs(af - prev) / af;
                if (ch == ch) mx = fmax(mx, ch);
            }
        }
    }
    for (int m = 32; m > 0; m >>= 1) mx = fmax(mx, __shfl_xor(mx, m));
    // positive doubles order as their bit patterns
    if ((threadIdx.x & 63) == 0 && mx > 0.0)
        atomicMax(&ph.change[c], (unsigned long long)__double_as_longlong(mx));
}

// Whether a thread per bin (k_photo_tau, k_photo_flux) is faster than
// k_photo_layers and k_photo_rt: its time is a chain over the layers, 7 us each,
// until the columns' bins fill the device, which k_photo_rt does with a few
// hundred.  Short columns leave most of its 32 threads a bin without a layer;
// from 213 layers its LDS lets two workgroups share a CU, from 320 one.  A thread
// per bin against the two kernels, us (bins x columns in thousands):
//   8 layers     50 /  42 (34)     75 /  98 (124)    807 / 2046 (2 588)
//   16 layers   140 / 131 (124)   260 / 381 (350)    834 / 1407 (1 294)
//   32 layers   314 / 289 (175)   437 / 431 (259)    947 / 1046 (647)
//   48 layers   379 / 266 (112)   567 / 494 (207)    932 /  988 (414)
//   64 layers  1078 / 941 (323)  2020 / 1835 (647)  4481 / 4296 (1 553)
//   150 layers 1455 / 810 (124)                     7492 / 6317 (1 035)
//   224 layers 2194 / 1772 (124) 3335 / 3615 (259)  6316 / 7204 (518)
//   300 layers 2910 / 2454 (124) 3783 / 4068 (210)  8444 / 9951 (518)
//   330 layers 2599 / 2354 (62)  2813 / 3490 (93)
//   416 layers 3306 / 2886 (62)  3512 / 4285 (93)   7350 / 14151 (311)
static bool photo_per_bin(int max_nz, long bins) {
    if (max_nz > RT_LANES * RT_ROUNDS) return true;
    if (max_nz < 64) return bins >= 8000L * max_nz;
    const long per_cu = 160 * 1024 / (long)rt_lds(max_nz);
    return per_cu <= 2 && bins >= 90000 * per_cu;
}

template <int R>
void launch_photo_rt(const PhotoDev &d, const vk_columns *cols, hipStream_t s) {
    hipLaunchKernelGGL((k_photo_rt<R>), dim3((d.nbin + RT_BINS - 1) / RT_BINS, cols->ncols), dim3(PT),
                       rt_lds(cols->max_nz), s, d, cols->d_off);
}

// photolysis rates of every branch (op.py:2751-2787): trapezoidal sums over
// the two uniform bin widths; the branch's rate column of k = J f_diurnal.
// One wave per branch for the LT layers of a workgroup, whose actinic flux
// is in LDS.  The cross sections are read once per workgroup from L2 (36
// branches of 2 588 bins: 0.75 MB; at one layer each, 48 columns read 4.8 GB
// in 0.65 ms; at four 0.38 ms), so batches take as many layers as LDS holds; a column or two
// take one, with the branches split over the grid's y dimension to fill the
// device.
constexpr int J_NT = 1024, J_LDS = 10400;   // doubles: four layers of 2 600 bins, or one of 10 400
// Below this many bins a workgroup has 4 waves, for the branches to share them
// evenly (36 over 16 waves take three rounds of which the last is a quarter
// full): 30 000 layers of 20, 100, 300 bins 362, 359, 410 -> 297, 299, 342 us, of
// 700 bins 530 us with 16.
constexpr int J_SMALL = 512, J_SMALL_NT = 256;

// STAGE: the actinic flux through LDS (spectra beyond J_LDS bins read it from
// memory for every branch)
template <int LT, int NTH, bool STAGE = true>
__global__ void __launch_bounds__(NTH) k_photo_J(PhotoDev ph, const int *__restrict__ layer_col, int nr,
                                                  double *__restrict__ k) {
    extern __shared__ double lds[];
    const int l0 = LT * blockIdx.x, nb = ph.nbin, nl = min(LT, ph.L - l0);
    const int w = threadIdx.x >> 6, lane = threadIdx.x & 63, nw = NTH / 64;
    const bool due = lane < nl && ph.due[layer_col[l0 + min(lane, nl - 1)]];   // lane: layer
    if (!__any(due)) return;
    const double *af = ph.aflux + (size_t)l0 * nb;
    if constexpr (STAGE) {
#pragma unroll 8
        for (int e = threadIdx.x; e < LT * nb; e += NTH) {
            const double a = af[min(e, nl * nb - 1)];
            lds[e] = e < nl * nb ? a : 0.0;
        }
        __syncthreads();
        af = lds;
    }
    const int d = ph.din12 >= 0 ? ph.din12 : nb - 1;
    for (int br = w + nw * blockIdx.y; br < ph.nbranch; br += nw * gridDim.y) {
        const int tt = ph.br_T[br];
        const double *cr = tt >= 0 ? ph.cross_J_T + ((size_t)tt * ph.L + l0) * nb : ph.cross_J + (size_t)br * nb;
        // the next layer's table (the last layer's own where there is none)
        auto row = [&](int q) { return tt >= 0 ? cr + (size_t)min(q, nl - 1) * nb : cr; };
        double s1[LT], s2[LT];
#pragma unroll
        for (int q = 0; q < LT; q++) s1[q] = s2[q] = 0.0;
        auto sum = [&](double (&s)[LT], int b0, int b1, double width) {
            if (tt >= 0) {
#pragma unroll 4
                for (int b = b0 + lane; b < b1; b += 64)
#pragma unroll
                    for (int q = 0; q < LT; q++) s[q] += af[q * nb + b] * row(q)[b] * width;
            } else {
#pragma unroll 8
                for (int b = b0 + lane; b < b1; b += 64) {
                    const double x = cr[b];
#pragma unroll
                    for (int q = 0; q < LT; q++) s[q] += af[q * nb + b] * x * width;
                }
            }
        };
        sum(s1, 0, d, ph.dbin1);
        sum(s2, d, nb, ph.dbin2);
        // lane q finishes layer q
        const double *x = row(lane), *a = af + min(lane, LT - 1) * nb;
        const double x0 = x[0], x1 = x[d - 1], x2 = x[d], x3 = x[nb - 1];
        double t1 = 0.0, t2 = 0.0;
#pragma unroll
        for (int q = 0; q < LT; q++) {
            for (int m = 32; m > 0; m >>= 1) {
                s1[q] += __shfl_xor(s1[q], m);
                s2[q] += __shfl_xor(s2[q], m);
            }
            t1 = lane == q ? s1[q] : t1;
            t2 = lane == q ? s2[q] : t2;
        }
        if (due) {
            double J = t1;
            J -= 0.5 * (a[0] * x0 + a[d - 1] * x1) * ph.dbin1;
            J += t2;
            J -= 0.5 * (a[d] * x2 + a[nb - 1] * x3) * ph.dbin2;
            k[(size_t)(l0 + lane) * nr + ph.br_col[br]] = J * ph.f_diurnal;
        }
    }
}

__global__ void k_photo_change(int ncols, const int *__restrict__ due, const unsigned long long *__restrict__ change,
                               vk_colstate *__restrict__ st) {
    const int c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= ncols || !due[c] || !st) return;
    st[c].aflux_change = __longlong_as_double((long long)change[c]);
}

template <typename T>
int dup(std::vector<void *> &v, T **p, const T *src, size_t n) {
    if (n == 0) n = 1, src = nullptr;
    if (hipMalloc((void **)p, sizeof(T) * n) != hipSuccess) return VK_ENOMEM;
    v.push_back(*p);
    if (src && hipMemcpy(*p, src, sizeof(T) * n, hipMemcpyHostToDevice) != hipSuccess) return VK_ENOMEM;
    if (!src && hipMemset(*p, 0, sizeof(T) * n) != hipSuccess) return VK_ENOMEM;
    return 0;
}

}  // namespace

extern "C" int vk_photo_create(const vk_plan *plan, const vk_columns *cols, const vk_photo_desc *d, vk_photo **out) {
    if (!plan || !cols || !d || !out || d->nbin < 2 || d->nabs < 0 || d->nscat < 0 || d->nbranch < 0 || d->nT < 0 ||
        d->nTJ < 0)
        return VK_EINVAL;
    if (d->din12 >= d->nbin || d->din12 == 0 || (d->din12 < 0 && d->din12 != -1)) return VK_EINVAL;
    for (int a = 0; a < d->nabs; a++)
        if (d->abs_sp[a] < 0 || d->abs_sp[a] >= plan->ni || d->abs_T[a] >= d->nT) return VK_EINVAL;
    for (int q = 0; q < d->nscat; q++)
        if (d->scat_sp[q] < 0 || d->scat_sp[q] >= plan->ni) return VK_EINVAL;
    for (int r = 0; r < d->nbranch; r++)
        if (d->br_col[r] < 0 || d->br_col[r] >= plan->nr || d->br_T[r] >= d->nTJ) return VK_EINVAL;
    vk_photo *h = new vk_photo();
    PhotoDev *p = &h->d;
    p->nbin = d->nbin; p->nabs = d->nabs; p->nscat = d->nscat; p->nbranch = d->nbranch;
    p->nT = d->nT; p->nTJ = d->nTJ; p->din12 = d->din12;
    p->dbin1 = d->dbin1; p->dbin2 = d->dbin2; p->cos_sl = d->cos_sl; p->edd = d->edd;
    p->f_diurnal = d->f_diurnal; p->flux_atol = d->flux_atol;
    p->ncols = cols->ncols; p->L = cols->L;
    const size_t nb = d->nbin, L = cols->L, lev = (size_t)(cols->L + cols->ncols);
    std::vector<double> hcb(nb);
    for (size_t b = 0; b < nb; b++) hcb[b] = d->hc / d->bins[b];   // hc/bins (op.py:2735)
    auto &v = h->allocs;
    int r = 0;
    r = r ? r : dup(v, &p->abs_sp, d->abs_sp, d->nabs);
    r = r ? r : dup(v, &p->abs_T, d->abs_T, d->nabs);
    r = r ? r : dup(v, &p->scat_sp, d->scat_sp, d->nscat);
    r = r ? r : dup(v, &p->br_col, d->br_col, d->nbranch);
    r = r ? r : dup(v, &p->br_T, d->br_T, d->nbranch);
    r = r ? r : dup(v, &p->bins, d->bins, nb);
    r = r ? r : dup(v, &p->hc_bin, (const double *)hcb.data(), nb);
    r = r ? r : dup(v, &p->sflux_top, d->sflux_top, nb);
    r = r ? r : dup(v, &p->cross, d->cross, (size_t)d->nabs * nb);
    r = r ? r : dup(v, &p->cross_T, d->cross_T, (size_t)d->nT * L * nb);
    r = r ? r : dup(v, &p->cross_scat, d->cross_scat, (size_t)d->nscat * nb);
    r = r ? r : dup(v, &p->cross_J, d->cross_J, (size_t)d->nbranch * nb);
    r = r ? r : dup(v, &p->cross_J_T, d->cross_J_T, (size_t)d->nTJ * L * nb);
    r = r ? r : dup<double>(v, &p->tau, nullptr, lev * nb);
    r = r ? r : dup<double>(v, &p->sflux, nullptr, lev * nb);
    r = r ? r : dup<double>(v, &p->dflux_u, nullptr, lev * nb);
    r = r ? r : dup<double>(v, &p->dflux_d, nullptr, lev * nb);
    r = r ? r : dup<double>(v, &p->w0, nullptr, L * nb);
    r = r ? r : dup<double>(v, &p->aflux, nullptr, L * nb);
    r = r ? r : dup<unsigned long long>(v, &p->change, nullptr, cols->ncols);
    r = r ? r : dup<int>(v, &p->due, nullptr, cols->ncols);
    r = r ? r : dup<int>(v, &p->switched, nullptr, cols->ncols);
    if (!r) {
        std::vector<int> last(cols->ncols, -1);
        r = dup(v, &p->last, (const int *)last.data(), cols->ncols);
    }
    if (r) { vk_photo_destroy(h); return r; }
    *out = h;
    return 0;
}

extern "C" int vk_photo_destroy(vk_photo *p) {
    if (!p) return 0;
    for (void *q : p->allocs) (void)hipFree(q);
    delete p;
    return 0;
}

// tau, fluxes and J for the columns whose update is due (every column with force)
int vk_launch_photo(vk_photo *ph, const vk_plan *plan, const vk_columns *cols, const double *y, const double *ymix,
                    const double *dz, double *k, vk_colstate *st, int force, int ini_frq, int final_frq,
                    double yconv_min, hipStream_t s) {
    const PhotoDev &d = ph->d;
    if (d.ncols != cols->ncols || d.L != cols->L) return VK_EINVAL;
    const int nc = cols->ncols;
    hipLaunchKernelGGL(k_photo_due, dim3((nc + 127) / 128), dim3(128), 0, s, nc, st, force, ini_frq, final_frq,
                       yconv_min, d.last, d.switched, d.due, d.change);
    if (!photo_per_bin(cols->max_nz, (long)d.nbin * nc)) {
        hipLaunchKernelGGL(k_photo_layers, dim3((d.nbin + PT - 1) / PT * ((cols->L + TAU_LAYERS - 1) / TAU_LAYERS)), dim3(PT),
                           0, s, d, plan->ni, cols->d_layer_col, y, ymix, dz);
        switch ((cols->max_nz + RT_LANES - 1) / RT_LANES) {
        case 1: case 2: case 3: launch_photo_rt<3>(d, cols, s); break;
        case 4: case 5: launch_photo_rt<5>(d, cols, s); break;
        case 6: case 7: launch_photo_rt<7>(d, cols, s); break;
        default: launch_photo_rt<RT_ROUNDS>(d, cols, s);
        }
    } else {
        const dim3 grid((d.nbin + PT - 1) / PT, nc);
        hipLaunchKernelGGL(k_photo_tau, grid, dim3(PT), 0, s, d, plan->ni, cols->d_off, y, ymix, dz);
        hipLaunchKernelGGL(k_photo_flux, grid, dim3(PT), 0, s, d, cols->d_off);
    }
    const int L = cols->L, ncu = std::max(1, vk_device_cus());
    auto rates = [&](auto kernel, int layers, int threads, int gy, bool stage) {
        hipLaunchKernelGGL(kernel, dim3((L + layers - 1) / layers, gy), dim3(threads),
                           stage ? sizeof(double) * layers * (size_t)d.nbin : 0, s, d, cols->d_layer_col, plan->nr, k);
    };
    // about two workgroups per CU, at least a branch per wave
    const int gy = std::max(1, std::min((d.nbranch + J_NT / 64 - 1) / (J_NT / 64), (2 * ncu + L - 1) / L));
    if (d.nbin < J_SMALL && L >= 8 * ncu)
        rates(k_photo_J<4, J_SMALL_NT>, 4, J_SMALL_NT, 1, true);
    else if (4 * d.nbin <= J_LDS && L >= 8 * ncu)
        rates(k_photo_J<4, J_NT>, 4, J_NT, 1, true);
    else if (2 * d.nbin <= J_LDS && L >= 4 * ncu)
        rates(k_photo_J<2, J_NT>, 2, J_NT, 1, true);
    else if (d.nbin <= J_LDS)
        rates(k_photo_J<1, J_NT>, 1, J_NT, gy, true);
    else
        rates(k_photo_J<1, J_NT, false>, 1, J_NT, gy, false);
    hipLaunchKernelGGL(k_photo_change, dim3((nc + 127) / 128), dim3(128), 0, s, nc, d.due, d.change, st);
    VK_CHECK(hipGetLastError());
    return 0;
}

extern "C" int vk_photo_update(vk_photo *p, const vk_plan *plan, const vk_columns *cols, const double *d_y,
                               const double *d_ymix, const double *d_dz, double *d_k, vk_colstate *d_st, int force,
                               int ini_frq, int final_frq, double yconv_min, void *stream) {
    if (!p || !plan || !cols || !d_y || !d_ymix || !d_dz || !d_k) return VK_EINVAL;
    if (!force && (!d_st || ini_frq < 1 || final_frq < 1)) return VK_EINVAL;
    // a limit of this entry alone: the kernels, and the integration's own refresh, take longer spectra
    if ((size_t)p->d.nbin * sizeof(double) > 64 * 1024) return VK_ETOOBIG;
    return vk_launch_photo(p, plan, cols, d_y, d_ymix, d_dz, d_k, d_st, force, ini_frq, final_frq, yconv_min,
                           (hipStream_t)stream);
}

extern "C" int vk_photo_read(const vk_photo *p, int what, double *h_out) {
    if (!p || !h_out) return VK_EINVAL;
    const PhotoDev &d = p->d;
    const size_t nb = d.nbin, lev = (size_t)(d.L + d.ncols) * nb, lay = (size_t)d.L * nb;
    const double *src = nullptr;
    size_t n = 0;
    switch (what) {
    case VK_PHOTO_TAU: src = d.tau; n = lev; break;
    case VK_PHOTO_SFLUX: src = d.sflux; n = lev; break;
    case VK_PHOTO_DFLUX_U: src = d.dflux_u; n = lev; break;
    case VK_PHOTO_DFLUX_D: src = d.dflux_d; n = lev; break;
    case VK_PHOTO_AFLUX: src = d.aflux; n = lay; break;
    default: return VK_EINVAL;
    }
    VK_CHECK(hipDeviceSynchronize());
    VK_CHECK(hipMemcpy(h_out, src, sizeof(double) * n, hipMemcpyDeviceToHost));
    return 0;
}
