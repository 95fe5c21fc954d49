// Block-Thomas factorisation and solves for the Ros2 left-hand side
//
//     lhs = blocktridiag(diag(Lsub_j), D_j, diag(Usup_j))
//
// The off-diagonal blocks are diagonal (diffusion couples a species only to
// itself in the neighbouring layers, op.py:2012-2040), so the Schur update
//     S_j = D_j - diag(Lsub_j) S_{j-1}^-1 diag(Usup_{j-1})
// is elementwise and the dense work is the inversion of each S_j (kernels
// in vk_factor_reg.hip, vk_factor_blk.hip, vk_factor_wave.hip; the block
// cyclic reduction alternative in vk_bcr.hip).  This file holds the solves,
// the residual of iterative refinement and the dispatch over variants.
//
// The chain over layers is split in two (twisted factorisation): one
// workgroup eliminates upwards from layer 0, another downwards from layer
// nz-1, and the meeting layer nz/2 is inverted last.  Same arithmetic as a
// single chain, half the dependence length; the solves are split the same
// way.
//
// The inverses go to Dinv, stored transposed (Dinv[l][m][i] = S_l^-1[i][m])
// so that the solve sweeps read them coalesced; D is left intact for the
// residuals of iterative refinement.
//
// Sweeps with explicit block inverses, like block elimination without
// pivoting across layers, are less accurate than LAPACK's band LU on
// ill-conditioned blocks (early steps from a far-from-equilibrium state);
// one refinement step with a residual computed in double-double arithmetic
// (k_residual) brings the solution to full FP64 accuracy.
#include <atomic>

#include "vk_blk.h"

namespace {

// D = A B for A[i][k] = i + 0.25 k + 1, B[k][j] = 1 - 0.5 k + 0.125 j (16 x 4 x 16)
// through one v_mfma_f64_16x16x4f64 with the operand layout the blocked
// inversion assumes; out[i*16+j] = D[i][j].
__global__ void k_selftest_mfma_f64(double *out) {
    const int l = threadIdx.x & 63;
    const double a = (double)(l & 15) + 0.25 * (double)(l >> 4) + 1.0;
    const double b = 1.0 - 0.5 * (double)(l >> 4) + 0.125 * (double)(l & 15);
    f64x4 acc = {0.0, 0.0, 0.0, 0.0};
    acc = __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, acc, 0, 0, 0);
#pragma unroll
    for (int r = 0; r < 4; r++) out[(4 * r + (l >> 4)) * 16 + (l & 15)] = acc[r];
}

__global__ void k_zero_int(int n, int *__restrict__ p) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0;
}

// ---------------------------------------------------------------------------
// Twisted block solves, one workgroup per chain.  Wave w owns rows
// [w CH, w CH + CH) of each transposed inverse and forms their share of every
// sum; a lane holds C neighbouring columns, one 8- to 24-byte load per row.
// After the step's one barrier G lanes add the W shares of each of the wave's
// own species, which is all the wave needs for its rows of the next step
// (handed out with readlane), and keep that species' couplings and
// right-hand side.
//
// Everything a step reads from memory is issued DEP steps ahead.  The loads
// stay in flight only because nothing waits for more than it needs: the loop
// is unrolled DEP times instead of moving buffers down (a move waits for the
// load), has no exit but its end and no access that a branch skips (the count
// of what is in flight stays known); rows past the block and steps past the
// end are buffer accesses out of range, which load zero and store nothing.
// 256 columns of 80 to 200 layers, 93 species: 675 -> 482 us a sweep (3.7 ->
// 5.1 TB/s; the kernel before moved its buffers down and so had one layer in
// flight); 80 columns of 100 to 150 layers, 150 species: 565 -> 465 us (160
// chains leave 96 CUs idle); one column of 60 layers, 30 species: 22 -> 18 us
// (0.45 us a step: barrier, LDS round trip and 70 instructions of one wave).
// Both sweeps stay within the column: layer indices run over [0, nz).
// ---------------------------------------------------------------------------
typedef double f64x2 __attribute__((ext_vector_type(2)));
typedef unsigned u32x2 __attribute__((ext_vector_type(2)));

// v plus the value of the lane that the DPP control CTRL pairs this one with
template <int CTRL>
__device__ __forceinline__ double add_pair(double v) {
    const u32x2 b = __builtin_bit_cast(u32x2, v);
    const u32x2 o = {(unsigned)__builtin_amdgcn_mov_dpp((int)b[0], CTRL, 0xf, 0xf, true),
                     (unsigned)__builtin_amdgcn_mov_dpp((int)b[1], CTRL, 0xf, 0xf, true)};
    return v + __builtin_bit_cast(double, o);
}

// W CH >= 16 NB rows, 64 C >= 16 NB columns; C <= 16 (NB - 1) + 1, so a
// lane's columns always fit in the block.  Eight waves at no more than 128
// registers put two chains on a CU (one of 16 waves with 3 layers in flight:
// 512 against 482 us below); from 97 species a layer's share takes 16 waves,
// and a CU holds one chain.  DEP steps' loads and stores stay
// below the 63 a wave can track.
template <int NB>
struct Sweep {
    static constexpr int C = NB <= 4 ? 1 : (NB <= 8 ? 2 : 3);
    static constexpr int W = NB == 1 ? 4 : (NB <= 6 ? 8 : 16);
    static constexpr int CH = 16 * NB / W;
    static constexpr int G = CH <= 4 ? W : (CH <= 8 ? 8 : 4);    // lanes per species: CH G <= 64
    static constexpr int DEP = NB <= 4 ? 4 : (NB <= 8 ? 2 : 1);
    static constexpr int NTH = 64 * W, MINW = NB <= 4 ? 2 : 4;
    static constexpr int RP = 64 * C + 8;                        // row pitch: G rows on different banks
    static_assert(W * CH == 16 * NB && 64 * C >= 16 * NB && C <= 16 * (NB - 1) + 1 && CH * G <= 64 && W % G == 0,
                  "sweep shape");
    typedef double Share[W][RP];

    int ni, w, cs, from, rr, own;
    int voff[CH];
    bool in;

    __device__ __forceinline__ Sweep(int n) {
        ni = n;
        const int lane = threadIdx.x & 63;
        w = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
        const int c0 = min(C * lane, ni - C);               // first column of the lane
        cs = C * lane < ni ? c0 : C * lane;                 // lanes past the block: columns that nobody reads
#pragma unroll
        for (int q = 0; q < CH; q++) voff[q] = ((w * CH + q) * ni + c0) * 8;
        const int q = lane / G, row = w * CH + q;           // species whose sum the lane helps to add
        in = q < CH && row < ni;
        rr = min(row, ni - 1) * 8;
        from = (lane % G) * RP + (rr >> 3);
        own = in && lane % G == 0 ? rr : 0x7ffffff0;        // out of any buffer: the store is dropped
    }

    // n doubles at p as a buffer, or nothing
    static __device__ __forceinline__ __amdgpu_buffer_rsrc_t buffer(const double *p, int n, bool on) {
        return __builtin_amdgcn_make_buffer_rsrc(const_cast<double *>(p), (short)0, on ? n * 8 : 0, 0x00020000);
    }
    // the lane's species from a layer's row of a (layer, species) array, and to it
    __device__ __forceinline__ double get(const double *p, bool on = true) const {
        return __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(buffer(p, ni, on), rr, 0, 0));
    }
    __device__ __forceinline__ void put(double *p, double x, bool on = true) const {
        __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2, x), buffer(p, ni, on), own, 0, 0);
    }

    // r[q][e] = Xt[w CH + q][c0 + e], zero for rows past the block
    __device__ __forceinline__ void load(double (&r)[CH][C], const double *Xt, bool on) const {
        const __amdgpu_buffer_rsrc_t rs = buffer(Xt, ni * ni, on);
#pragma unroll
        for (int q = 0; q < CH; q++) {
            if constexpr (C >= 2) {
                const f64x2 x = __builtin_bit_cast(f64x2, __builtin_amdgcn_raw_buffer_load_b128(rs, voff[q], 0, 0));
                r[q][0] = x[0];
                r[q][1] = x[1];
            }
            if constexpr (C != 2)
                r[q][C - 1] =
                    __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(rs, voff[q] + 8 * (C - 1), 0, 0));
        }
    }

    // the wave's share of the sums; v: the value of the lane's species
    __device__ __forceinline__ void product(const double (&r)[CH][C], double v, Share &share) const {
        double y[C] = {};
        v = in ? v : 0.0;
#pragma unroll
        for (int q = 0; q < CH; q++) {
            const double vq = lane_bcast(v, q * G);
#pragma unroll
            for (int e = 0; e < C; e++) y[e] = fma(r[q][e], vq, y[e]);
        }
#pragma unroll
        for (int e = 0; e < C; e++) share[w][cs + e] = y[e];
    }

    // the lane's species from all waves' shares, in two parts: what the lane
    // reads, and the sum over its group
    __device__ __forceinline__ void shares(double (&y)[W / G], const Share &share) const {
#pragma unroll
        for (int h = 0; h < W / G; h++) y[h] = (&share[0][0])[from + h * G * RP];
    }
    static __device__ __forceinline__ double total(const double (&p)[W / G]) {
        double y = p[0];
#pragma unroll
        for (int h = 1; h < W / G; h++) y += p[h];
        y = add_pair<0xB1>(y);                      // quad_perm 1 0 3 2
        y = add_pair<0x4E>(y);                      // quad_perm 2 3 0 1
        if (G == 8) y = add_pair<0x141>(y);         // row_half_mirror
        return y;
    }
};

template <int NB>
__global__ void __launch_bounds__(Sweep<NB>::NTH, Sweep<NB>::MINW)
    k_solve_fwd(int ni, const int *__restrict__ off, const int *__restrict__ order, const double *__restrict__ Dinv,
                const double *__restrict__ Lsub, const double *__restrict__ Usup, const double *in, double *tmp,
                const vk_colstate *__restrict__ st) {
    using W = Sweep<NB>;
    constexpr int DEP = W::DEP;
    const int chain = order ? order[blockIdx.x] : (int)blockIdx.x;   // 2c + side
    const int c = chain >> 1, side = chain & 1;
    if (st && st[c].done) return;
    const W sw(ni);
    const int l0 = off[c], nz = off[c + 1] - l0, m = nz / 2;
    __shared__ __align__(16) typename W::Share share[2];         // by step parity: one barrier a step
    const int j0 = side == 0 ? 0 : nz - 1, dj = side == 0 ? 1 : -1;
    const int nsteps = side == 0 ? m : nz - 1 - m;
    // where the next load and store lie; they end on the last layer
    const size_t first = (size_t)(l0 + j0);
    const double *pD = Dinv + first * ni * ni, *pi = in + first * ni, *pc = (side == 0 ? Lsub : Usup) + first * ni;
    double *pt = tmp + first * ni;
    double buf[DEP][W::CH][W::C], inb[DEP], cpb[DEP];
    auto load = [&](int d, int s) {
        const bool on = s < nsteps;
        const long go = s + 1 < nsteps ? dj * ni : 0;
        inb[d] = sw.get(pi, on);
        cpb[d] = sw.get(pc, on);
        sw.load(buf[d], pD, on);
        pi += go;
        pc += go;
        pD += go * ni;
    };
    double y[W::W / W::G];
    auto step = [&](int d, int s, double v) {
        sw.product(buf[d], v, share[s & 1]);
        __builtin_amdgcn_sched_barrier(0);        // the new loads into the registers just read
        load(d, s + DEP);
        __syncthreads();
        sw.shares(y, share[s & 1]);
    };
#pragma unroll
    for (int d = 0; d < DEP; d++) load(d, d);
    step(0, 0, inb[0]);
    // step s closes step s - 1; those past the end (up to a multiple of DEP)
    // load and store nothing
    for (int s0 = 1; s0 <= nsteps; s0 += DEP) {
#pragma unroll
        for (int e = 0; e < DEP; e++) {
            const int s = s0 + e, d = (1 + e) % DEP;
            const double z = sw.total(y);
            sw.put(pt, z, s <= nsteps);
            pt += s < nsteps ? dj * ni : 0;
            step(d, s, inb[d] - cpb[d] * z);
        }
    }
    // park b_m in the unused slot m so the backward kernel never reads `in`
    // (which may alias `out`)
    if (side == 0) sw.put(tmp + ((size_t)l0 + m) * ni, sw.get(in + ((size_t)l0 + m) * ni));
}

template <int NB, bool ACC>
__global__ void __launch_bounds__(Sweep<NB>::NTH, Sweep<NB>::MINW)
    k_solve_bwd(int ni, const int *__restrict__ off, const int *__restrict__ order, const double *__restrict__ Dinv,
                const double *__restrict__ Lsub, const double *__restrict__ Usup, const double *tmp, double *out,
                const vk_colstate *__restrict__ st, double *acc) {
    using W = Sweep<NB>;
    constexpr int DEP = W::DEP;
    const int chain = order ? order[blockIdx.x] : (int)blockIdx.x;   // 2c + side
    const int c = chain >> 1, side = chain & 1;
    if (st && st[c].done) return;
    const W sw(ni);
    const int l0 = off[c], nz = off[c + 1] - l0, m = nz / 2;
    const size_t lm = ((size_t)l0 + m) * ni;
    __shared__ __align__(16) typename W::Share share[2];
    const int dj = side == 0 ? -1 : 1;
    const int nsteps = 1 + (side == 0 ? m : nz - 1 - m);     // the middle layer, then the chain outwards
    const double *pD = Dinv + lm * ni, *pc = (side == 0 ? Usup : Lsub) + lm, *pt = tmp + lm;
    const double *pa = acc + (ACC ? lm : 0);
    double *po = out + lm, *pao = acc + (ACC ? lm : 0);
    double buf[DEP][W::CH][W::C], cpb[DEP], tb[DEP], ab[DEP];
    auto load = [&](int d, int s) {
        const bool on = s < nsteps;
        const long go = s + 1 < nsteps ? dj * ni : 0;
        cpb[d] = sw.get(pc, on);
        sw.load(buf[d], pD, on);
        pc += go;
        pD += go * ni;
    };
    // what the end of step s needs, which falls into step s + 1
    auto load_end = [&](int d, int s) {
        const bool on = s < nsteps;
        const long go = s + 1 < nsteps ? dj * ni : 0;
        tb[d] = sw.get(pt, on);
        pt += go;
        if (ACC) {
            ab[d] = sw.get(pa, on);
            pa += go;
        }
    };
    double y[W::W / W::G];
    auto step = [&](int d, int s, double v) {
        sw.product(buf[d], v, share[s & 1]);
        __builtin_amdgcn_sched_barrier(0);
        load(d, s + DEP);
        __syncthreads();
        sw.shares(y, share[s & 1]);
    };
    // the solution of step s from its shares; the middle layer (the shares'
    // sum itself) is stored by one side
    auto finish = [&](int d, int s) {
        const double z = sw.total(y), x = s == 0 ? z : tb[d] - z;
        const bool on = s >= side && s < nsteps;
        const long go = s + 1 < nsteps ? dj * ni : 0;
        sw.put(po, x, on);
        po += go;
        if (ACC) {
            sw.put(pao, ab[d] + x, on);
            pao += go;
        }
        return x;
    };
#pragma unroll
    for (int d = 0; d < DEP; d++) {
        load(d, d);
        load_end(d, d);
    }
    // x_m = M^-1 (b_m - Lsub_m z_{m-1} - Usup_m w_{m+1}); both sides compute it
    double v = tb[0];
    if (m > 0) v = v - sw.get(Lsub + lm) * sw.get(tmp + lm - ni);
    if (m < nz - 1) v = v - sw.get(Usup + lm) * sw.get(tmp + lm + ni);
    step(0, 0, v);
    for (int s0 = 1; s0 <= nsteps; s0 += DEP) {
#pragma unroll
        for (int e = 0; e < DEP; e++) {
            const double x = finish(e, s0 + e - 1);
            load_end(e, s0 + e - 1 + DEP);
            step((1 + e) % DEP, s0 + e, cpb[(1 + e) % DEP] * x);
        }
    }
}

// r = b - A x with A = blocktridiag(diag(Lsub), D, diag(Usup)), accumulated
// in double-double (exact products via fma, error-free sums), one
// workgroup per layer, one thread per row
__device__ inline void dd_sub_prod(double &hi, double &lo, double a, double b) {
    const double p = a * b;
    const double pe = fma(a, b, -p);          // a*b = p + pe exactly
    const double s = hi - p;
    const double bb = s - hi;
    const double se = (hi - (s - bb)) + (-p - bb);   // hi - p = s + se exactly
    hi = s;
    lo = lo + (se - pe);
}

// r = b - A x, 32 rows of one layer per workgroup: 8 threads share a row,
// each a double-double partial over every eighth column (read straight into
// registers: every load is issued before the first product), and the
// partials, b and the two coupling terms are combined in double-double.  The
// eight threads of a row read 64 contiguous bytes at a time: with an eighth of
// the columns in one run each, every 8-byte load was an access of the vector
// cache by itself, at one a cycle 0.5 of the 0.62 ms that 36 000 layers of 93
// species took, now 0.53 (4.7 TB/s).
constexpr int RES_ROWS = 32, RES_PARTS = NT / RES_ROWS;

__device__ inline void dd_add(double &hi, double &lo, double a_hi, double a_lo) {
    const double s = hi + a_hi;
    const double bb = s - hi;
    const double e = (hi - (s - bb)) + (a_hi - bb);     // hi + a_hi = s + e exactly
    hi = s;
    lo = lo + (e + a_lo);
}

// CH: the columns of a thread, 16 NB / RES_PARTS for blocks of up to 16 NB rows
template <int CH>
__global__ void __launch_bounds__(NT) k_residual(int ni, const int *__restrict__ off,
                                                  const int *__restrict__ layer_col, const double *__restrict__ D,
                                                  const double *__restrict__ Lsub, const double *__restrict__ Usup,
                                                  const double *__restrict__ x, const double *__restrict__ b,
                                                  double *__restrict__ r, const vk_colstate *__restrict__ st) {
    extern __shared__ double rsm[];
    double *xs = rsm;                        // ni
    double *ph = xs + ni;                    // RES_ROWS x RES_PARTS partial sums (hi)
    double *pl = ph + NT;                    // (lo)
    const int l = blockIdx.x;
    const int c = layer_col[l];
    if (st && st[c].done) return;
    const int j = l - off[c], nz = off[c + 1] - off[c];
    const int i0 = blockIdx.y * RES_ROWS;
    const int nrows = min(RES_ROWS, ni - i0);
    const double *Dl = D + ((size_t)l * ni + i0) * ni;
    const int tid = threadIdx.x;
    const int rr = tid / RES_PARTS, pp = tid % RES_PARTS;
    // this thread's columns of its row (indices clamped into the row; entries
    // past it are loaded but not used)
    double dr[CH];
    const double *row = Dl + (size_t)min(rr, nrows - 1) * ni;
#pragma unroll
    for (int k = 0; k < CH; k++) dr[k] = row[min(RES_PARTS * k + pp, ni - 1)];
    for (int m = tid; m < ni; m += NT) xs[m] = x[(size_t)l * ni + m];
    __syncthreads();
    double hi = 0.0, lo = 0.0;
    if (rr < nrows) {
#pragma unroll
        for (int k = 0; k < CH; k++)
            if (RES_PARTS * k + pp < ni) dd_sub_prod(hi, lo, dr[k], xs[RES_PARTS * k + pp]);
    }
    ph[tid] = hi;
    pl[tid] = lo;
    __syncthreads();
    if (pp == 0 && rr < nrows) {
        const int i = i0 + rr;
        double h = b[(size_t)l * ni + i], o = 0.0;
        for (int q = 0; q < RES_PARTS; q++) dd_add(h, o, ph[tid + q], pl[tid + q]);
        if (j > 0) dd_sub_prod(h, o, Lsub[(size_t)l * ni + i], x[(size_t)(l - 1) * ni + i]);
        if (j < nz - 1) dd_sub_prod(h, o, Usup[(size_t)l * ni + i], x[(size_t)(l + 1) * ni + i]);
        r[(size_t)l * ni + i] = h + o;
    }
}


}  // namespace


// info_zeroed: the caller has cleared info in an earlier launch on s
int vk_launch_factor(const vk_plan *plan, const vk_columns *cols, const double *D, const double *Lsub,
                     const double *Usup, double *Dinv, int *info, const vk_colstate *st, const vk_bcr_ws *ws,
                     hipStream_t s, bool info_zeroed = false) {
    const int ni = plan->ni;
    const int n = (ni + 15) / 16;
    const int nc = cols->ncols;
    const int v = plan->factor_variant;
    if (n < 1 || n > 10) return VK_ETOOBIG;
    if (info && !info_zeroed) hipLaunchKernelGGL(k_zero_int, dim3((nc + 255) / 256), dim3(256), 0, s, nc, info);
    int r;
    switch (v) {
    case VK_FACTOR_BCR:
        if (!ws || !ws->A) return VK_EINVAL;
        return vk_launch_bcr_factor(n, ni, cols, D, Lsub, Usup, Dinv, info, st, ws, s);
    case VK_FACTOR_BLOCKED:
        r = vk_launch_factor_blocked1(n, ni, nc, cols->d_off, cols->d_chain_order[0], D, Lsub, Usup, Dinv, info, st, s);
        break;
    case VK_FACTOR_BLOCKED_OCC2:
        r = vk_launch_factor_blocked2(n, ni, nc, cols->d_off, cols->d_chain_order[1], D, Lsub, Usup, Dinv, info, st, s);
        break;
    case VK_FACTOR_WAVE:
        if (n <= 7) {
            r = vk_launch_factor_wave(n, ni, nc, cols->d_off, D, Lsub, Usup, Dinv, info, st, s);
            break;
        }
        // fall through: the two-wave kernel holds at most 112 species
    default:
        r = vk_launch_factor_register(n, ni, nc, cols->d_off, D, Lsub, Usup, Dinv, info, st, s);
    }
    if (r) return r;
    VK_CHECK(hipGetLastError());
    return 0;
}

// out = lhs^-1 in (tmp: L*ni scratch, may not alias in/out; in may alias out)
namespace {
// order: the chain each workgroup runs (the pairing of the two-per-CU
// factorisation: long chains share a CU with short ones)
template <int NB>
void launch_solve_n(int ni, int ncols, const int *off, const int *order, const double *Dinv, const double *Lsub,
                    const double *Usup, const double *in, double *out, double *tmp, const vk_colstate *st, double *acc,
                    hipStream_t s) {
    const dim3 grid(2 * ncols), block(Sweep<NB>::NTH);
    hipLaunchKernelGGL((k_solve_fwd<NB>), grid, block, 0, s, ni, off, order, Dinv, Lsub, Usup, in, tmp, st);
    if (acc)
        hipLaunchKernelGGL((k_solve_bwd<NB, true>), grid, block, 0, s, ni, off, order, Dinv, Lsub, Usup, tmp, out, st, acc);
    else
        hipLaunchKernelGGL((k_solve_bwd<NB, false>), grid, block, 0, s, ni, off, order, Dinv, Lsub, Usup, tmp, out, st, acc);
}

}  // namespace

// acc (nullable): also add the solution into acc, row by row as it is written
int vk_launch_solve(const vk_plan *plan, const vk_columns *cols, const double *Dinv, const double *Lsub,
                    const double *Usup, const double *in, double *out, double *tmp, const vk_colstate *st,
                    const vk_bcr_ws *ws, hipStream_t s, double *acc = nullptr) {
    const int ni = plan->ni, nc = cols->ncols;
    const int *off = cols->d_off;
    if (plan->factor_variant == VK_FACTOR_BCR) {
        if (!ws || !ws->A) return VK_EINVAL;
        return vk_launch_bcr_solve(ni, cols, Dinv, Lsub, Usup, in, out, tmp, st, ws, acc, s);
    }
    switch ((ni + 15) / 16) {
    case 1: launch_solve_n<1>(ni, nc, off, cols->d_chain_order[1], Dinv, Lsub, Usup, in, out, tmp, st, acc, s); break;
    case 2: launch_solve_n<2>(ni, nc, off, cols->d_chain_order[1], Dinv, Lsub, Usup, in, out, tmp, st, acc, s); break;
    case 3: launch_solve_n<3>(ni, nc, off, cols->d_chain_order[1], Dinv, Lsub, Usup, in, out, tmp, st, acc, s); break;
    case 4: launch_solve_n<4>(ni, nc, off, cols->d_chain_order[1], Dinv, Lsub, Usup, in, out, tmp, st, acc, s); break;
    case 5: launch_solve_n<5>(ni, nc, off, cols->d_chain_order[1], Dinv, Lsub, Usup, in, out, tmp, st, acc, s); break;
    case 6: launch_solve_n<6>(ni, nc, off, cols->d_chain_order[1], Dinv, Lsub, Usup, in, out, tmp, st, acc, s); break;
    case 7: launch_solve_n<7>(ni, nc, off, cols->d_chain_order[1], Dinv, Lsub, Usup, in, out, tmp, st, acc, s); break;
    case 8: launch_solve_n<8>(ni, nc, off, cols->d_chain_order[1], Dinv, Lsub, Usup, in, out, tmp, st, acc, s); break;
    case 9: launch_solve_n<9>(ni, nc, off, cols->d_chain_order[1], Dinv, Lsub, Usup, in, out, tmp, st, acc, s); break;
    case 10: launch_solve_n<10>(ni, nc, off, cols->d_chain_order[1], Dinv, Lsub, Usup, in, out, tmp, st, acc, s); break;
    default: return VK_ETOOBIG;
    }
    VK_CHECK(hipGetLastError());
    return 0;
}

int vk_launch_residual(const vk_plan *plan, const vk_columns *cols, const double *D, const double *Lsub,
                       const double *Usup, const double *x, const double *b, double *r, const vk_colstate *st,
                       hipStream_t s) {
    const int ni = plan->ni;
    const size_t smem = sizeof(double) * ((size_t)ni + 2 * NT);
    const dim3 grid(cols->L, (ni + RES_ROWS - 1) / RES_ROWS);
    // runs of ceil(ni / RES_PARTS) <= ceil(16 nb / RES_PARTS) entries
    switch ((ni + 15) / 16) {
#define VK_RES(NB)                                                                                                   \
    case NB:                                                                                                         \
        hipLaunchKernelGGL(k_residual<(16 * NB + RES_PARTS - 1) / RES_PARTS>, grid, dim3(NT), smem, s, ni, cols->d_off, \
                           cols->d_layer_col, D, Lsub, Usup, x, b, r, st);                                           \
        break;
        VK_RES(1) VK_RES(2) VK_RES(3) VK_RES(4) VK_RES(5) VK_RES(6) VK_RES(7) VK_RES(8) VK_RES(9) VK_RES(10)
#undef VK_RES
    default: return VK_ETOOBIG;
    }
    VK_CHECK(hipGetLastError());
    return 0;
}

// x = A^-1 b with `refine` steps of iterative refinement (work, tmp: L*ni scratch each)
int vk_launch_solve_refined(const vk_plan *plan, const vk_columns *cols, const double *D, const double *Dinv,
                            const double *Lsub, const double *Usup, const double *b, double *x, double *work,
                            double *tmp, int refine, const vk_colstate *st, const vk_bcr_ws *ws, hipStream_t s) {
    int r = vk_launch_solve(plan, cols, Dinv, Lsub, Usup, b, x, tmp, st, ws, s);
    if (r) return r;
    for (int q = 0; q < refine; q++) {
        r = vk_launch_residual(plan, cols, D, Lsub, Usup, x, b, work, st, s);
        if (r) return r;
        // the correction is added into x by the solve's backward sweep
        r = vk_launch_solve(plan, cols, Dinv, Lsub, Usup, work, work, tmp, st, ws, s, x);
        if (r) return r;
    }
    return 0;
}

// stream-ordered workspace of the cyclic reduction (freed with the object)
struct BcrTmp {
    vk_bcr_ws ws;
    hipStream_t s;
    explicit BcrTmp(hipStream_t st) : s(st) {}
    int alloc(const vk_plan *plan, const vk_columns *cols) {
        const size_t nn = (size_t)plan->ni * plan->ni, L = (size_t)cols->L, ns = (size_t)cols->bcr.nsurv + 1;
        if (hipMallocAsync((void **)&ws.A, sizeof(double) * L * nn, s) != hipSuccess ||
            hipMallocAsync((void **)&ws.B, sizeof(double) * L * nn, s) != hipSuccess ||
            hipMallocAsync((void **)&ws.C, sizeof(double) * L * nn, s) != hipSuccess ||
            hipMallocAsync((void **)&ws.P, sizeof(double) * ns * nn, s) != hipSuccess ||
            hipMallocAsync((void **)&ws.Q, sizeof(double) * ns * nn, s) != hipSuccess ||
            hipMallocAsync((void **)&ws.XB, sizeof(double) * L * nn, s) != hipSuccess ||
            hipMallocAsync((void **)&ws.XC, sizeof(double) * L * nn, s) != hipSuccess)
            return VK_ENOMEM;
        return 0;
    }
    ~BcrTmp() {
        for (double *p : {ws.A, ws.B, ws.C, ws.P, ws.Q, ws.XB, ws.XC})
            if (p) (void)hipFreeAsync(p, s);
    }
};

extern "C" int vk_block_solve_system(const vk_plan *plan, const vk_columns *cols, const double *d_D,
                                     const double *d_Lsub, const double *d_Usup, const double *d_b, double *d_x,
                                     int refine, int *d_info, void *stream) {
    if (!plan || !cols || !d_D || !d_Lsub || !d_Usup || !d_b || !d_x || refine < 0 || d_b == d_x) return VK_EINVAL;
    hipStream_t s = (hipStream_t)stream;
    const size_t nn = (size_t)plan->ni * plan->ni, L = (size_t)cols->L;
    double *Dinv = nullptr, *work = nullptr, *tmp = nullptr;
    BcrTmp bt(s);
    int r = 0;
    if (hipMallocAsync((void **)&Dinv, sizeof(double) * L * nn, s) != hipSuccess ||
        hipMallocAsync((void **)&work, sizeof(double) * L * plan->ni, s) != hipSuccess ||
        hipMallocAsync((void **)&tmp, sizeof(double) * L * plan->ni, s) != hipSuccess)
        r = VK_ENOMEM;
    if (!r && plan->factor_variant == VK_FACTOR_BCR) r = bt.alloc(plan, cols);
    if (!r) r = vk_launch_factor(plan, cols, d_D, d_Lsub, d_Usup, Dinv, d_info, nullptr, &bt.ws, s);
    if (!r)
        r = vk_launch_solve_refined(plan, cols, d_D, Dinv, d_Lsub, d_Usup, d_b, d_x, work, tmp, refine, nullptr,
                                    &bt.ws, s);
    for (double *p : {Dinv, work, tmp})
        if (p) (void)hipFreeAsync(p, s);
    return r;
}

// Workspace of vk_block_solve_system_noalloc: one static array per device
// (each device holds its own copy until the process ends).  Host code never
// uses the array's name as an address: scratch_base() resolves it once per
// device with hipGetSymbolAddress, and only that pointer reaches kernels.
static __device__ __align__(256) double scratch[VK_NOALLOC_SCRATCH_BYTES / sizeof(double)];

static int scratch_base(double **out) {
    static std::atomic<double *> base[64];   // per device, zero-initialised
    int dev = 0;
    VK_CHECK(hipGetDevice(&dev));
    if (dev < 0 || dev >= 64) return VK_EINVAL;
    double *p = base[dev].load(std::memory_order_acquire);
    if (!p) {
        void *q = nullptr;
        VK_CHECK(hipGetSymbolAddress(&q, HIP_SYMBOL(scratch)));
        if (!q) return VK_ENOMEM;
        p = static_cast<double *>(q);
        base[dev].store(p, std::memory_order_release);
    }
    *out = p;
    return 0;
}

extern "C" int vk_block_solve_system_noalloc(const vk_plan *plan, const vk_columns *cols, const double *d_D,
                                             const double *d_Lsub, const double *d_Usup, const double *d_b,
                                             double *d_x, int refine, int *d_info, void *stream) {
    if (!plan || !cols || !d_D || !d_Lsub || !d_Usup || !d_b || !d_x || refine < 0 || d_b == d_x) return VK_EINVAL;
    hipStream_t s = (hipStream_t)stream;
    // carve the workspace of vk_block_solve_system out of the scratch, each
    // piece on a 256-byte boundary (32 doubles)
    const size_t nn = (size_t)plan->ni * plan->ni, L = (size_t)cols->L, ns = (size_t)cols->bcr.nsurv + 1;
    const bool bcr = plan->factor_variant == VK_FACTOR_BCR;
    auto up = [](size_t n) { return (n + 31) & ~(size_t)31; };
    const size_t sizes[10] = {L * nn, L * plan->ni, L * plan->ni,
                              bcr ? L * nn : 0, bcr ? L * nn : 0, bcr ? L * nn : 0, bcr ? ns * nn : 0,
                              bcr ? ns * nn : 0, bcr ? L * nn : 0, bcr ? L * nn : 0};
    size_t need = 0;
    for (size_t n : sizes) need += up(n);
    if (need > VK_NOALLOC_SCRATCH_BYTES / sizeof(double)) return VK_ETOOBIG;
    double *base = nullptr;
    int r = scratch_base(&base);
    if (r) return r;
    double *piece[10];
    size_t at = 0;
    for (int q = 0; q < 10; q++) {
        piece[q] = sizes[q] ? base + at : nullptr;
        at += up(sizes[q]);
    }
    vk_bcr_ws ws;
    ws.A = piece[3]; ws.B = piece[4]; ws.C = piece[5]; ws.P = piece[6]; ws.Q = piece[7];
    ws.XB = piece[8]; ws.XC = piece[9];
    r = vk_launch_factor(plan, cols, d_D, d_Lsub, d_Usup, piece[0], d_info, nullptr, &ws, s);
    if (!r)
        r = vk_launch_solve_refined(plan, cols, d_D, piece[0], d_Lsub, d_Usup, d_b, d_x, piece[1], piece[2], refine,
                                    nullptr, &ws, s);
    return r;
}

extern "C" int vk_block_factor(const vk_plan *plan, const vk_columns *cols, const double *d_D,
                               const double *d_Lsub, const double *d_Usup, double *d_Dinv, int *d_info,
                               void *stream) {
    if (!plan || !cols || !d_D || !d_Lsub || !d_Usup || !d_Dinv || d_D == d_Dinv) return VK_EINVAL;
    if (plan->factor_variant == VK_FACTOR_BCR) return VK_EINVAL;
    return vk_launch_factor(plan, cols, d_D, d_Lsub, d_Usup, d_Dinv, d_info, nullptr, nullptr, (hipStream_t)stream);
}

extern "C" int vk_block_solve(const vk_plan *plan, const vk_columns *cols, const double *d_Dinv,
                              const double *d_Lsub, const double *d_Usup, double *d_rhs, void *stream) {
    if (!plan || !cols || !d_Dinv || !d_Lsub || !d_Usup || !d_rhs) return VK_EINVAL;
    if (plan->factor_variant == VK_FACTOR_BCR) return VK_EINVAL;
    hipStream_t s = (hipStream_t)stream;
    double *tmp = nullptr;
    VK_CHECK(hipMallocAsync((void **)&tmp, sizeof(double) * (size_t)cols->L * plan->ni, s));
    int r = vk_launch_solve(plan, cols, d_Dinv, d_Lsub, d_Usup, d_rhs, d_rhs, tmp, nullptr, nullptr, s);
    VK_CHECK(hipFreeAsync(tmp, s));
    return r;
}

extern "C" int vk_block_residual(const vk_plan *plan, const vk_columns *cols, const double *d_D,
                                 const double *d_Lsub, const double *d_Usup, const double *d_x, const double *d_b,
                                 double *d_r, void *stream) {
    if (!plan || !cols || !d_D || !d_Lsub || !d_Usup || !d_x || !d_b || !d_r) return VK_EINVAL;
    return vk_launch_residual(plan, cols, d_D, d_Lsub, d_Usup, d_x, d_b, d_r, nullptr, (hipStream_t)stream);
}

namespace {
// a well-conditioned block system of the columns' shape for timing
__global__ void k_fill_tune(int ni, long n_d, double *__restrict__ D, long n_c, double *__restrict__ Lsub,
                            double *__restrict__ Usup) {
    const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (t < n_d) {
        const long e = t % ((long)ni * ni);
        const int i = (int)(e / ni), j = (int)(e % ni);
        D[t] = (i == j) ? 2.0 * ni : 1.0 / (1.0 + i + 2.0 * j);
    }
    if (t < n_c) {
        Lsub[t] = -0.25;
        Usup[t] = -0.5;
    }
}
}  // namespace

static bool variant_ok(const vk_plan *plan, int v) {
    return v >= 0 && v < VK_FACTOR_NVARIANTS && (v != VK_FACTOR_WAVE || plan->ni <= 112);
}

// cyclic reduction pays off while the columns leave most of the device idle
static constexpr int BCR_TUNE_MAX_COLS = 64;

extern "C" int vk_plan_set_factor_variant(vk_plan *plan, int variant) {
    if (!plan || !variant_ok(plan, variant)) return VK_EINVAL;
    plan->factor_variant = variant;
    return 0;
}

extern "C" int vk_plan_factor_variant(const vk_plan *plan) { return plan ? plan->factor_variant : VK_EINVAL; }

extern "C" int vk_tune_factor(vk_plan *plan, const vk_columns *cols, int reps, float *ms, void *stream) {
    if (!plan || !cols || reps < 1 || !ms) return VK_EINVAL;
    hipStream_t s = (hipStream_t)stream;
    const size_t nn = (size_t)plan->ni * plan->ni, L = (size_t)cols->L;
    const bool try_bcr = cols->ncols <= BCR_TUNE_MAX_COLS;
    double *D = nullptr, *Dinv = nullptr, *Lsub = nullptr, *Usup = nullptr, *x = nullptr, *tmp = nullptr;
    hipEvent_t e0 = nullptr, e1 = nullptr;
    BcrTmp bt(s);
    int rc = 0;
    if (hipMallocAsync((void **)&D, sizeof(double) * L * nn, s) != hipSuccess ||
        hipMallocAsync((void **)&Dinv, sizeof(double) * L * nn, s) != hipSuccess ||
        hipMallocAsync((void **)&Lsub, sizeof(double) * L * plan->ni, s) != hipSuccess ||
        hipMallocAsync((void **)&Usup, sizeof(double) * L * plan->ni, s) != hipSuccess ||
        hipMallocAsync((void **)&x, sizeof(double) * L * plan->ni, s) != hipSuccess ||
        hipMallocAsync((void **)&tmp, sizeof(double) * L * plan->ni, s) != hipSuccess ||
        hipEventCreate(&e0) != hipSuccess || hipEventCreate(&e1) != hipSuccess ||
        (try_bcr && bt.alloc(plan, cols))) {
        rc = VK_ENOMEM;
    } else {
        const long nd = (long)(L * nn);
        hipLaunchKernelGGL(k_fill_tune, dim3((unsigned)((nd + 255) / 256)), dim3(256), 0, s, plan->ni, nd, D,
                           (long)(L * plan->ni), Lsub, Usup);
        const int keep = plan->factor_variant;
        int bestv = keep;
        float bestms = 0.f;
        bool have = false;
        // one repetition: a factorisation and the two solves of an attempt
        auto rep = [&]() -> int {
            int r = vk_launch_factor(plan, cols, D, Lsub, Usup, Dinv, nullptr, nullptr, &bt.ws, s);
            for (int q = 0; q < 2 && !r; q++) r = vk_launch_solve(plan, cols, Dinv, Lsub, Usup, Lsub, x, tmp, nullptr,
                                                                  &bt.ws, s);
            return r;
        };
        for (int v = 0; v < VK_FACTOR_NVARIANTS && rc == 0; v++) {
            ms[v] = -1.0f;
            if (!variant_ok(plan, v) || (v == VK_FACTOR_BCR && !try_bcr)) continue;
            plan->factor_variant = v;
            rc = rep();   // warm-up
            if (rc) break;
            hipError_t e = hipEventRecord(e0, s);
            if (e != hipSuccess) { rc = -(int)e; break; }
            for (int q = 0; q < reps && rc == 0; q++) rc = rep();
            if (rc) break;
            e = hipEventRecord(e1, s);
            if (e == hipSuccess) e = hipEventSynchronize(e1);
            float t = 0.f;
            if (e == hipSuccess) e = hipEventElapsedTime(&t, e0, e1);
            if (e != hipSuccess) { rc = -(int)e; break; }
            ms[v] = t / reps;
            if (!have || ms[v] < bestms) { bestms = ms[v]; bestv = v; have = true; }
        }
        plan->factor_variant = rc ? keep : bestv;
    }
    for (double *p : {D, Dinv, Lsub, Usup, x, tmp})
        if (p) (void)hipFreeAsync(p, s);
    if (e0) (void)hipEventDestroy(e0);
    if (e1) (void)hipEventDestroy(e1);
    return rc;
}

namespace {
__global__ void k_selftest_wave_max(const unsigned *in, unsigned *out) {
    out[threadIdx.x] = wave_max_u32(in[threadIdx.x]);
}
__global__ void k_selftest_recip(int n, const double *in, double *out) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) out[i] = blk_recip(in[i]);
}
}  // namespace

extern "C" int vk_selftest_recip_f64(int n, const double *d_in, double *d_out, void *stream) {
    if (n < 0 || (n > 0 && (!d_in || !d_out))) return VK_EINVAL;
    if (n == 0) return 0;
    hipLaunchKernelGGL(k_selftest_recip, dim3((n + 255) / 256), dim3(256), 0, (hipStream_t)stream, n, d_in, d_out);
    VK_CHECK(hipGetLastError());
    return 0;
}

extern "C" int vk_selftest_wave_max_u32(const unsigned *d_in, unsigned *d_out, void *stream) {
    if (!d_in || !d_out) return VK_EINVAL;
    hipLaunchKernelGGL(k_selftest_wave_max, dim3(1), dim3(64), 0, (hipStream_t)stream, d_in, d_out);
    VK_CHECK(hipGetLastError());
    return 0;
}

extern "C" int vk_selftest_mfma_f64(double *d_out, void *stream) {
    if (!d_out) return VK_EINVAL;
    hipLaunchKernelGGL(k_selftest_mfma_f64, dim3(1), dim3(64), 0, (hipStream_t)stream, d_out);
    VK_CHECK(hipGetLastError());
    return 0;
}
