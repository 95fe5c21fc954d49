// Block cyclic reduction factorisation and solves (factor variant 4).
#include <algorithm>

#include "vk_blk.h"

namespace {

// ---------------------------------------------------------------------------
// Block cyclic reduction (factor variant 4)
//
// Every level eliminates every other active layer of each column at once
// (the even positions of an odd count, the odd ones of an even count, so
// that floor(n/2) layers survive): their blocks are inverted in parallel, with
// the diagonal as pivots (blk_invert_diag) or, where a block refuses it, searched
// ones (blk_invert), and each surviving layer j with eliminated neighbours l
// (left) and r (right) takes
//     P_j = B_j A_l^-1,   Q_j = C_j A_r^-1,
//     A_j -= P_j C_l + Q_j B_r,   B_j = -P_j B_l,   C_j = -Q_j C_r
// (B: coupling to the previous active layer, C: to the next; diagonal at
// level 0, dense above).  The chain over layers becomes floor(log2 nz)
// levels of independent work and one inversion on top: the Schur-complement
// updates above level 0 are dense n x n products on FP64 MFMA, level 0 is
// elementwise.  P and Q are kept for the right-hand side reduction of the solves.
//
// Storage: A row-major (the survivors' Schur complements, formed from D by
// the level-0 update; level 0 inverts from D itself); P, Q, B, C
// transposed (Pt[b][a] = P[a][b]), so that the solve sweeps, one thread per
// row a, read them coalesced; inverses transposed as in the chain variants.
// ---------------------------------------------------------------------------

// How a column's blocks below level 0 are inverted.  A block that refuses the
// diagonal has paid for the attempt, and the slowest block is a level's time.  So
// where a good part of a column's level-0 blocks refused, its later ones search
// their pivots at once.  The decision rests on level 0 alone, so it does not depend
// on the order in which blocks run, and it takes no memory: a layer eliminated at
// level 0 leaves its block of the workspace's A unused, which notes the refusal,
// and the layers that survive level 0 find the decision as a mark in the output
// they will write.  One column, factorisation and a solve, every block refusing
// at its last pivots: 93 species 805 -> 641 us (605 with pivots searched
// throughout, 396 where all are kept), 112 species 1068 -> 802 (747, 582); every
// third block refusing half way 671 -> 627, 1012 -> 807.
constexpr int BCR_SEARCH_PART = 8;      // one in so many

// invert A[layer] for the listed layers (the eliminated ones of a level, or
// the top layer of each column) into Dinv[layer] (transposed storage); W0: the
// workspace's A at level 0
template <int NB, int SEARCH, int MINW>
__global__ void __launch_bounds__(blk_nt(NB), blk_nt(NB) > NT ? 1 : MINW) k_bcr_invert(
    int ni, int n, const int4 *__restrict__ el, const int2 *__restrict__ top, const int *__restrict__ off,
    const double *__restrict__ A, double *__restrict__ W0, double *__restrict__ Dinv, int *__restrict__ info,
    const vk_colstate *__restrict__ st) {
    const int q = blockIdx.x;
    if (q >= n) return;
    const int layer = el ? el[q].x : top[q].x, c = el ? el[q].w : top[q].y;
    const size_t nn = (size_t)ni * ni;
    // asked for beside the column's state
    const bool marked = (SEARCH == BLK_SEARCH_ONLY || !W0) && blk_marked(Dinv + layer * nn);
    if (st && st[c].done) return;
    if (SEARCH == BLK_SEARCH_ONLY && !marked) return;
    __shared__ BlkShared<NB> sh;
    if (threadIdx.x == 0) sh.info = 0;
    const bool kept = blk_invert_schur<NB, SEARCH>(ni, A + layer * nn, nullptr, nullptr, nullptr, nullptr, nullptr,
                                                   nullptr, Dinv + layer * nn, sh, layer - off[c] + 1, marked);
    if (threadIdx.x == 0) {
        if (SEARCH != BLK_SEARCH_ONLY && W0) *(int *)(W0 + layer * nn) = !kept;
        if (SEARCH != BLK_SEARCH_MARK && info && sh.info) atomicCAS(&info[c], 0, sh.info);
    }
}

// the inversions of one launch's blocks.  Launches of at most one block per
// CU bound a level's latency: one kernel does both inversions, with the
// registers of one workgroup per CU.  Larger ones run diagonal pivots alone
// at the occupancy their registers allow, then a launch that takes only the
// blocks which refused them.
template <int NB>
void launch_bcr_invert(int ni, int n, const int4 *el, const int2 *top, const int *off, const double *A, double *W0,
                       double *Dinv, int *info, const vk_colstate *st, int ncu, hipStream_t s) {
    auto launch = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, dim3(n), dim3(blk_nt(NB)), 0, s, ni, n, el, top, off, A, W0, Dinv, info, st);
    };
    if constexpr (blk_nt(NB) == NT) {
        if (n <= ncu) {
            launch(k_bcr_invert<NB, BLK_SEARCH_HERE, 1>);
            return;
        }
    }
    launch(k_bcr_invert<NB, BLK_SEARCH_MARK, 2>);
    launch(k_bcr_invert<NB, BLK_SEARCH_ONLY, 2>);
}

// level 0: couplings are the diagonals Lsub (B) and Usup (C); elementwise.
// Survivors: 32 x 32 tiles (a: block row, b: block column), the grid's y
// dimension over a block's tiles; P, Q, B, C (transposed storage, index
// tt = b*ni + a) are written in the loop order with a fastest, the Schur
// update of A (row-major) goes through LDS and is written with b fastest:
// A = D - update (A holds nothing before level 0: the level's eliminated
// blocks are inverted from D directly).
// Workgroups n .. n+ne-1 form the back-substitution operators of the
// eliminated layers instead: XB = A_k^-1 diag(Lsub_k), XC = A_k^-1 diag(Usup_k)
// (over tt, the block's range split over the grid's y dimension); the last ncols
// decide which columns search their pivots from here on.
__global__ void k_bcr_update0(int ni, int n, const int4 *__restrict__ sv, const int *__restrict__ sflag,
                              int slot0, const double *__restrict__ Lsub, const double *__restrict__ Usup,
                              double *Dinv, const double *__restrict__ D, double *__restrict__ A,
                              double *__restrict__ Bt, double *__restrict__ Ct, double *__restrict__ Pt,
                              double *__restrict__ Qt, const int4 *__restrict__ el, int ne,
                              double *__restrict__ XBt, double *__restrict__ XCt, int ncols,
                              const int *__restrict__ off, const vk_colstate *__restrict__ st) {
    const int q = blockIdx.x;
    if (q >= n + ne + ncols) return;
    if (q >= n + ne) {
        const int c = q - n - ne;
        if (blockIdx.y != 0 || (st && st[c].done)) return;
        // level 0 eliminates the even layers of an odd count, else the odd ones
        const int nz = off[c + 1] - off[c], gone = off[c] + (nz & 1 ? 0 : 1), stay = off[c] + (nz & 1), ng = (nz + 1) / 2;
        const size_t nn = (size_t)ni * ni;
        int refused = 0;
        for (int u0 = 0; u0 < ng; u0 += NT) {
            const int u = u0 + threadIdx.x;
            refused += __syncthreads_count(u < ng && *(const int *)(A + (gone + 2 * u) * nn));
        }
        for (int u = threadIdx.x; u < nz - ng; u += NT) {
            double *X = Dinv + (stay + 2 * u) * nn;
            if (BCR_SEARCH_PART * refused > ng) blk_mark(X);
            else *X = 0.0;
        }
        return;
    }
    if (q >= n) {
        const int4 e = el[q - n];
        if (st && st[e.w].done) return;
        const size_t nn = (size_t)ni * ni, k = e.x;
        const double *X = Dinv + k * nn;     // X[b][a] = inv[a][b]
        const int span = (ni * ni + gridDim.y - 1) / gridDim.y, t0 = blockIdx.y * span;
        const int t1 = min(ni * ni, t0 + span);
        for (int tt = t0 + threadIdx.x; tt < t1; tt += blockDim.x) {
            const int b = tt / ni;
            XBt[k * nn + tt] = X[tt] * Lsub[k * ni + b];
            XCt[k * nn + tt] = X[tt] * Usup[k * ni + b];
        }
        return;
    }
    const int4 e = sv[q];
    if (st && st[e.w].done) return;
    const int fl = sflag[q];
    const size_t nn = (size_t)ni * ni, j = e.x;
    const size_t slot = (size_t)(slot0 + q) * nn;
    const double *XL = e.y >= 0 ? Dinv + (size_t)e.y * nn : nullptr;   // X[m][i] = inv[i][m]
    const double *XR = e.z >= 0 ? Dinv + (size_t)e.z * nn : nullptr;
    __shared__ double up[32][33];
    const int tpr = (ni + 31) / 32;
    for (int tile = blockIdx.y; tile < tpr * tpr; tile += gridDim.y) {
        const int a0 = 32 * (tile % tpr), b0 = 32 * (tile / tpr);
        for (int u = threadIdx.x; u < 32 * 32; u += blockDim.x) {
            const int al = u & 31, bl = u >> 5, a = a0 + al, b = b0 + bl;
            double upd = 0.0;
            if (a < ni && b < ni) {
                const size_t tt = (size_t)b * ni + a;
                if (XL) {
                    const double p = Lsub[j * ni + a] * XL[tt];
                    Pt[slot + tt] = p;
                    upd = p * Usup[(size_t)e.y * ni + b];
                    Bt[j * nn + tt] = (fl & 1) ? -(p * Lsub[(size_t)e.y * ni + b]) : 0.0;
                } else {
                    Bt[j * nn + tt] = 0.0;
                }
                if (XR) {
                    const double qv = Usup[j * ni + a] * XR[tt];
                    Qt[slot + tt] = qv;
                    upd = upd + qv * Lsub[(size_t)e.z * ni + b];
                    Ct[j * nn + tt] = (fl & 2) ? -(qv * Usup[(size_t)e.z * ni + b]) : 0.0;
                } else {
                    Ct[j * nn + tt] = 0.0;
                }
            }
            up[al][bl] = upd;
        }
        __syncthreads();
        for (int u = threadIdx.x; u < 32 * 32; u += blockDim.x) {
            const int bl = u & 31, al = u >> 5, a = a0 + al, b = b0 + bl;
            if (a < ni && b < ni) {
                const size_t o = j * nn + (size_t)a * ni + b;
                A[o] = D[o] - up[al][bl];
            }
        }
        __syncthreads();
    }
}

// Levels >= 1: dense couplings, products on FP64 MFMA, one workgroup per
// (layer, 32-row slab, 32 output columns): a slab's output rows depend
// only on the same rows of the left operands, so the slabs are
// independent, and the column groups split a slab's MFMA chain and right
// operands over several workgroups.  Two launches
// after the level's inversions, each one product deep:
//
// k_bcr_pq, survivors j (x < n):       P_j = B_j A_l^-1,  Q_j = C_j A_r^-1
//           eliminated k (x >= n):     the back-substitution operators
//                                      XB_k = A_k^-1 B_k,  XC_k = A_k^-1 C_k
//           (an eliminated layer's couplings are final: only survivors'
//           couplings change at this level)
// k_bcr_update, survivors j, slice 0:    A_j -= P_j C_l + Q_j B_r
//                            slice 1:    B_j = -P_j B_l,  C_j = -Q_j C_r
//           (slice 0 reads the eliminated neighbours' couplings, slice 1
//           writes the survivor's own: the two slices are independent)
// Grid z: column group (k_bcr_pq), slice * BCR_NCS<NB> + column group
// (k_bcr_update).
template <int NB>
constexpr int BCR_NBH = NB >= 2 ? 2 : 1;                        // column blocks per workgroup
template <int NB>
constexpr int BCR_NCS = (NB + BCR_NBH<NB> - 1) / BCR_NBH<NB>;   // workgroups across a block's columns

template <int NB, int KC>
__global__ void __launch_bounds__(NT) k_bcr_pq(int ni, int n, const int4 *__restrict__ sv, int slot0,
                                               const double *__restrict__ Dinv, const double *__restrict__ Bt,
                                               const double *__restrict__ Ct, double *__restrict__ Pt,
                                               double *__restrict__ Qt, const int4 *__restrict__ el, int ne,
                                               double *__restrict__ XBt, double *__restrict__ XCt,
                                               const vk_colstate *__restrict__ st) {
    constexpr int NBH = BCR_NBH<NB>;
    const int q = blockIdx.x, r0 = 32 * blockIdx.y, c0 = 16 * NBH * (int)blockIdx.z;
    if (q >= n + ne || r0 >= ni || c0 >= ni) return;
    const int4 e = q >= n ? el[q - n] : sv[q];
    if (st && st[e.w].done) return;
    __shared__ SlabShared<NBH, KC> g;
    const size_t nn = (size_t)ni * ni;
    f64x4 acc[(NBH + 1) / 2], acc2[(NBH + 1) / 2];
    slab_zero<NBH>(acc);
    slab_zero<NBH>(acc2);
    if (q >= n) {
        const size_t k = e.x;
        // A_k^-1 (a, c) = X[c][a]: the transposed-storage inverse is the At operand
        slab_gemm2<NBH, false, KC>(acc, acc2, ni, r0, Dinv + k * nn, Bt + k * nn, Dinv + k * nn, Ct + k * nn, g, c0);
        slab_store<NBH>(acc, ni, r0, XBt + k * nn, true, 1.0, nullptr, c0);
        slab_store<NBH>(acc2, ni, r0, XCt + k * nn, true, 1.0, nullptr, c0);
        return;
    }
    const size_t j = e.x, slot = (size_t)(slot0 + q) * nn;
    const bool hl = e.y >= 0, hr = e.z >= 0;
    // B_j(a, c) = Bt_j[c][a], inv(c, b) = X[b][c]
    if (hl) slab_gemm2<NBH, false, KC>(acc, acc2, ni, r0, Bt + j * nn, Dinv + (size_t)e.y * nn,
                                      hr ? Ct + j * nn : nullptr, hr ? Dinv + (size_t)e.z * nn : nullptr, g, c0);
    else if (hr) slab_gemm2<NBH, false, KC>(acc2, acc, ni, r0, Ct + j * nn, Dinv + (size_t)e.z * nn, nullptr, nullptr,
                                           g, c0);
    if (hl) slab_store<NBH>(acc, ni, r0, Pt + slot, true, 1.0, nullptr, c0);
    if (hr) slab_store<NBH>(acc2, ni, r0, Qt + slot, true, 1.0, nullptr, c0);
}

template <int NB, int KC>
__global__ void __launch_bounds__(NT) k_bcr_update(int ni, int n, const int4 *__restrict__ sv,
                                                   const int *__restrict__ sflag, int slot0, double *__restrict__ A,
                                                   double *__restrict__ Bt, double *__restrict__ Ct,
                                                   const double *__restrict__ Pt, const double *__restrict__ Qt,
                                                   const vk_colstate *__restrict__ st) {
    constexpr int NBH = BCR_NBH<NB>;
    const int q = blockIdx.x, r0 = 32 * blockIdx.y, cg = (int)blockIdx.z % BCR_NCS<NB>;
    const int slice = (int)blockIdx.z / BCR_NCS<NB>, c0 = 16 * NBH * cg;
    if (q >= n || r0 >= ni || c0 >= ni) return;
    const int4 e = sv[q];
    if (st && st[e.w].done) return;
    __shared__ SlabShared<NBH, KC> g;
    const size_t nn = (size_t)ni * ni, j = e.x;
    const double *Ptj = Pt + (size_t)(slot0 + q) * nn, *Qtj = Qt + (size_t)(slot0 + q) * nn;
    f64x4 acc[(NBH + 1) / 2], acc2[(NBH + 1) / 2];
    slab_zero<NBH>(acc);
    slab_zero<NBH>(acc2);
    if (slice == 0) {
        // one accumulator for both products
        const bool hl = e.y >= 0, hr = e.z >= 0;
        if (hl) slab_gemm2<NBH, true, KC>(acc, acc2, ni, r0, Ptj, Ct + (size_t)e.y * nn, hr ? Qtj : nullptr,
                                         hr ? Bt + (size_t)e.z * nn : nullptr, g, c0);
        else if (hr) slab_gemm2<NBH, true, KC>(acc, acc2, ni, r0, Qtj, Bt + (size_t)e.z * nn, nullptr, nullptr, g, c0);
        slab_store<NBH>(acc, ni, r0, A + j * nn, false, -1.0, A + j * nn, c0);
        return;
    }
    // the new couplings reach past the eliminated neighbours (zero where there is no layer beyond)
    const int fl = sflag[q];
    const bool nl = fl & 1, nr = fl & 2;
    if (nl) slab_gemm2<NBH, false, KC>(acc, acc2, ni, r0, Ptj, Bt + (size_t)e.y * nn, nr ? Qtj : nullptr,
                                      nr ? Ct + (size_t)e.z * nn : nullptr, g, c0);
    else if (nr) slab_gemm2<NBH, false, KC>(acc2, acc, ni, r0, Qtj, Ct + (size_t)e.z * nn, nullptr, nullptr, g, c0);
    slab_store<NBH>(acc, ni, r0, Bt + j * nn, true, -1.0, nullptr, c0);
    slab_store<NBH>(acc2, ni, r0, Ct + j * nn, true, -1.0, nullptr, c0);
}

// Solve sweeps: each block's products are split over row groups of 32 (one
// workgroup each, grid y), so a block's operators are read by several CUs at
// once; 256 threads, thread t owns row a0 + t % 32 and part h = t / 32 of the
// b range (chunks of ceil(ni/8) <= CH).  Every operator entry a thread needs
// is loaded into registers before the first product, and the eight partial
// sums of a row are combined through LDS in part order.  9 columns of 61
// to 110 layers, 150 species: a sweep pair 685 -> 217 us against one workgroup
// per block without loads ahead; one column of 150 layers, 93 species: 9 % of
// a sweep from loads that no branch splits.
constexpr int MV_NT = 256, MV_RG = 32, MV_SP = 8;

// m[i] = Mt[h ch + i][a], zero past the block (out of the buffer's range)
template <int CH>
__device__ __forceinline__ void mv_load(double (&m)[CH], const double *Mt, int ni, int a, int h, int ch) {
    const __amdgpu_buffer_rsrc_t rs =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<double *>(Mt), (short)0, ni * ni * 8, 0x00020000);
    const int voff = (h * ch * ni + min(a, ni - 1)) * 8;
#pragma unroll
    for (int i = 0; i < CH; i++)
        if (i < ch)
            m[i] = __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(rs, voff + i * ni * 8, 0, 0));
}

// v: MV_SP CH entries, zero past the block
template <int CH>
__device__ __forceinline__ double mv_dot(const double (&m)[CH], const double *v, int h, int ch) {
    double s0 = 0.0, s1 = 0.0;
#pragma unroll
    for (int i = 0; i < CH; i += 2) {
        if (i < ch) s0 = fma(m[i], v[h * ch + i], s0);
        if (i + 1 < ch) s1 = fma(m[i + 1], v[h * ch + i + 1], s1);
    }
    return s0 + s1;
}

// rin: the right-hand sides read (the solve's input at level 0, else r
// itself); at level 0 (sflag non-null) the sweep also places the
// eliminated layers' right-hand sides into r, each layer once: by its
// right survivor, or by its left one where it ends the column (no layer
// beyond it: sflag bit 1 clear).
template <int CH>
__global__ void __launch_bounds__(MV_NT) k_bcr_fwd_s(int ni, int n, const int4 *__restrict__ sv, int slot0,
                                                     const double *__restrict__ P, const double *__restrict__ Q,
                                                     const double *rin, double *r, const int *__restrict__ sflag,
                                                     const vk_colstate *__restrict__ st) {
    const int q = blockIdx.x, a0 = MV_RG * blockIdx.y;
    if (q >= n || a0 >= ni) return;
    const int4 e = sv[q];
    if (st && st[e.w].done) return;
    const size_t nn = (size_t)ni * ni;
    const int lr = threadIdx.x % MV_RG, a = a0 + lr, h = threadIdx.x / MV_RG, ch = (ni + MV_SP - 1) / MV_SP;
    double mp[CH] = {}, mq[CH] = {};
    if (e.y >= 0) mv_load<CH>(mp, P + (size_t)(slot0 + q) * nn, ni, a, h, ch);
    if (e.z >= 0) mv_load<CH>(mq, Q + (size_t)(slot0 + q) * nn, ni, a, h, ch);
    __shared__ double rl[MV_SP * CH], rr[MV_SP * CH], pp[MV_SP][MV_RG];
    for (int i = threadIdx.x; i < MV_SP * CH; i += MV_NT) {
        rl[i] = i < ni && e.y >= 0 ? rin[(size_t)e.y * ni + i] : 0.0;
        rr[i] = i < ni && e.z >= 0 ? rin[(size_t)e.z * ni + i] : 0.0;
    }
    __syncthreads();
    pp[h][lr] = mv_dot<CH>(mp, rl, h, ch) + mv_dot<CH>(mq, rr, h, ch);
    __syncthreads();
    if (threadIdx.x < MV_RG && a < ni) {
        double t = 0.0;
#pragma unroll
        for (int k = 0; k < MV_SP; k++) t += pp[k][threadIdx.x];
        r[(size_t)e.x * ni + a] = rin[(size_t)e.x * ni + a] - t;
        if (sflag) {
            if (e.y >= 0) r[(size_t)e.y * ni + a] = rl[a];
            if (e.z >= 0 && !(sflag[q] & 2)) r[(size_t)e.z * ni + a] = rr[a];
        }
    }
}

template <int CH>
__global__ void __launch_bounds__(MV_NT) k_bcr_bwd_s(int ni, int n, const int4 *__restrict__ el,
                                                     const int2 *__restrict__ top, const double *__restrict__ Dinv,
                                                     const double *__restrict__ XB, const double *__restrict__ XC,
                                                     const double *__restrict__ r, double *__restrict__ x,
                                                     const vk_colstate *__restrict__ st, double *acc) {
    const int q = blockIdx.x, a0 = MV_RG * blockIdx.y;
    if (q >= n || a0 >= ni) return;
    int k, left = -1, right = -1, c;
    if (el) { const int4 e = el[q]; k = e.x; left = e.y; right = e.z; c = e.w; }
    else { k = top[q].x; c = top[q].y; }
    if (st && st[c].done) return;
    const size_t nn = (size_t)ni * ni;
    const int lr = threadIdx.x % MV_RG, a = a0 + lr, h = threadIdx.x / MV_RG, ch = (ni + MV_SP - 1) / MV_SP;
    // x_k = A_k^-1 r_k - XB x_l - XC x_r: one pass over three operators
    double mx[CH], mb[CH] = {}, mc[CH] = {};
    mv_load<CH>(mx, Dinv + (size_t)k * nn, ni, a, h, ch);   // X[m][a] = inv[a][m]: the transposed inverse
    if (left >= 0) mv_load<CH>(mb, XB + (size_t)k * nn, ni, a, h, ch);
    if (right >= 0) mv_load<CH>(mc, XC + (size_t)k * nn, ni, a, h, ch);
    __shared__ double rk[MV_SP * CH], xl[MV_SP * CH], xr[MV_SP * CH], pp[MV_SP][MV_RG];
    for (int i = threadIdx.x; i < MV_SP * CH; i += MV_NT) {
        rk[i] = i < ni ? r[(size_t)k * ni + i] : 0.0;
        xl[i] = i < ni && left >= 0 ? x[(size_t)left * ni + i] : 0.0;
        xr[i] = i < ni && right >= 0 ? x[(size_t)right * ni + i] : 0.0;
    }
    __syncthreads();
    pp[h][lr] = (mv_dot<CH>(mx, rk, h, ch) - mv_dot<CH>(mb, xl, h, ch)) - mv_dot<CH>(mc, xr, h, ch);
    __syncthreads();
    if (threadIdx.x < MV_RG && a < ni) {
        double t = 0.0;
#pragma unroll
        for (int p2 = 0; p2 < MV_SP; p2++) t += pp[p2][threadIdx.x];
        x[(size_t)k * ni + a] = t;
        if (acc) acc[(size_t)k * ni + a] = acc[(size_t)k * ni + a] + t;
    }
}

// The last level of one column when it holds two layers, the top survivor
// s and the eliminated layer e to its right: r_s -= Q_s r_e, x_s = A_s^-1
// r_s, x_e = A_e^-1 r_e - XB_e x_s, in one workgroup of MV_NT-thread row
// groups (ni <= 96) instead of three launches.  Each product is formed as
// in k_bcr_fwd_s / k_bcr_bwd_s (same partition of the columns, same order
// of the sums; their product with an absent neighbour is exactly +0.0 and
// stands here as that constant), so the results are theirs.
constexpr int TAIL_G = 3, TAIL_NIMAX = TAIL_G * MV_RG, TAIL_CH = TAIL_NIMAX / MV_SP;
__global__ void __launch_bounds__(MV_NT *TAIL_G) k_bcr_tail_s(int ni, const int4 *__restrict__ sv, int slot0,
                                                              const int4 *__restrict__ el, const double *__restrict__ Q,
                                                              const double *__restrict__ Dinv,
                                                              const double *__restrict__ XB, double *r, double *x,
                                                              const vk_colstate *__restrict__ st, double *acc) {
    const int4 es = sv[0], ee = el[0];
    if (st && st[es.w].done) return;
    const size_t nn = (size_t)ni * ni;
    const int g = threadIdx.x / MV_NT, tt = threadIdx.x % MV_NT;
    const int lr = tt % MV_RG, a = MV_RG * g + lr, h = tt / MV_RG, ch = (ni + MV_SP - 1) / MV_SP;
    const int ks = es.x, ke = ee.x;
    // every operator up front: Q_s, A_s^-1, A_e^-1, XB_e
    constexpr int CH = TAIL_CH;
    double mq[CH], mxs[CH], mxe[CH], mb[CH];
    mv_load<CH>(mq, Q + (size_t)slot0 * nn, ni, a, h, ch);
    mv_load<CH>(mxs, Dinv + (size_t)ks * nn, ni, a, h, ch);
    mv_load<CH>(mxe, Dinv + (size_t)ke * nn, ni, a, h, ch);
    mv_load<CH>(mb, XB + (size_t)ke * nn, ni, a, h, ch);
    __shared__ double re[TAIL_NIMAX], rs[TAIL_NIMAX], xs[TAIL_NIMAX], pp[TAIL_G][MV_SP][MV_RG];
    for (int i = threadIdx.x; i < TAIL_NIMAX; i += blockDim.x) {
        re[i] = i < ni ? r[(size_t)ke * ni + i] : 0.0;
        rs[i] = xs[i] = 0.0;                     // past the block; the block's entries follow below
    }
    __syncthreads();
    auto total = [&]() {
        double t = 0.0;
#pragma unroll
        for (int k = 0; k < MV_SP; k++) t += pp[g][k][lr];
        return t;
    };
    // forward: r_s -= P_s r_l + Q_s r_r, no left neighbour
    pp[g][h][lr] = 0.0 + mv_dot<CH>(mq, re, h, ch);
    __syncthreads();
    if (h == 0 && a < ni) {
        const double v = r[(size_t)ks * ni + a] - total();
        r[(size_t)ks * ni + a] = v;
        rs[a] = v;
    }
    __syncthreads();
    // top: x_s = A_s^-1 r_s, no neighbours
    pp[g][h][lr] = (mv_dot<CH>(mxs, rs, h, ch) - 0.0) - 0.0;
    __syncthreads();
    if (h == 0 && a < ni) {
        const double t = total();
        x[(size_t)ks * ni + a] = t;
        if (acc) acc[(size_t)ks * ni + a] = acc[(size_t)ks * ni + a] + t;
        xs[a] = t;
    }
    __syncthreads();
    // back-substitution of e: x_e = A_e^-1 r_e - XB_e x_s, no right neighbour
    pp[g][h][lr] = (mv_dot<CH>(mxe, re, h, ch) - mv_dot<CH>(mb, xs, h, ch)) - 0.0;
    __syncthreads();
    if (h == 0 && a < ni) {
        const double t = total();
        x[(size_t)ke * ni + a] = t;
        if (acc) acc[(size_t)ke * ni + a] = acc[(size_t)ke * ni + a] + t;
    }
}

// the two product launches of a level >= 1
template <int NB, int KC>
void launch_bcr_products(int ni, int ns, int ne, int ny, const int4 *sv, const int *sflag, int slot0,
                         const int4 *el, const double *Dinv, const vk_bcr_ws *ws, const vk_colstate *st,
                         hipStream_t s) {
    hipLaunchKernelGGL((k_bcr_pq<NB, KC>), dim3(ns + ne, ny, BCR_NCS<NB>), dim3(NT), 0, s, ni, ns, sv, slot0, Dinv,
                       ws->B, ws->C, ws->P, ws->Q, el, ne, ws->XB, ws->XC, st);
    hipLaunchKernelGGL((k_bcr_update<NB, KC>), dim3(ns, ny, 2 * BCR_NCS<NB>), dim3(NT), 0, s, ni, ns, sv, sflag, slot0,
                       ws->A, ws->B, ws->C, ws->P, ws->Q, st);
}

template <int NB>
int launch_bcr_factor_n(int ni, const vk_columns *cols, const double *D, const double *Lsub, const double *Usup,
                        double *Dinv, int *info, const vk_colstate *st, const vk_bcr_ws *ws, hipStream_t s) {
    const vk_bcr_sched &b = cols->bcr;
    // deep chunks where every workgroup of a launch is resident at once,
    // at most two per CU (with three, measured slower than shallow chunks)
    constexpr long per_cu = sizeof(SlabShared<BCR_NBH<NB>, SlabKC<NB>::deep>) <= 80 * 1024 ? 2 : 1;
    const long cap = per_cu * vk_device_cus();
    const int ny = (ni + 31) / 32;
    const int tpr = (ni + 31) / 32;
    for (int lev = 0; lev < b.nlev; lev++) {
        const int e0 = b.elim_off[lev], ne = b.elim_off[lev + 1] - e0;
        const int s0 = b.surv_off[lev], ns = b.surv_off[lev + 1] - s0;
        // level 0 inverts its eliminated blocks from D (the level-0 update writes A)
        if (ne > 0)
            launch_bcr_invert<NB>(ni, ne, b.d_elim + e0, nullptr, cols->d_off, lev == 0 ? D : ws->A,
                                  lev == 0 ? ws->A : nullptr, Dinv, info, st, vk_device_cus(), s);
        if (ns > 0) {
            if (lev == 0)
                hipLaunchKernelGGL(k_bcr_update0, dim3(ns + ne + cols->ncols, std::min(tpr * tpr, 16)), dim3(NT), 0, s, ni, ns,
                                   b.d_surv + s0, b.d_sflag + s0, s0, Lsub, Usup, Dinv, D, ws->A, ws->B, ws->C,
                                   ws->P, ws->Q, b.d_elim + e0, ne, ws->XB, ws->XC, cols->ncols, cols->d_off, st);
            else if ((long)(ns + ne) * ny * BCR_NCS<NB> <= cap && 2L * ns * ny * BCR_NCS<NB> <= cap)
                launch_bcr_products<NB, SlabKC<NB>::deep>(ni, ns, ne, ny, b.d_surv + s0, b.d_sflag + s0, s0,
                                                          b.d_elim + e0, Dinv, ws, st, s);
            else
                launch_bcr_products<NB, SlabKC<NB>::shallow>(ni, ns, ne, ny, b.d_surv + s0, b.d_sflag + s0, s0,
                                                             b.d_elim + e0, Dinv, ws, st, s);
        }
    }
    launch_bcr_invert<NB>(ni, b.ntop, nullptr, b.d_top, cols->d_off, ws->A, nullptr, Dinv, info, st, vk_device_cus(), s);
    VK_CHECK(hipGetLastError());
    return 0;
}

}  // namespace

int vk_launch_bcr_factor(int nb, int ni, const vk_columns *cols, const double *D, const double *Lsub,
                         const double *Usup, double *Dinv, int *info, const vk_colstate *st, const vk_bcr_ws *ws,
                         hipStream_t s) {
    switch (nb) {
    case 1: return launch_bcr_factor_n<1>(ni, cols, D, Lsub, Usup, Dinv, info, st, ws, s);
    case 2: return launch_bcr_factor_n<2>(ni, cols, D, Lsub, Usup, Dinv, info, st, ws, s);
    case 3: return launch_bcr_factor_n<3>(ni, cols, D, Lsub, Usup, Dinv, info, st, ws, s);
    case 4: return launch_bcr_factor_n<4>(ni, cols, D, Lsub, Usup, Dinv, info, st, ws, s);
    case 5: return launch_bcr_factor_n<5>(ni, cols, D, Lsub, Usup, Dinv, info, st, ws, s);
    case 6: return launch_bcr_factor_n<6>(ni, cols, D, Lsub, Usup, Dinv, info, st, ws, s);
    case 7: return launch_bcr_factor_n<7>(ni, cols, D, Lsub, Usup, Dinv, info, st, ws, s);
    case 8: return launch_bcr_factor_n<8>(ni, cols, D, Lsub, Usup, Dinv, info, st, ws, s);
    case 9: return launch_bcr_factor_n<9>(ni, cols, D, Lsub, Usup, Dinv, info, st, ws, s);
    case 10: return launch_bcr_factor_n<10>(ni, cols, D, Lsub, Usup, Dinv, info, st, ws, s);
    default: return VK_ETOOBIG;
    }
}

template <int CH>
static int launch_bcr_solve(int ni, const vk_columns *cols, const double *Dinv, const double *in, double *out,
                            double *tmp, const vk_colstate *st, const vk_bcr_ws *ws, double *acc, hipStream_t s) {
    const vk_bcr_sched &b = cols->bcr;
    const int gy = (ni + MV_RG - 1) / MV_RG;
    // the last level and the top in one launch (one column, ni <= 96)
    const bool tail = b.tail && ni <= TAIL_NIMAX;
    // level 0 reads `in` and fills tmp
    for (int lev = 0; lev < b.nlev; lev++) {
        const int s0 = b.surv_off[lev], ns = b.surv_off[lev + 1] - s0;
        if (ns <= 0) continue;
        if (tail && lev == b.nlev - 1) {
            const int e0 = b.elim_off[lev];
            hipLaunchKernelGGL(k_bcr_tail_s, dim3(1), dim3(MV_NT * gy), 0, s, ni, b.d_surv + s0, s0, b.d_elim + e0,
                               ws->Q, Dinv, ws->XB, tmp, out, st, acc);
            break;
        }
        hipLaunchKernelGGL(k_bcr_fwd_s<CH>, dim3(ns, gy), dim3(MV_NT), 0, s, ni, ns, b.d_surv + s0, s0, ws->P, ws->Q,
                           lev == 0 ? in : tmp, tmp, lev == 0 ? b.d_sflag + s0 : (const int *)nullptr, st);
    }
    if (!tail)
        hipLaunchKernelGGL(k_bcr_bwd_s<CH>, dim3(b.ntop, gy), dim3(MV_NT), 0, s, ni, b.ntop, (const int4 *)nullptr,
                           b.d_top, Dinv, ws->XB, ws->XC, tmp, out, st, acc);
    for (int lev = b.nlev - 1 - (tail ? 1 : 0); lev >= 0; lev--) {
        const int e0 = b.elim_off[lev], ne = b.elim_off[lev + 1] - e0;
        if (ne > 0)
            hipLaunchKernelGGL(k_bcr_bwd_s<CH>, dim3(ne, gy), dim3(MV_NT), 0, s, ni, ne, b.d_elim + e0,
                               (const int2 *)nullptr, Dinv, ws->XB, ws->XC, tmp, out, st, acc);
    }
    VK_CHECK(hipGetLastError());
    return 0;
}

int vk_launch_bcr_solve(int ni, const vk_columns *cols, const double *Dinv, const double *Lsub, const double *Usup,
                        const double *in, double *out, double *tmp, const vk_colstate *st, const vk_bcr_ws *ws,
                        double *acc, hipStream_t s) {
    // CH: entries of a row a thread holds, MV_SP CH >= ni
    static_assert(VK_NI_MAX <= MV_SP * 20, "row chunks of the solve sweeps");
    if (ni <= MV_SP * 8) return launch_bcr_solve<8>(ni, cols, Dinv, in, out, tmp, st, ws, acc, s);
    if (ni <= MV_SP * 12) return launch_bcr_solve<12>(ni, cols, Dinv, in, out, tmp, st, ws, acc, s);
    if (ni <= MV_SP * 16) return launch_bcr_solve<16>(ni, cols, Dinv, in, out, tmp, st, ws, acc, s);
    return launch_bcr_solve<20>(ni, cols, Dinv, in, out, tmp, st, ws, acc, s);
}
