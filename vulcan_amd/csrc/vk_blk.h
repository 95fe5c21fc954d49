// Device building blocks shared by the block-inversion kernels: the blocked
// Gauss-Jordan inversion on FP64 MFMA tiles (chain factorisation and cyclic
// reduction) and the slab products of the cyclic-reduction updates.
#pragma once
#include <cstddef>

#include "vk_internal.h"

namespace {

constexpr int NT = 256;

// Threads of a blocked-inversion workgroup: 4 waves up to 96 rows, 8 waves
// above (the accumulator tiles of 128-160 rows would not fit 4 waves'
// registers), with the waves in a 2 x (waves / 2) grid over the tiles.
constexpr int blk_nt(int nb) { return nb >= 7 ? 512 : 256; }
template <int NB>
struct BlkGrid {
    static constexpr int NTH = blk_nt(NB), NW = NTH / 64, WC = NW / 2;
    static constexpr int TBR = (NB + 1) / 2, TBC = (NB + WC - 1) / WC;   // tiles per wave: rows, columns
};

// ---------------------------------------------------------------------------
// Blocked Gauss-Jordan inversion on FP64 MFMA with searched pivots (factor
// variants 1, 2 and 4, for blocks that refuse their diagonal as pivots, below)
//
// The pivot steps are grouped into panels of 16 columns.  One wave runs the
// 16 pivot steps of a panel on the panel columns alone (rows spread over the
// lanes, pivot search by a wave-wide max over 32-bit (|value|, row) keys,
// pivot row handed over through LDS: no workgroup barrier inside a panel;
// the panel wave rotates with the panel and the workgroup index, so that
// co-resident workgroups do not run their panels on the same SIMD; a version
// spreading the panel over four waves, two barriers per step, measured
// slower).  The other columns then receive the whole panel at once, as the
// rank-16 Schur update
//     A[i][j] = (i in P ? 0 : A[i][j]) + sum_s Pan[i][s] A_old[p_s][j]
// (P: the panel's pivot rows p_s, Pan: the factored panel columns), which is
// a 16-deep GEMM and runs on v_mfma_f64_16x16x4f64.  Three barriers per
// panel.  The matrix lives in the MFMA
// accumulator layout: 16 x 16 tiles, wave (wr, wc) of the 2 x WC wave grid
// (WC = 2 or 4, BlkGrid) owns row blocks wr, wr+2, ... and column blocks
// wc, wc+WC, ...; lane l,
// register r of a tile holds element (4*r + l/16, l%16) (operands: A(i, k)
// in lane i + 16 k, B(k, j) in lane j + 16 k; checked by
// vk_selftest_mfma_f64).
// Pivoting is implicit (rows are not swapped): ipos[r] is the pivot step at
// which row r was chosen, perm[k] the pivot row of step k, and the inverse is
// inv[ipos[r]][perm[c]] = A[r][c] at the end.
// ---------------------------------------------------------------------------
typedef double f64x4 __attribute__((ext_vector_type(4)));

// Pivots per panel of blk_invert_diag.  A pivot step broadcasts a row of the
// panel and updates its columns, so narrow panels halve it, and twice as many
// panels cost a round of publishing and two barriers each.  Panels of 8 against
// 16, chains of 1, 80 and 256 columns of 60 layers (us):
//   30 species   182 : 192    194 : 208    266 : 322
//   48           392 : 372    409 : 392    582 : 604
//   49           459 : 444    481 : 461    768 : 674
//   93           978 : 855   1051 : 930   1477 : 1445
//   96          1037 : 911   1108 : 989   1484 : 1558
//   97          1405 : 1519  1542 : 1621  2373 : 3145
//   112         1615 : 1620  1759 : 1735  2585 : 3434
//   128         1844 : 1868  1977 : 2003
//   160         3143 : 3001  3373 : 3236
// so 8 up to 48 and above 96 species, where up to 112 the registers it saves
// also let two workgroups share a CU.
template <int NB>
constexpr int DIAG_PW = NB <= 3 || blk_nt(NB) > NT ? 8 : 16;

template <int NB>
struct alignas(16) BlkShared {
    static constexpr int N16 = 16 * NB;
    // above 128 rows the panel wave parks its accumulator tiles here during
    // the panel (its registers then hold the panel alone)
    static constexpr bool PARK = NB >= 9;
    union {
        struct {                      // blk_invert
            double pan[2][16][N16 + 1];   // panel columns, [k][row], double-buffered by panel parity
            double rb[16][N16];           // old pivot rows of the panel, [s][col]
            double dump[blk_nt(NB)];      // per-thread target of discarded writes
            double prow[16];              // current pivot row of the panel factorisation
            int ipos[N16];
            int perm[N16];
            double park[PARK ? 4 * ((NB + 1) / 2) * ((NB + 3) / 4) : 1][64];
        };
        struct {                      // blk_invert_diag
            double dpan[DIAG_PW<NB>][N16 + 1];   // panel columns, [k][row]
            double dfac[DIAG_PW<NB>][N16 + 1];   // the factored panel
            double drb[2][DIAG_PW<NB>][N16];     // old pivot rows, [s][col], by panel parity
            double diag[N16];             // the block's diagonal as given
        };
    };
    // behind the arrays, whose 16-byte accesses need the alignment: in front of
    // them they cost the searched inversion of up to 32 rows the fourth
    // workgroup of a CU (140 registers for 106: every chain of 512 columns of
    // 30 species searched, 1.75 ms against 1.02) and that of 64 rows a tenth
    // of its time
    int info;
    int refused;                      // a diagonal pivot was refused (blk_invert_diag)
};
static_assert(offsetof(BlkShared<6>, pan) % 16 == 0 && offsetof(BlkShared<6>, prow) % 16 == 0 &&
                  offsetof(BlkShared<10>, park) % 16 == 0,
              "arrays of the searched inversion on 16 bytes");

template <int CTRL>
__device__ __forceinline__ unsigned long long dpp_u64(unsigned long long v) {
    const int lo = __builtin_amdgcn_update_dpp(0, (int)(unsigned)(v & 0xffffffffull), CTRL, 0xf, 0xf, false);
    const int hi = __builtin_amdgcn_update_dpp(0, (int)(unsigned)(v >> 32), CTRL, 0xf, 0xf, false);
    return ((unsigned long long)(unsigned)hi << 32) | (unsigned long long)(unsigned)lo;
}

// Maximum over the 64 lanes (all active), wave-uniform: DPP max within rows
// of 16 (quad swaps, half-row and row mirrors), then row_bcast:15 and
// row_bcast:31 carry the row maxima up to lane 63, read once.
__device__ __forceinline__ unsigned wave_max_u32(unsigned v) {
    v = max(v, (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0xB1, 0xf, 0xf, false));
    v = max(v, (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0x4E, 0xf, 0xf, false));
    v = max(v, (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0x141, 0xf, 0xf, false));
    v = max(v, (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0x140, 0xf, 0xf, false));
    v = max(v, (unsigned)__builtin_amdgcn_update_dpp((int)v, (int)v, 0x142, 0xa, 0xf, false));   // rows 1, 3 += row 0, 2
    v = max(v, (unsigned)__builtin_amdgcn_update_dpp((int)v, (int)v, 0x143, 0xc, 0xf, false));   // rows 2, 3 += row 1
    return (unsigned)__builtin_amdgcn_readlane((int)v, 63);
}

// 1 / d: the hardware reciprocal estimate refined by two Newton-Raphson
// steps (e = 1 - d r, r = r + r e), within about an ulp; the IEEE division
// sequence (scale, estimate, refinement, fix-up) is twice as long on the
// pivot step's path.
__device__ __forceinline__ double blk_recip(double d) {
    double r = __builtin_amdgcn_rcp(d);
    double e = fma(-d, r, 1.0);
    r = fma(r, e, r);
    e = fma(-d, r, 1.0);
    return fma(r, e, r);
}

// Pivot steps p0 .. p0+kend-1 on the panel pan[k][row] (one wave).  The
// pivot key is the upper word of |value| with the row in its low byte: the
// largest magnitude to 12 mantissa bits, ties to the lowest row.  The pivot
// bookkeeping (ipos of the chosen rows, perm of the steps) stays in
// registers until the panel ends: no LDS write waits inside a step.
//
// A step subtracts (v[kk] / pivot) x the pivot row from every other row.
// The update is linear in the row, so a chosen pivot row is kept unscaled
// (its own multiplier is 0 and its pivot-column entry 1): later steps update
// it like any row, and the panel's end multiplies it by its 1 / pivot,
// giving the Gauss-Jordan values (the scaled row, 1 / pivot in the pivot
// column) without scaling the row inside the step.
template <int NB>
__device__ __forceinline__ void blk_panel(BlkShared<NB> &sh, double (*pan)[16 * NB + 1], int ni, int p0, int kend,
                                          int tag) {
    constexpr int N16 = 16 * NB;
    constexpr int RPL = (N16 + 63) / 64;
    const int l = threadIdx.x & 63;
    double v[RPL][16];
    // this lane's row q: -1 still available, -2 not a candidate (padding or
    // chosen in an earlier panel), >= 0 the pivot step that chose it
    int code[RPL];
    double pinv[RPL];   // 1 / pivot of a row chosen in this panel
    bool zero = false;
#pragma unroll
    for (int q = 0; q < RPL; q++) {
        const int r = l + 64 * q;
#pragma unroll
        for (int k = 0; k < 16; k++) v[q][k] = (r < N16) ? pan[k][r] : 0.0;
        code[q] = (r < ni) && sh.ipos[r] < 0 ? -1 : -2;
        pinv[q] = 1.0;
    }
#pragma unroll
    for (int kk = 0; kk < 16; kk++) {
        if (kk >= kend) continue;   // uniform; keeps the trip count static
        unsigned best = 0;
#pragma unroll
        for (int q = 0; q < RPL; q++) {
            const int r = l + 64 * q;
            const unsigned key =
                ((unsigned)(__double_as_longlong(fabs(v[q][kk])) >> 32) & ~0xffu) | (unsigned)(255 - r);
            best = code[q] == -1 && key > best ? key : best;
        }
        best = wave_max_u32(best);
        const int p = best ? 255 - (int)(best & 0xffu) : 0;
        zero = zero || (best >> 8) == 0u;   // zero (or no) pivot
        const int pl = p & 63, qp = p >> 6;
        // the owner lane hands the pivot row to the wave through LDS (in order within the wave)
#pragma unroll
        for (int q = 0; q < RPL; q++)
            if (q == qp && l == pl) {
#pragma unroll
                for (int k = 0; k < 16; k++) sh.prow[k] = v[q][k];
            }
        // lanes exchange data here: without the barrier the compiler may let the
        // other lanes read before the owner's (exec-masked) writes
        __builtin_amdgcn_wave_barrier();
        double rs[16];
#pragma unroll
        for (int k = 0; k < 16; k++) rs[k] = sh.prow[k];
        const double inv = blk_recip(rs[kk]);
#pragma unroll
        for (int q = 0; q < RPL; q++) {
            const bool own = q == qp && l == pl;
            const double f = own ? 0.0 : v[q][kk] * inv;
#pragma unroll
            for (int k = 0; k < 16; k++) v[q][k] = fma(-f, rs[k], v[q][k]);
            v[q][kk] = own ? 1.0 : -f;
            code[q] = own ? p0 + kk : code[q];
            pinv[q] = own ? inv : pinv[q];
        }
        if (l == 0) sh.perm[p0 + kk] = p;
    }
    if (zero && l == 0 && sh.info == 0) sh.info = tag;
#pragma unroll
    for (int q = 0; q < RPL; q++) {
        const int r = l + 64 * q;
        if (code[q] >= 0) sh.ipos[r] = code[q];
        if (r < N16) {
            // rows chosen in this panel take their 1 / pivot (the others 1.0, exact)
#pragma unroll
            for (int k = 0; k < 16; k++) pan[k][r] = v[q][k] * pinv[q];
        }
    }
    for (int s = kend; s < 16; s++)
        for (int c = l; c < N16; c += 64) sh.rb[s][c] = 0.0;
}


// Inverts the matrix held in acc (MFMA tile layout) and writes the inverse
// transposed to X (X[m][i] = inv[i][m]).  A zero pivot records `tag` in
// sh.info (sticky).
template <int NB>
__device__ __forceinline__ void blk_invert(f64x4 (&acc)[BlkGrid<NB>::TBR][BlkGrid<NB>::TBC], int ni,
                                           double *__restrict__ X, BlkShared<NB> &sh, int tag) {
    using G = BlkGrid<NB>;
    constexpr int N16 = 16 * NB, TBR = G::TBR, TBC = G::TBC, WC = G::WC;
    const int tid = threadIdx.x, w = tid >> 6, l = tid & 63;
    const int wr = w / WC, wc = w % WC;
    const int lg = l >> 4, lc = l & 15;
    for (int t = tid; t < N16; t += G::NTH) sh.ipos[t] = -1;
    __syncthreads();
    const int npan = (ni + 15) >> 4;
    for (int pb = 0; pb < npan; pb++) {
        double(*pan)[N16 + 1] = sh.pan[pb & 1];
        const int p0 = 16 * pb, kend = min(16, ni - p0);
        // the owners of column block pb publish the panel
#pragma unroll
        for (int tj = 0; tj < TBC; tj++) {
            if (wc + WC * tj != pb) continue;   // static register index, uniform test
#pragma unroll
            for (int ti = 0; ti < TBR; ti++) {
                const int bi = wr + 2 * ti;
                if (bi < NB) {
#pragma unroll
                    for (int r = 0; r < 4; r++) pan[lc][16 * bi + 4 * r + lg] = acc[ti][tj][r];
                }
            }
        }
        __syncthreads();
        if (w == ((pb + (int)blockIdx.x) & (G::NW - 1))) {
            if constexpr (BlkShared<NB>::PARK) {
#pragma unroll
                for (int ti = 0; ti < TBR; ti++)
#pragma unroll
                    for (int tj = 0; tj < TBC; tj++)
#pragma unroll
                        for (int r = 0; r < 4; r++) sh.park[(ti * TBC + tj) * 4 + r][l] = acc[ti][tj][r];
            }
            blk_panel<NB>(sh, pan, ni, p0, kend, tag);
            if constexpr (BlkShared<NB>::PARK) {
#pragma unroll
                for (int ti = 0; ti < TBR; ti++)
#pragma unroll
                    for (int tj = 0; tj < TBC; tj++)
#pragma unroll
                        for (int r = 0; r < 4; r++) acc[ti][tj][r] = sh.park[(ti * TBC + tj) * 4 + r][l];
            }
        }
        __syncthreads();
        // panel tiles take the factored panel; the other tiles hand their
        // pivot-row entries to rb and clear them
#pragma unroll
        for (int ti = 0; ti < TBR; ti++) {
            const int bi = wr + 2 * ti;
            if (bi >= NB) continue;
            int sr[4];
#pragma unroll
            for (int r = 0; r < 4; r++) sr[r] = sh.ipos[16 * bi + 4 * r + lg] - p0;
#pragma unroll
            for (int tj = 0; tj < TBC; tj++) {
                const int bj = wc + WC * tj;
                if (bj >= NB) continue;
                if (bj == pb) {
#pragma unroll
                    for (int r = 0; r < 4; r++) acc[ti][tj][r] = pan[lc][16 * bi + 4 * r + lg];
                } else {
                    // branch-free: entries of other rows go to the thread's own dump slot
#pragma unroll
                    for (int r = 0; r < 4; r++) {
                        const bool piv = (unsigned)sr[r] < 16u;
                        double *dst = piv ? &sh.rb[sr[r]][16 * bj + lc] : &sh.dump[tid];
                        *dst = acc[ti][tj][r];
                        acc[ti][tj][r] = piv ? 0.0 : acc[ti][tj][r];
                    }
                }
            }
        }
        __syncthreads();
        // rank-16 update on MFMA
#pragma unroll
        for (int ti = 0; ti < TBR; ti++) {
            const int bi = wr + 2 * ti;
            if (bi >= NB) continue;
            double a[4];
#pragma unroll
            for (int s4 = 0; s4 < 4; s4++) a[s4] = pan[4 * s4 + (l >> 4)][16 * bi + lc];
#pragma unroll
            for (int tj = 0; tj < TBC; tj++) {
                const int bj = wc + WC * tj;
                if (bj >= NB || bj == pb) continue;
#pragma unroll
                for (int s4 = 0; s4 < 4; s4++)
                    acc[ti][tj] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[s4], sh.rb[4 * s4 + (l >> 4)][16 * bj + lc],
                                                                        acc[ti][tj], 0, 0, 0);
            }
        }
    }
    // inv[ipos[r]][perm[c]] = A[r][c]  ->  X[perm[c]][ipos[r]]
#pragma unroll
    for (int ti = 0; ti < TBR; ti++) {
        const int bi = wr + 2 * ti;
        if (bi >= NB) continue;
        int qi[4];
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int i = 16 * bi + 4 * r + lg;
            qi[r] = i < ni ? sh.ipos[i] : -1;
        }
#pragma unroll
        for (int tj = 0; tj < TBC; tj++) {
            const int bj = wc + WC * tj;
            const int cc = 16 * bj + lc;
            if (bj >= NB || cc >= ni) continue;
            const size_t rowoff = (size_t)sh.perm[cc] * ni;
#pragma unroll
            for (int r = 0; r < 4; r++)
                if (qi[r] >= 0) X[rowoff + qi[r]] = acc[ti][tj][r];
        }
    }
    __syncthreads();
}

// ---------------------------------------------------------------------------
// The same inversion with the diagonal as pivots, for blocks that allow it.
//
// Searching the pivots makes the panel a serial chain on one wave: a
// wave-wide maximum, a row hand-over through LDS and the whole panel's
// update per step, some 900 cycles (36 of an inversion's 58 us at 93 rows)
// while the workgroup's other waves wait.  With the pivot rows known in
// advance, every wave holds the panel's pivot rows in its first lanes
// (all waves run the same steps on them) and its own share of the other rows
// in the lanes above, one row a lane: the pivot row of a step is lane kk's,
// read by v_readlane into scalar registers, no row crosses waves, and a
// panel takes two barriers instead of three (the old pivot rows are
// published with the panel).
//
// Which blocks allow it: the Ros2 lhs blocks c0 I - J - diffusion and their
// Schur complements behave like M-matrices, whose elimination in natural
// order takes from each diagonal entry and never adds to it.  A block is
// accepted when every pivot d has the sign of its entry a of the given block
// and at most twice its size (a / d >= DIAG_KEEP; zero and NaN pivots fail).
// The test does not depend on the scaling of rows or columns.  On the blocks
// of the 30-, 93- and 150-species columns over 140 to 200 steps (dt 1e-14 to
// 2e5 s) a / d was never below 1; the inverses were as near the exact ones
// as with searched pivots or nearer (18 to 40 times on blocks with species
// scaled over four decades); of 2 200 random normal matrices of 4 to 30 rows
// 17 were accepted, all of 4 rows.  Refused blocks are inverted by
// blk_invert (a third of the blocks in the first step from a random
// composition).
//
// One column of 150 layers and 93 species: factorisation and two solves 0.77
// -> 0.54 ms; chains of one column 5.25 -> 3.08 ms, of 256 columns (80 to 200
// layers) 9.3 -> 6.5 ms (5.6 with the chains' own Schur term and sweeps); nine
// 150-species columns 17.9 -> 12.5 ms.
// Returns whether the inverse has been written (uniform over the workgroup).
// ---------------------------------------------------------------------------
constexpr double DIAG_KEEP = 0.5;

__device__ __forceinline__ double lane_bcast(double v, int lane) {
    const unsigned long long b = (unsigned long long)__double_as_longlong(v);
    const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)b, lane);
    const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)(b >> 32), lane);
    return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}

template <int NB>
__device__ __forceinline__ bool blk_invert_diag(f64x4 (&acc)[BlkGrid<NB>::TBR][BlkGrid<NB>::TBC], int ni,
                                                double *__restrict__ X, BlkShared<NB> &sh) {
    using G = BlkGrid<NB>;
    constexpr int N16 = 16 * NB, TBR = G::TBR, TBC = G::TBC, WC = G::WC;
    constexpr int PW = DIAG_PW<NB>, SHARE = (N16 - PW + G::NW - 1) / G::NW;   // rows outside the pivots', per wave
    static_assert(SHARE + PW <= 64 && 16 % PW == 0 && PW % 4 == 0, "a wave's lanes hold the pivot rows and its share");
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));   // as in blk_load_schur: no index of this function lives across the caller's loop
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6), l = tid & 63;   // uniform: the tile tests are scalar branches
    const int wr = w / WC, wc = w % WC;
    const int lg = l >> 4, lc = l & 15;
    const int npan = (ni + PW - 1) / PW;
    // the padding is the identity's: its pivots are 1 and touch nothing, so
    // that every panel runs all its steps without a test
#pragma unroll
    for (int ti = 0; ti < TBR; ti++)
#pragma unroll
        for (int tj = 0; tj < TBC; tj++) {
            const int bi = wr + 2 * ti, bj = wc + WC * tj;
            if (bi != bj || bi >= NB) continue;
#pragma unroll
            for (int r = 0; r < 4; r++)
                if (4 * r + lg == lc) {
                    if (16 * bi + lc >= ni) acc[ti][tj][r] = 1.0;
                    sh.diag[16 * bi + lc] = acc[ti][tj][r];
                }
        }
    if (tid == 0) sh.refused = 0;
    for (int pb = 0; pb < npan; pb++) {
        double(*rb)[N16] = sh.drb[pb & 1];
        // the panel lies in tile row and column tb, at so
        const int p0 = PW * pb, tb = p0 >> 4, so = p0 & 15;
        const bool pc = lc - so >= 0 && lc - so < PW;      // the lane's column of tile tb is in the panel
        // the owners of the panel's columns and rows publish them and clear
        // them: the update below then writes them like any other entry (the
        // panel's columns as the factored panel times the identity)
#pragma unroll
        for (int ti = 0; ti < TBR; ti++) {
            const int bi = wr + 2 * ti;
            if (bi >= NB) continue;
#pragma unroll
            for (int tj = 0; tj < TBC; tj++) {
                const int bj = wc + WC * tj;
                if (bj >= NB) continue;
                if (bj == tb) {
#pragma unroll
                    for (int r = 0; r < 4; r++) {
                        if (pc) sh.dpan[lc - so][16 * bi + 4 * r + lg] = acc[ti][tj][r];
                        acc[ti][tj][r] = pc ? 0.0 : acc[ti][tj][r];
                    }
                }
                if (bi == tb) {
#pragma unroll
                    for (int r = 0; r < 4; r++) {
                        const int k = 4 * r - so;            // uniform: four pivot rows or none
                        if (k >= 0 && k < PW) {
                            const double one = lc - so == k + lg ? 1.0 : 0.0;
                            rb[k + lg][16 * bj + lc] = bj == tb && pc ? one : acc[ti][tj][r];
                            acc[ti][tj][r] = 0.0;
                        }
                    }
                }
            }
        }
        __syncthreads();
        {
            // lane -> row: the pivot rows, then this wave's share of the others
            const int o = w * SHARE + l - PW;
            const bool other = l >= PW && l < PW + SHARE && o < N16 - PW;
            const int row = l < PW ? p0 + l : (other ? (o < p0 ? o : o + PW) : p0);
            double v[PW], pinv = 1.0;
#pragma unroll
            for (int k = 0; k < PW; k++) v[k] = sh.dpan[k][row];
#pragma unroll
            for (int kk = 0; kk < PW; kk++) {
                const bool own = l == kk;
                // the pivot row, every entry into scalar registers of its own
                // (a shared pair would serialise read and use)
                double p[PW];
#pragma unroll
                for (int k = 0; k < PW; k++) p[k] = lane_bcast(v[k], kk);
                const double inv = blk_recip(p[kk]);
                const double f = own ? 0.0 : v[kk] * inv;
#pragma unroll
                for (int k = 0; k < PW; k++) asm volatile("" : "+s"(p[k]));
#pragma unroll
                for (int j = 1; j < PW; j++) {
                    const int k = (kk + j) % PW;      // the next pivot's column first
                    v[k] = fma(-f, p[k], v[k]);
                }
                v[kk] = own ? 1.0 : -f;
                pinv = own ? inv : pinv;
            }
            if (w == 0 && l < PW && !(sh.diag[row] * pinv >= DIAG_KEEP)) sh.refused = 1;
            if (other || (l < PW && w == 0)) {
#pragma unroll
                for (int k = 0; k < PW; k++) sh.dfac[k][row] = v[k] * pinv;
            }
        }
        __syncthreads();
        if (__builtin_amdgcn_readfirstlane(sh.refused)) return false;
        // rank-PW update on MFMA (tiles past the block read block 0's
        // operands, their values are never used)
        double b[TBC][PW / 4];
#pragma unroll
        for (int tj = 0; tj < TBC; tj++) {
            const int bj = wc + WC * tj;
#pragma unroll
            for (int s4 = 0; s4 < PW / 4; s4++) b[tj][s4] = rb[4 * s4 + lg][16 * (bj < NB ? bj : 0) + lc];
        }
#pragma unroll
        for (int ti = 0; ti < TBR; ti++) {
            const int bi = wr + 2 * ti;
            double a[PW / 4];
#pragma unroll
            for (int s4 = 0; s4 < PW / 4; s4++) a[s4] = sh.dfac[4 * s4 + lg][16 * (bi < NB ? bi : 0) + lc];
#pragma unroll
            for (int s4 = 0; s4 < PW / 4; s4++)
#pragma unroll
                for (int tj = 0; tj < TBC; tj++)
                    acc[ti][tj] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[s4], b[tj][s4], acc[ti][tj], 0, 0, 0);
        }
    }
#pragma unroll
    for (int ti = 0; ti < TBR; ti++) {
        const int bi = wr + 2 * ti;
        if (bi >= NB) continue;
#pragma unroll
        for (int tj = 0; tj < TBC; tj++) {
            const int bj = wc + WC * tj, cc = 16 * bj + lc;
            if (bj >= NB || cc >= ni) continue;
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int i = 16 * bi + 4 * r + lg;
                if (i < ni) X[(size_t)cc * ni + i] = acc[ti][tj][r];
            }
        }
    }
    __syncthreads();
    return true;
}

// acc = D_l - diag(cl) Xn^T diag(cn) [- diag(cl2) Xn2^T diag(cn2)] in the tile layout
//
// Branch-free: every thread loads all its entries unconditionally (padding
// rows and columns read element 0 and clear it with a bit mask, giving the
// +0.0 they hold), so a row block's loads are all in flight before the first
// wait.  With a conditional load per entry (or a select on the loaded
// value, which the compiler turns back into a branch) it waited on each
// entry's loads in turn.  Xn and Xn2 are uniform.
__device__ __forceinline__ double blk_masked(double v, unsigned long long m) {
    return __longlong_as_double(__double_as_longlong(v) & (long long)m);
}

template <int NB>
__device__ __forceinline__ void blk_load_schur(f64x4 (&acc)[BlkGrid<NB>::TBR][BlkGrid<NB>::TBC], int ni,
                                               const double *__restrict__ Dl, const double *cl, const double *Xn,
                                               const double *cn, const double *cl2, const double *Xn2,
                                               const double *cn2) {
    using G = BlkGrid<NB>;
    constexpr int TBR = G::TBR, TBC = G::TBC, WC = G::WC;
    int tid = threadIdx.x;
    // opaque to the optimiser: the indices below are formed here, at each
    // call, rather than hoisted out of the caller's loop and kept live in
    // registers through the inversion
    asm volatile("" : "+v"(tid));
    const int w = tid >> 6, l = tid & 63;
    const int wr = w / WC, wc = w % WC;
    const int lg = l >> 4, lc = l & 15;
    // column cc = 16 bj + lc of each column tile (index 0 and mask 0 outside the block)
    int cj[TBC];
    unsigned long long cm[TBC];
#pragma unroll
    for (int tj = 0; tj < TBC; tj++) {
        const int bj = wc + WC * tj, cc = 16 * bj + lc;
        const bool ok = bj < NB && cc < ni;
        cj[tj] = ok ? cc : 0;
        cm[tj] = ok ? ~0ull : 0ull;
    }
    // row i = 16 bi + 4 r + lg of each entry (index 0 and mask 0 outside the block)
    int ir[TBR][4];
    unsigned long long rm[TBR][4];
#pragma unroll
    for (int ti = 0; ti < TBR; ti++) {
        const int bi = wr + 2 * ti;
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int i = 16 * bi + 4 * r + lg;
            const bool rok = bi < NB && i < ni;
            ir[ti][r] = rok ? i : 0;
            rm[ti][r] = rok ? ~0ull : 0ull;
        }
    }
    // all of D's loads first, then (uniform) the Schur terms' loads
#pragma unroll
    for (int ti = 0; ti < TBR; ti++)
#pragma unroll
        for (int r = 0; r < 4; r++)
#pragma unroll
            for (int tj = 0; tj < TBC; tj++)
                acc[ti][tj][r] = blk_masked(Dl[(size_t)ir[ti][r] * ni + cj[tj]], rm[ti][r] & cm[tj]);
    // the Schur terms in groups of GR row tiles (all at once up to 96 rows;
    // one tile at a time above, where their loads would not fit the registers)
    constexpr int GR = TBR * TBC <= 9 ? TBR : 1;
    auto sub = [&](const double *c_l, const double *X, const double *c_n) {
        double cnv[TBC];
#pragma unroll
        for (int tj = 0; tj < TBC; tj++) cnv[tj] = c_n[cj[tj]];
#pragma unroll
        for (int t0 = 0; t0 < TBR; t0 += GR) {
            double li[GR][4], x[GR][4][TBC];
#pragma unroll
            for (int g = 0; g < GR; g++)
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    li[g][r] = c_l[ir[t0 + g][r]];
#pragma unroll
                    for (int tj = 0; tj < TBC; tj++) x[g][r][tj] = X[(size_t)cj[tj] * ni + ir[t0 + g][r]];
                }
#pragma unroll
            for (int g = 0; g < GR; g++)
#pragma unroll
                for (int r = 0; r < 4; r++)
#pragma unroll
                    for (int tj = 0; tj < TBC; tj++)
                        acc[t0 + g][tj][r] = blk_masked(acc[t0 + g][tj][r] - li[g][r] * (x[g][r][tj] * cnv[tj]),
                                                        rm[t0 + g][r] & cm[tj]);
        }
    };
    if (Xn) sub(cl, Xn, cn);
    if (Xn2) sub(cl2, Xn2, cn2);
}

// How a kernel inverts the blocks that refuse diagonal pivots:
enum BlkSearch {
    BLK_SEARCH_HERE,    // in place, with searched pivots (both inversions in the kernel's registers)
    BLK_SEARCH_MARK,    // not: their output is marked for a later launch, which takes ...
    BLK_SEARCH_ONLY     // ... the marked blocks alone, with searched pivots
};

// The mark: a signalling NaN pattern no operation returns, in the first
// entry of the block's output.
constexpr unsigned long long BLK_MARK = 0x7ff4756c63616e00ull;

__device__ __forceinline__ void blk_mark(double *X) { *(volatile unsigned long long *)X = BLK_MARK; }

__device__ __forceinline__ bool blk_marked(const double *X) {
    return *(const volatile unsigned long long *)X == BLK_MARK;
}

// X = the transposed inverse of D_l - diag(cl) Xn^T diag(cn) [- diag(cl2)
// Xn2^T diag(cn2)], with search (uniform) without an attempt on the diagonal;
// whether the diagonal's pivots were taken (uniform)
template <int NB, int SEARCH>
__device__ __forceinline__ bool blk_invert_schur(int ni, const double *__restrict__ Dl, const double *cl,
                                                 const double *Xn, const double *cn, const double *cl2,
                                                 const double *Xn2, const double *cn2, double *__restrict__ X,
                                                 BlkShared<NB> &sh, int tag, bool search = false) {
    f64x4 acc[BlkGrid<NB>::TBR][BlkGrid<NB>::TBC];
    if constexpr (SEARCH != BLK_SEARCH_ONLY) {
        if (!search) {
            blk_load_schur<NB>(acc, ni, Dl, cl, Xn, cn, cl2, Xn2, cn2);
            if (blk_invert_diag<NB>(acc, ni, X, sh)) return true;
        }
        if constexpr (SEARCH == BLK_SEARCH_MARK) {
            if (threadIdx.x == 0) blk_mark(X);
            return false;
        }
    }
    blk_load_schur<NB>(acc, ni, Dl, cl, Xn, cn, cl2, Xn2, cn2);
    blk_invert<NB>(acc, ni, X, sh, tag);
    return false;
}

// acc = D_l - diag(cl) acc diag(cn) in the tile layout, acc holding the
// neighbour's inverse as blk_invert_diag leaves it (no pivot order to undo):
// blk_load_schur without reading that inverse back (a chain step of the
// 256-column batch 39.8 -> 36.8 us, of 80 150-species columns 110 -> 101 us).
// All of D's loads are issued before the first product; padding as there.
template <int NB>
__device__ __forceinline__ void blk_next_schur(f64x4 (&acc)[BlkGrid<NB>::TBR][BlkGrid<NB>::TBC], int ni,
                                               const double *__restrict__ Dl, const double *cl, const double *cn) {
    using G = BlkGrid<NB>;
    constexpr int TBR = G::TBR, TBC = G::TBC, WC = G::WC;
    // row tiles in flight together: their D entries beside acc's own
    constexpr int GR = TBR * TBC <= 9 ? TBR : 2;
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));   // as in blk_load_schur
    const int w = tid >> 6, l = tid & 63;
    const int wr = w / WC, wc = w % WC;
    const int lg = l >> 4, lc = l & 15;
    int cj[TBC];
    unsigned long long cm[TBC];
    double cnv[TBC];
#pragma unroll
    for (int tj = 0; tj < TBC; tj++) {
        const int bj = wc + WC * tj, cc = 16 * bj + lc;
        const bool ok = bj < NB && cc < ni;
        cj[tj] = ok ? cc : 0;
        cm[tj] = ok ? ~0ull : 0ull;
        cnv[tj] = cn[cj[tj]];
    }
#pragma unroll
    for (int t0 = 0; t0 < TBR; t0 += GR) {
        double li[GR][4], d[GR][4][TBC];
        unsigned long long rm[GR][4];
#pragma unroll
        for (int g = 0; g < GR; g++) {
            if (t0 + g >= TBR) continue;
            const int bi = wr + 2 * (t0 + g);
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int i = 16 * bi + 4 * r + lg;
                const bool rok = bi < NB && i < ni;
                const int ir = rok ? i : 0;
                rm[g][r] = rok ? ~0ull : 0ull;
                li[g][r] = cl[ir];
#pragma unroll
                for (int tj = 0; tj < TBC; tj++) d[g][r][tj] = Dl[(size_t)ir * ni + cj[tj]];
            }
        }
#pragma unroll
        for (int g = 0; g < GR; g++) {
            if (t0 + g >= TBR) continue;
#pragma unroll
            for (int r = 0; r < 4; r++)
#pragma unroll
                for (int tj = 0; tj < TBC; tj++)
                    acc[t0 + g][tj][r] = blk_masked(d[g][r][tj] - li[g][r] * (acc[t0 + g][tj][r] * cnv[tj]),
                                                    rm[g][r] & cm[tj]);
        }
    }
}

// Products for the cyclic-reduction updates, one 32-row output slab (and
// the 16 NB output columns from c0) per workgroup, two products at a time:
//     acc1 += A1[r0:r0+32, :] B1[:, c0:],   acc2 (or acc1 if SAME) += A2[r0:r0+32, :] B2[:, c0:]
// over k < ni, with every operand stored transposed:
//     A(a, c) = At[c*ni + a],  B(c, b) = Bt[b*ni + c].
// A null A2 skips the second product.  Output tiles are 16 x 16 (MFMA C
// layout: lane l, register r holds row 4r + l/16, column l%16 of the tile);
// wave w owns row block w & 1 of the slab and column blocks (w >> 1) + 2t.
// K runs in chunks of KC staged through LDS; the next chunk's global loads
// are issued into registers before the current chunk's MFMAs, and each
// chunk is read with the operand's unit-stride index fastest across threads
// (A: the row a, B: the inner index c).  Each chunk costs about one global
// load latency, so deep chunks suit launches whose workgroups are all
// resident at once, shallow ones keep more workgroups per CU resident.
// Two staged operand pairs take 16 KC (34 + 16 NB) bytes of LDS (NB: the
// slab's column blocks); SlabKC is indexed by the block's column blocks.
template <int NB>
struct SlabKC {
    static constexpr int shallow = NB <= 7 ? 24 : 16;   // <= 56 KiB
    static constexpr int deep = NB <= 6 ? 48 : 32;      // <= 98 KiB (gfx950: 160 KiB per workgroup)
};

template <int NB, int KC>
struct SlabShared {
    double sa[2][KC][33];
    double sb[2][KC][16 * NB + 1];
};

template <int NB, int KC>
struct SlabRegs {
    static_assert(KC % 8 == 0, "chunk depth: a multiple of 8");
    static constexpr int PA = KC * 32 / NT, PB = (KC * 16 * NB + NT - 1) / NT;
    double a[2][PA], b[2][PB];
};

template <int NB, int KC>
__device__ __forceinline__ void slab_load(SlabRegs<NB, KC> &R, int u, int ni, int r0, int k0,
                                          const double *__restrict__ At, const double *__restrict__ Bt, int c0) {
#pragma unroll
    for (int q = 0; q < SlabRegs<NB, KC>::PA; q++) {
        const int e = threadIdx.x + NT * q, k = e >> 5, r = e & 31;   // a = r0 + r fastest
        const int a = r0 + r, c = k0 + k;
        R.a[u][q] = (a < ni && c < ni) ? At[(size_t)c * ni + a] : 0.0;
    }
#pragma unroll
    for (int q = 0; q < SlabRegs<NB, KC>::PB; q++) {
        const int e = threadIdx.x + NT * q, r = e / KC, k = e - r * KC;   // c = k0 + k fastest
        const int c = k0 + k, b = c0 + r;
        R.b[u][q] = (e < KC * 16 * NB && b < ni && c < ni) ? Bt[(size_t)b * ni + c] : 0.0;
    }
}

template <int NB, int KC>
__device__ __forceinline__ void slab_stage(const SlabRegs<NB, KC> &R, int u, SlabShared<NB, KC> &g) {
#pragma unroll
    for (int q = 0; q < SlabRegs<NB, KC>::PA; q++) {
        const int e = threadIdx.x + NT * q;
        g.sa[u][e >> 5][e & 31] = R.a[u][q];
    }
#pragma unroll
    for (int q = 0; q < SlabRegs<NB, KC>::PB; q++) {
        const int e = threadIdx.x + NT * q, r = e / KC;
        if (e < KC * 16 * NB) g.sb[u][e - r * KC][r] = R.b[u][q];
    }
}

template <int NB, bool SAME, int KC>
__device__ __forceinline__ void slab_gemm2(f64x4 (&acc1)[(NB + 1) / 2], f64x4 (&acc2)[(NB + 1) / 2], int ni, int r0,
                                           const double *__restrict__ A1, const double *__restrict__ B1,
                                           const double *__restrict__ A2, const double *__restrict__ B2,
                                           SlabShared<NB, KC> &g, int c0) {
    constexpr int TB = (NB + 1) / 2;
    const int w = threadIdx.x >> 6, l = threadIdx.x & 63;
    const int bi = w & 1, wc = w >> 1, lc = l & 15, lk = l >> 4;
    const int nch = (ni + KC - 1) / KC;
    const bool two = A2 != nullptr;
    SlabRegs<NB, KC> R;
    slab_load<NB, KC>(R, 0, ni, r0, 0, A1, B1, c0);
    if (two) slab_load<NB, KC>(R, 1, ni, r0, 0, A2, B2, c0);
    for (int ch = 0; ch < nch; ch++) {
        __syncthreads();   // the previous chunk's reads of g are done
        slab_stage<NB, KC>(R, 0, g);
        if (two) slab_stage<NB, KC>(R, 1, g);
        __syncthreads();
        if (ch + 1 < nch) {
            slab_load<NB, KC>(R, 0, ni, r0, (ch + 1) * KC, A1, B1, c0);
            if (two) slab_load<NB, KC>(R, 1, ni, r0, (ch + 1) * KC, A2, B2, c0);
        }
#pragma unroll
        for (int k4 = 0; k4 < KC / 4; k4++) {
            const double a1 = g.sa[0][4 * k4 + lk][16 * bi + lc];
#pragma unroll
            for (int tj = 0; tj < TB; tj++) {
                const int bj = wc + 2 * tj;
                if (bj >= NB) continue;
                acc1[tj] = __builtin_amdgcn_mfma_f64_16x16x4f64(a1, g.sb[0][4 * k4 + lk][16 * bj + lc], acc1[tj], 0, 0,
                                                                 0);
            }
            if (two) {
                const double a2 = g.sa[1][4 * k4 + lk][16 * bi + lc];
#pragma unroll
                for (int tj = 0; tj < TB; tj++) {
                    const int bj = wc + 2 * tj;
                    if (bj >= NB) continue;
                    if (SAME)
                        acc1[tj] = __builtin_amdgcn_mfma_f64_16x16x4f64(a2, g.sb[1][4 * k4 + lk][16 * bj + lc],
                                                                         acc1[tj], 0, 0, 0);
                    else
                        acc2[tj] = __builtin_amdgcn_mfma_f64_16x16x4f64(a2, g.sb[1][4 * k4 + lk][16 * bj + lc],
                                                                         acc2[tj], 0, 0, 0);
                }
            }
        }
    }
    __syncthreads();
}

template <int NB>
__device__ __forceinline__ void slab_zero(f64x4 (&acc)[(NB + 1) / 2]) {
#pragma unroll
    for (int tj = 0; tj < (NB + 1) / 2; tj++) acc[tj] = f64x4{0.0, 0.0, 0.0, 0.0};
}

// out(i, c) = sgn * acc (+ add(i, c) if add) for the slab rows i and the
// columns c0 .. c0 + 16 NB - 1, ni x ni, stored row-major (out[i*ni + c])
// or transposed (out[c*ni + i])
template <int NB>
__device__ __forceinline__ void slab_store(const f64x4 (&acc)[(NB + 1) / 2], int ni, int r0, double *__restrict__ out,
                                           bool transposed, double sgn, const double *add, int c0) {
    const int w = threadIdx.x >> 6, l = threadIdx.x & 63;
    const int bi = w & 1, wc = w >> 1, lg = l >> 4, lc = l & 15;
#pragma unroll
    for (int tj = 0; tj < (NB + 1) / 2; tj++) {
        const int bj = wc + 2 * tj, cc = c0 + 16 * bj + lc;
        if (bj >= NB || cc >= ni) continue;
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int i = r0 + 16 * bi + 4 * r + lg;
            if (i < ni) {
                const size_t e = transposed ? (size_t)cc * ni + i : (size_t)i * ni + cc;
                out[e] = add ? add[e] + sgn * acc[tj][r] : sgn * acc[tj][r];
            }
        }
    }
}

}  // namespace
