// Warm-start MLP kernels: BF16 MFMA GEMM with FP32 accumulation and the
// elementwise pieces of forward, backward and Adam.
//
// GEMM: C[M][N] (fp32) = A(m,k) * B(k,n) (+ bias[n]) with A, B BF16 at
// arbitrary (row, column) strides, so that X*W, dZ*W^T and X^T*dZ share one
// interface.  Operands with a unit stride go to k_gemm_tiled, others to
// k_gemm_any.  Both run v_mfma_f32_32x32x8_bf16 over k in the same order,
// so an output's bits do not depend on which one, or which tile, formed it.
// Optional fused epilogue: Y = SiLU(C) written as BF16 for the next layer.
#include "vk_internal.h"

namespace {

typedef short bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

__device__ __forceinline__ unsigned short f2bf(float f) {
    unsigned int u = __float_as_uint(f);
    if ((u & 0x7fffffffu) > 0x7f800000u) return (unsigned short)((u >> 16) | 0x40);   // NaN stays NaN
    u += 0x7fffu + ((u >> 16) & 1u);                                                   // round to nearest even
    return (unsigned short)(u >> 16);
}

__device__ __forceinline__ float bf2f(unsigned short h) { return __uint_as_float(((unsigned int)h) << 16); }

__device__ __forceinline__ float silu(float z) { return z / (1.0f + expf(-z)); }

// Epilogue of a wave's 32 x 32 tile at (m0, n0): acc[q] is row 8*(q/4) +
// 4*(lane/32) + q%4, column lane%32
__device__ __forceinline__ void store_tile(const f32x16 &acc, int M, int N, int m0, int n0, int lane,
                                           float *__restrict__ C, long ldc, const float *__restrict__ bias,
                                           int accumulate, unsigned short *__restrict__ Yact, long ldy) {
    const int col = n0 + (lane & 31);
    if (col >= N) return;
    const float bc = bias ? bias[col] : 0.0f;
    float *cp = C + (long)(m0 + 4 * (lane >> 5)) * ldc + col;
    if (!accumulate && !Yact) {
#pragma unroll
        for (int q = 0; q < 16; q++) {
            const int r = 8 * (q >> 2) + (q & 3);
            if (m0 + 4 * (lane >> 5) + r < M) cp[(long)r * ldc] = bias ? acc[q] + bc : acc[q];
        }
        return;
    }
#pragma unroll
    for (int q = 0; q < 16; q++) {
        const int r = 8 * (q >> 2) + (q & 3), row = m0 + 4 * (lane >> 5) + r;
        if (row < M) {
            float v = bias ? acc[q] + bc : acc[q];
            if (accumulate) v += cp[(long)r * ldc];
            cp[(long)r * ldc] = v;
            if (Yact) Yact[(long)row * ldy + col] = f2bf(silu(v));
        }
    }
}

constexpr int TM = 64, TN = 64, TK = 32, KP = TK + 4;   // LDS row pitch (in bf16) avoids bank conflicts

__global__ void __launch_bounds__(256) k_gemm_any(int M, int N, int K, const unsigned short *__restrict__ A, long sam,
                                                  long sak, const unsigned short *__restrict__ B, long sbk, long sbn,
                                                  float *__restrict__ C, long ldc, const float *__restrict__ bias,
                                                  int accumulate, unsigned short *__restrict__ Yact, long ldy) {
    __shared__ unsigned short As[TM][KP];
    __shared__ unsigned short Bs[TN][KP];
    const int tid = threadIdx.x;
    const int wave = tid >> 6, lane = tid & 63;
    const int m0 = blockIdx.y * TM, n0 = blockIdx.x * TN;
    const int wm = (wave >> 1) * 32, wn = (wave & 1) * 32;
    f32x16 acc;
    for (int q = 0; q < 16; q++) acc[q] = 0.0f;
    const bool a_kfast = (sak == 1);
    const bool b_kfast = (sbk == 1);
    for (int k0 = 0; k0 < K; k0 += TK) {
        // A tile: 64 x 32 elements, 8 per thread; consecutive threads walk the unit-stride dimension
        for (int e = tid; e < TM * TK; e += 256) {
            int r, kk;
            if (a_kfast) { r = e / TK; kk = e % TK; } else { kk = e / TM; r = e % TM; }
            const int gm = m0 + r, gk = k0 + kk;
            As[r][kk] = (gm < M && gk < K) ? A[(long)gm * sam + (long)gk * sak] : (unsigned short)0;
        }
        for (int e = tid; e < TN * TK; e += 256) {
            int c, kk;
            if (b_kfast) { c = e / TK; kk = e % TK; } else { kk = e / TN; c = e % TN; }
            const int gn = n0 + c, gk = k0 + kk;
            Bs[c][kk] = (gn < N && gk < K) ? B[(long)gk * sbk + (long)gn * sbn] : (unsigned short)0;
        }
        __syncthreads();
#pragma unroll
        for (int kk = 0; kk < TK; kk += 8) {
            const int kq = kk + (lane >> 5) * 4;
            bf16x4 a, b;
            const unsigned short *pa = &As[wm + (lane & 31)][kq];
            const unsigned short *pb = &Bs[wn + (lane & 31)][kq];
            a[0] = pa[0]; a[1] = pa[1]; a[2] = pa[2]; a[3] = pa[3];
            b[0] = pb[0]; b[1] = pb[1]; b[2] = pb[2]; b[3] = pb[3];
            acc = __builtin_amdgcn_mfma_f32_32x32x8bf16_1k(a, b, acc, 0, 0, 0);
        }
        __syncthreads();
    }
    store_tile(acc, M, N, m0 + wm, n0 + wn, lane, C, ldc, bias, accumulate, Yact, ldy);
}

// ---------------------------------------------------------------------------
// The same product with both operands' unit-stride dimension read in 8- and
// 16-byte loads.  A workgroup forms a BM x BN tile of C, each computing wave
// WM x WN of it; all four waves stage.  K runs in chunks of KC through two
// LDS buffers, one barrier a chunk, with the next two chunks' loads in
// registers.  LDS holds both operands row by row
// (row: m or n) with the 4-entry pieces of every 16 k in the order 0 2 1 3
// (Stage::at), so that one 16-byte read gives a lane its operands of two
// MFMAs.  An operand whose rows are the unit stride is transposed 4 x 4 in
// registers on the way.
//
// An output's sum over k is one serial chain of MFMAs (32 cycles per 8 k), so
// the tile decides how many CUs a product fills: 32 x 32 tiles, one
// computing wave, when 64 x 64 ones would leave CUs without work, and
// 128 x 64 ones, fewer LDS reads per MFMA, when there are two for each CU.
//
// Measured against k_gemm_any (two-byte loads, 64 x 64 tiles) at 256 rows:
// 1024 x 1024 layers 123 -> 11 us (64 of the 256 CUs worked), the 1024 x
// 13 950 head 198 -> 38 us, its weight gradient 157 -> 49 us, a training step
// of the 307 -> 4 x 1024 -> 13 950 network 3.60 -> 0.47 ms.  The head's input
// gradient (k = 13 950 on 32 x 32 tiles, 70 us) is 1 744 dependent MFMAs on one
// wave of four; at 32 cycles each these are 23 us, and a chunk's barrier, its
// LDS reads and the staging by the same wave lie between them.
// ---------------------------------------------------------------------------
struct GemmArgs {
    int M, N, K;
    const unsigned short *A, *B;
    long lda, ldb;               // stride of the dimension that is not the unit one
    float *C;
    long ldc;
    const float *bias;
    int accumulate;
    unsigned short *Yact;
    long ldy;
};

// staging registers and steps of one operand: R rows x KC; KFAST: k is the unit stride
template <int R, int KC, bool KFAST>
struct Stage {
    static constexpr int PITCH = KC + 8;            // in entries: rows 16 bytes past a multiple of 128
    static constexpr int UNITS = KFAST ? R * KC / 8 : R * KC / 16, PER = (UNITS + 255) / 256;
    uint2 v[PER][KFAST ? 2 : 4];

    // four or eight entries of a unit: whole vectors inside the operand; a
    // tile or chunk at its edge (a uniform test) reads entry by entry with
    // the indices clamped and zeroes what lies past it, without branches
    __device__ __forceinline__ void load(const unsigned short *__restrict__ X, long ld, int rows, int K, int r0, int k0) {
        const bool inside = r0 + R <= rows && k0 + KC <= K;
        if (inside) {
#pragma unroll
            for (int q = 0; q < PER; q++) {
                const int u = unit(q);
                if constexpr (KFAST) {
                    uint4 w;
                    __builtin_memcpy(&w, X + (long)(r0 + u / (KC / 8)) * ld + k0 + 8 * (u % (KC / 8)), 16);
                    v[q][0] = make_uint2(w.x, w.y);
                    v[q][1] = make_uint2(w.z, w.w);
                } else {
#pragma unroll
                    for (int i = 0; i < 4; i++)
                        __builtin_memcpy(&v[q][i], X + (long)(k0 + 4 * (u / (R / 4)) + i) * ld + r0 + 4 * (u % (R / 4)), 8);
                }
            }
            return;
        }
#pragma unroll
        for (int q = 0; q < PER; q++) {
            const int u = unit(q);
            if constexpr (KFAST) {
                const int r = r0 + u / (KC / 8), k = k0 + 8 * (u % (KC / 8));
                const unsigned short *p = X + (long)min(r, rows - 1) * ld;
                unsigned short e[8];
#pragma unroll
                for (int i = 0; i < 8; i++) e[i] = p[min(k + i, K - 1)];
#pragma unroll
                for (int i = 0; i < 8; i++) e[i] = r < rows && k + i < K ? e[i] : (unsigned short)0;
                __builtin_memcpy(&v[q][0], e, 8);
                __builtin_memcpy(&v[q][1], e + 4, 8);
            } else {
                const int r = r0 + 4 * (u % (R / 4)), k = k0 + 4 * (u / (R / 4));
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    const unsigned short *p = X + (long)min(k + i, K - 1) * ld;
                    unsigned short e[4];
#pragma unroll
                    for (int j = 0; j < 4; j++) e[j] = p[min(r + j, rows - 1)];
#pragma unroll
                    for (int j = 0; j < 4; j++) e[j] = k + i < K && r + j < rows ? e[j] : (unsigned short)0;
                    __builtin_memcpy(&v[q][i], e, 8);
                }
            }
        }
    }

    // threads past the last unit stage one that another thread stages too
    static __device__ __forceinline__ int unit(int q) {
        const int u = threadIdx.x + 256 * q;
        return UNITS % 256 != 0 ? u % UNITS : u;
    }

    // entry of the 4-entry piece c (k = 4 c ..) of a row: 16-byte granules of
    // two pieces, a granule's place exchanged within four by bits 4 and 5 of
    // the row (the transposing stores write rows 4 apart, whose banks repeat
    // every 16 rows without it: 8 conflict cycles an access; the reads of 16
    // consecutive rows stay free of conflicts)
    static __device__ __forceinline__ int at(int r, int c) {
        return r * PITCH + 8 * (((c >> 2) * 2 + (c & 1)) ^ ((r >> 4) & 3)) + 4 * ((c >> 1) & 1);
    }

    __device__ __forceinline__ void store(unsigned short *sm) const {
#pragma unroll
        for (int q = 0; q < PER; q++) {
            const int u = unit(q);
            if constexpr (KFAST) {
                const int r = u / (KC / 8), c = 2 * (u % (KC / 8));
                *(uint2 *)(sm + at(r, c)) = v[q][0];
                *(uint2 *)(sm + at(r, c + 1)) = v[q][1];
            } else {
                const int r = 4 * (u % (R / 4)), c = u / (R / 4);
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    // entry j of the four k rows
                    const unsigned sel = j & 1 ? 0x07060302u : 0x05040100u;
                    const unsigned x0 = j < 2 ? v[q][0].x : v[q][0].y, x1 = j < 2 ? v[q][1].x : v[q][1].y;
                    const unsigned x2 = j < 2 ? v[q][2].x : v[q][2].y, x3 = j < 2 ? v[q][3].x : v[q][3].y;
                    *(uint2 *)(sm + at(r + j, c)) =
                        make_uint2(__builtin_amdgcn_perm(x1, x0, sel), __builtin_amdgcn_perm(x3, x2, sel));
                }
            }
        }
    }
};

template <int BM, int BN, int WM, int WN, int KC, bool AK, bool BK>
__global__ void __launch_bounds__(256, BM == 128 ? 2 : 4) k_gemm_tiled(GemmArgs g) {
    using SA = Stage<BM, KC, AK>;
    using SB = Stage<BN, KC, BK>;
    constexpr int P = SA::PITCH, TA = WM / 32, TB = WN / 32, WX = BN / WN, NWC = (BM / WM) * WX;
    static_assert(NWC <= 4, "four waves");
    __shared__ __align__(16) unsigned short sm[2][(BM + BN) * P];
    // workgroups go to the 8 XCDs in turn: each XCD takes a contiguous range
    // of tiles, m fastest, so that the tiles sharing B's columns share an L2
    const int tm = (g.M + BM - 1) / BM, tiles = tm * ((g.N + BN - 1) / BN), per = (tiles + 7) / 8;
    const int t = (int)(blockIdx.x % 8) * per + (int)(blockIdx.x / 8);
    if ((int)(blockIdx.x / 8) >= per || t >= tiles) return;
    const int m0 = BM * (t % tm), n0 = BN * (t / tm);
    const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int wm = WM * (w / WX), wn = WN * (w % WX);
    const bool computes = NWC == 4 || w < NWC;
    f32x16 acc[TA][TB];
#pragma unroll
    for (int i = 0; i < TA; i++)
#pragma unroll
        for (int j = 0; j < TB; j++)
#pragma unroll
            for (int q = 0; q < 16; q++) acc[i][j][q] = 0.0f;
    // a lane's operands of two MFMAs (16 k from k) of the 32 rows from r0
    auto operand = [&](int r0, int k) {
        const int r = r0 + (lane & 31);
        return r * P + 8 * ((k / 8 + (lane >> 5)) ^ ((r >> 4) & 3));
    };
    // chunk c + 1 waits in registers while chunk c is multiplied, c + 2 is in
    // flight
    constexpr int AHEAD = 2;
    SA sa[AHEAD];
    SB sb[AHEAD];
    const int nch = (g.K + KC - 1) / KC;
    auto load = [&](int slot, int c) {
        if (c < nch) {
            sa[slot].load(g.A, g.lda, g.M, g.K, m0, c * KC);
            sb[slot].load(g.B, g.ldb, g.N, g.K, n0, c * KC);
        }
    };
#pragma unroll
    for (int d = 0; d < AHEAD; d++) load(d, d);
    sa[0].store(sm[0]);
    sb[0].store(sm[0] + BM * P);
    load(0, AHEAD);
    for (int c0 = 0; c0 < nch; c0 += AHEAD) {
#pragma unroll
        for (int d = 0; d < AHEAD; d++) {
            const int c = c0 + d, slot = (d + 1) % AHEAD;
            if (c >= nch) break;
            // the other buffer's readers (chunk c - 1) are past this barrier
            __syncthreads();
            if (computes) {
                const unsigned short *pa = sm[c & 1], *pb = pa + BM * P;
#pragma unroll
                for (int k = 0; k < KC; k += 16) {
                    bf16x4 a[TA][2], b[TB][2];
#pragma unroll
                    for (int i = 0; i < TA; i++)
                        __builtin_memcpy(a[i], __builtin_assume_aligned(pa + operand(wm + 32 * i, k), 16), 16);
#pragma unroll
                    for (int j = 0; j < TB; j++)
                        __builtin_memcpy(b[j], __builtin_assume_aligned(pb + operand(wn + 32 * j, k), 16), 16);
#pragma unroll
                    for (int h = 0; h < 2; h++)
#pragma unroll
                        for (int i = 0; i < TA; i++)
#pragma unroll
                            for (int j = 0; j < TB; j++)
                                acc[i][j] =
                                    __builtin_amdgcn_mfma_f32_32x32x8bf16_1k(a[i][h], b[j][h], acc[i][j], 0, 0, 0);
                }
            }
            if (c + 1 < nch) {
                sa[slot].store(sm[(c + 1) & 1]);
                sb[slot].store(sm[(c + 1) & 1] + BM * P);
                load(slot, c + 1 + AHEAD);
            }
        }
    }
    if (computes)
#pragma unroll
        for (int i = 0; i < TA; i++)
#pragma unroll
            for (int j = 0; j < TB; j++)
                store_tile(acc[i][j], g.M, g.N, m0 + wm + 32 * i, n0 + wn + 32 * j, lane, g.C, g.ldc, g.bias,
                           g.accumulate, g.Yact, g.ldy);
}

template <int BM, int BN, int WM, int WN, int KC>
void launch_gemm(const GemmArgs &g, bool ak, bool bk, hipStream_t s) {
    const long tiles = (long)((g.M + BM - 1) / BM) * ((g.N + BN - 1) / BN);
    const dim3 grid((unsigned)(8 * ((tiles + 7) / 8)));
    if (ak && bk) hipLaunchKernelGGL((k_gemm_tiled<BM, BN, WM, WN, KC, true, true>), grid, dim3(256), 0, s, g);
    else if (ak) hipLaunchKernelGGL((k_gemm_tiled<BM, BN, WM, WN, KC, true, false>), grid, dim3(256), 0, s, g);
    else if (bk) hipLaunchKernelGGL((k_gemm_tiled<BM, BN, WM, WN, KC, false, true>), grid, dim3(256), 0, s, g);
    else hipLaunchKernelGGL((k_gemm_tiled<BM, BN, WM, WN, KC, false, false>), grid, dim3(256), 0, s, g);
}

// dZ = dY * silu'(Z), written as fp32 and BF16; silu'(z) = s (1 + z (1 - s)), s = sigmoid(z)
__global__ void k_silu_bwd(long n, const float *__restrict__ Z, const float *__restrict__ dY, float *__restrict__ dZ,
                           unsigned short *__restrict__ dZb) {
    long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float z = Z[i];
    const float s = 1.0f / (1.0f + expf(-z));
    const float d = dY[i] * (s * (1.0f + z * (1.0f - s)));
    dZ[i] = d;
    dZb[i] = f2bf(d);
}

// MSE over masked entries: dY = 2 w (Y - T) / count (fp32 + BF16), loss partials per block
__global__ void k_mse(long n, const float *__restrict__ Y, const float *__restrict__ T,
                      const float *__restrict__ W, float inv_count, float *__restrict__ dY,
                      unsigned short *__restrict__ dYb, float *__restrict__ loss_part) {
    __shared__ float red[256];
    long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    float l = 0.0f;
    if (i < n) {
        const float w = W ? W[i] : 1.0f;
        const float d = Y[i] - T[i];
        const float g = 2.0f * w * d * inv_count;
        dY[i] = g;
        dYb[i] = f2bf(g);
        l = w * d * d * inv_count;
    }
    red[threadIdx.x] = l;
    __syncthreads();
    for (int s = 128; s > 0; s >>= 1) {
        if (threadIdx.x < s) red[threadIdx.x] += red[threadIdx.x + s];
        __syncthreads();
    }
    if (threadIdx.x == 0) loss_part[blockIdx.x] = red[0];
}

// column sums: out[n] = sum_m X[m][n]  (bias gradients), in order of m.  One
// thread per column, one wave per workgroup (a hidden layer's 1024 columns
// on 16 CUs), 16 rows' loads in flight ahead of their sums: a load at a time
// took a memory round trip per row (26 us for 256 x 1024).
__global__ void __launch_bounds__(64) k_colsum(int M, int N, const float *__restrict__ X, float *__restrict__ out) {
    const int n = blockIdx.x * 64 + threadIdx.x;
    if (n >= N) return;
    const float *p = X + n;
    float s = 0.0f;
    int m = 0;
    for (; m + 16 <= M; m += 16) {
        float x[16];
#pragma unroll
        for (int i = 0; i < 16; i++) x[i] = p[(long)(m + i) * N];
#pragma unroll
        for (int i = 0; i < 16; i++) s += x[i];
    }
    for (; m < M; m++) s += p[(long)m * N];
    out[n] = s;
}

__global__ void k_to_bf16(long n, const float *__restrict__ x, unsigned short *__restrict__ y) {
    long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) y[i] = f2bf(x[i]);
}

// Adam (Kingma & Ba 2015) on fp32 master weights; refreshes the BF16 copy
__global__ void k_adam(long n, float *__restrict__ w, const float *__restrict__ g, float *__restrict__ m,
                       float *__restrict__ v, float lr, float b1, float b2, float eps, float c1, float c2,
                       float wd, unsigned short *__restrict__ wb) {
    long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float gi = g[i] + wd * w[i];
    const float mi = b1 * m[i] + (1.0f - b1) * gi;
    const float vi = b2 * v[i] + (1.0f - b2) * gi * gi;
    m[i] = mi;
    v[i] = vi;
    const float wi = w[i] - lr * (mi / c1) / (sqrtf(vi / c2) + eps);
    w[i] = wi;
    if (wb) wb[i] = f2bf(wi);
}

inline dim3 grid1(long n) { return dim3((unsigned)((n + 255) / 256)); }

}  // namespace

extern "C" int vk_mlp_gemm(int M, int N, int K, const void *d_A, long sam, long sak, const void *d_B, long sbk,
                           long sbn, float *d_C, long ldc, const float *d_bias, int accumulate, void *d_Yact,
                           long ldy, void *stream) {
    if (M <= 0 || N <= 0 || K <= 0 || !d_A || !d_B || !d_C) return VK_EINVAL;
    hipStream_t s = (hipStream_t)stream;
    // The tiled kernel where each operand has a unit stride.  Its chunks are 64 or
    // 128 deep; with a product less deep, many outputs are faster through
    // k_gemm_any, 32 at a time (1024 x 13 950 outputs, k = 8, 32, 48, 63, 64, 96: 20,
    // 23, 32, 34, 34, 46 us against 36, 37, 38, 40, 30, 41; 1024 x 1024, k = 32, 48:
    // 9.8, 10.6 against 9.0, 8.9).
    const bool ak = sak == 1, am = sam == 1, bk = sbk == 1, bn = sbn == 1;
    const long t64 = (long)((M + 63) / 64) * ((N + 63) / 64), t128 = (long)((M + 127) / 128) * ((N + 63) / 64);
    const int ncu = vk_device_cus();
    const bool shallow = K < 64 && t64 >= 2L * ncu && (M + TM - 1) / TM <= 65535;
    if ((ak || am) && (bk || bn) && !shallow) {
        const GemmArgs g = {M, N, K, (const unsigned short *)d_A, (const unsigned short *)d_B, ak ? sam : sak,
                            bk ? sbn : sbk, d_C, ldc, d_bias, accumulate, (unsigned short *)d_Yact, ldy};
        // 128 rows a tile only where at most an eighth of them lies past the
        // last row (64 x 262 144 outputs, k = 128: FIGM)
        if (t128 >= 2L * ncu && 8 * (2 * t128 - t64) <= t64) launch_gemm<128, 64, 64, 32, 64>(g, ak, bk, s);
        else if (t64 >= ncu) launch_gemm<64, 64, 32, 32, 64>(g, ak, bk, s);
        else launch_gemm<32, 32, 32, 32, 128>(g, ak, bk, s);
    } else {
        dim3 grid((N + TN - 1) / TN, (M + TM - 1) / TM);
        hipLaunchKernelGGL(k_gemm_any, grid, dim3(256), 0, s, M, N, K, (const unsigned short *)d_A, sam, sak,
                           (const unsigned short *)d_B, sbk, sbn, d_C, ldc, d_bias, accumulate,
                           (unsigned short *)d_Yact, ldy);
    }
    VK_CHECK(hipGetLastError());
    return 0;
}

extern "C" int vk_mlp_silu_bwd(long n, const float *d_Z, const float *d_dY, float *d_dZ, void *d_dZb, void *stream) {
    if (n <= 0 || !d_Z || !d_dY || !d_dZ || !d_dZb) return VK_EINVAL;
    hipLaunchKernelGGL(k_silu_bwd, grid1(n), dim3(256), 0, (hipStream_t)stream, n, d_Z, d_dY, d_dZ,
                       (unsigned short *)d_dZb);
    VK_CHECK(hipGetLastError());
    return 0;
}

extern "C" int vk_mlp_mse(long n, const float *d_Y, const float *d_T, const float *d_W, float inv_count, float *d_dY,
                          void *d_dYb, float *d_loss_part, void *stream) {
    if (n <= 0 || !d_Y || !d_T || !d_dY || !d_dYb || !d_loss_part) return VK_EINVAL;
    hipLaunchKernelGGL(k_mse, grid1(n), dim3(256), 0, (hipStream_t)stream, n, d_Y, d_T, d_W, inv_count, d_dY,
                       (unsigned short *)d_dYb, d_loss_part);
    VK_CHECK(hipGetLastError());
    return 0;
}

extern "C" int vk_mlp_colsum(int M, int N, const float *d_X, float *d_out, void *stream) {
    if (M <= 0 || N <= 0 || !d_X || !d_out) return VK_EINVAL;
    hipLaunchKernelGGL(k_colsum, dim3((N + 63) / 64), dim3(64), 0, (hipStream_t)stream, M, N, d_X, d_out);
    VK_CHECK(hipGetLastError());
    return 0;
}

extern "C" int vk_mlp_to_bf16(long n, const float *d_x, void *d_y, void *stream) {
    if (n <= 0 || !d_x || !d_y) return VK_EINVAL;
    hipLaunchKernelGGL(k_to_bf16, grid1(n), dim3(256), 0, (hipStream_t)stream, n, d_x, (unsigned short *)d_y);
    VK_CHECK(hipGetLastError());
    return 0;
}

extern "C" int vk_mlp_adam(long n, float *d_w, const float *d_g, float *d_m, float *d_v, float lr, float b1,
                           float b2, float eps, int step, float wd, void *d_wb, void *stream) {
    if (n <= 0 || !d_w || !d_g || !d_m || !d_v || step < 1) return VK_EINVAL;
    const float c1 = 1.0f - powf(b1, (float)step), c2 = 1.0f - powf(b2, (float)step);
    hipLaunchKernelGGL(k_adam, grid1(n), dim3(256), 0, (hipStream_t)stream, n, d_w, d_g, d_m, d_v, lr, b1, b2, eps,
                       c1, c2, wd, (unsigned short *)d_wb);
    VK_CHECK(hipGetLastError());
    return 0;
}
