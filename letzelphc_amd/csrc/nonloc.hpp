// nonloc.hpp -- Kleinman-Bylander part of g: add_elphNonLocal
// (src/nonloc/Vbare_nloc.c:35-577) and sum_VNL_KKp
// (src/nonloc/sum_VNL_KKp.c:8-58).
//
// Per side, K = S(k+G) cartesian without 2pi (nlbatch.hpp: all sides of many
// pairs at once):
//   1. k_nl_sides  : the rotated coefficients (su2, translation phase
//                    e^{-i 2pi K.tau}) and beta[a][p][x][G] = F_l(K)
//                    e^{-i 2pi K.tau_a} Y_lm(K) {1, sign K_x,y,z}, phases and
//                    tables in FP64
//   2. k_nl_gemm   : <beta|psi> on MFMA (zgemm_nt_body; conjugation by time
//                    reversal, Vbare_nloc.c:397-418), k_nl_reduce
//   3. k_nl_kkp    : the 4-term K/K' sum per atom (sum_VNL_KKp)
//   4. k_nl_mode   : cart -> mode with prefactor -2 pi i e^2, accumulated
//                    onto g (Vbare_nloc.c:541-558)
#pragma once

#include "common.hpp"
#include "contract.hpp"

__device__ inline double d_fact(int n)
{
    double f = 1.0;
    for (int i = 2; i <= n; ++i) f *= i;
    return n < 0 ? 0.0 : f;
}

// legendre (src/common/numerical_func.c:29-94) for m >= 0, as Ylm uses it
__device__ inline double d_legendre(int l, int m, double x)
{
    if (l == 0 && m == 0) return 1.0;
    if (m > l) return 0.0;
    double p = 1.0;
    const double s = sqrt(1 - x * x);
    for (int i = 1; i <= m; ++i) p *= (2 * i - 1) * s;
    if (l == m) return p;
    double pmm = p;
    p *= (2 * m + 1) * x;
    if (l == m + 1) return p;
    for (int i = m + 2; i <= l; ++i)
    {
        double t = p;
        p = (2 * i - 1) * x * p - (i + m - 1) * pmm;
        p = p / (i - m);
        pmm = t;
    }
    return p;
}

// Ylm (src/common/numerical_func.c:97-152): real harmonics, Blanco et al.;
// the direction once, then any number of (l, m)
struct YlmDir
{
    double cost, phi;
    bool zero;
    __device__ explicit YlmDir(const double* v)
    {
        const double nrm = sqrt(v[0] * v[0] + v[1] * v[1] + v[2] * v[2]);
        zero = nrm < LELPH_EPS6;
        cost = zero ? 0.0 : v[2] / nrm;
        phi = zero ? 0.0 : atan2(v[1], v[0]);
    }
};
__device__ inline double d_Ylm(int l, int m, const YlmDir& dir)
{
    if (dir.zero) return l != 0 ? 0.0 : 1.0 / sqrt(4 * LELPH_RPI);
    const double cost = dir.cost, phi = dir.phi;
    double sh;
    if (m > 0)
        sh = sqrt(2.0) * cos(m * phi);
    else if (m < 0)
    {
        m = -m;
        sh = sqrt(2.0) * sin(m * phi);
    }
    else
        sh = 1;
    sh *= d_legendre(l, m, cost);
    sh *= sqrt(d_fact(l - m) * (2 * l + 1) / (4 * LELPH_RPI * d_fact(l + m)));
    return sh;
}

struct NlSide
{
    double S[9];   // cartesian symmetry
    double k[3];   // iBZ k, cartesian no 2pi
    double tau[3]; // fractional translation (cart)
    int conj_w;    // conjugate the wavefunction in the projector GEMM
    z64 su2[4];
};

// projector list of an atom: entry p -> (lidx, l, m index)
struct NlProj
{
    int natom, pmax, ntype;
};

// part[split][M][Nc] = A[M][K] op(B[Nc][K])^T over the split's K range,
// complex; op = conj when conjB.  Block: 64 x 64, 4 waves of 32 x 32; chunks
// of 16 columns of K are loaded a chunk ahead into registers and double
// buffered in LDS (one barrier per chunk).  16 x 16 blocks past the last row
// or column are skipped: a chunk of 64 x 64 is 64 MFMAs of 64 cycles a wave.
#define GZ_MB 64
#define GZ_NB 64
template <typename T>
__device__ __forceinline__ void zgemm_nt_body(gptr<T> A, gptr<T> B, int M, int Nc, int64_t K,
                                              int conjB, int64_t chunks_per_split, z64* part)
{
    typedef typename Mfma<T>::acc acc_t;
    constexpr int KC = 16, LD = KC + 1, L = GZ_MB * KC / 256;
    static_assert(GZ_MB == GZ_NB && KC == CT_KC, "");
    __shared__ cpx<T> sA[2][GZ_MB][LD];
    __shared__ cpx<T> sB[2][GZ_NB][LD];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int ntn = (Nc + GZ_NB - 1) / GZ_NB;
    const int m0 = (blockIdx.x / ntn) * GZ_MB, n0 = (blockIdx.x % ntn) * GZ_NB;
    const int split = blockIdx.y;
    const int64_t nchunks = (K + KC - 1) / KC;
    const int64_t c0 = (int64_t)split * chunks_per_split;
    const int64_t c1 = (c0 + chunks_per_split < nchunks) ? c0 + chunks_per_split : nchunks;
    const int wr_ = wave >> 1, wc = wave & 1, kk = tid % KC;
    bool on[2][2];
    acc_t accr[2][2], acci[2][2];
    for (int a = 0; a < 2; ++a)
        for (int b = 0; b < 2; ++b)
        {
            on[a][b] = m0 + wr_ * 32 + a * 16 < M && n0 + wc * 32 + b * 16 < Nc;
            for (int v = 0; v < 4; ++v)
            {
                accr[a][b][v] = 0;
                acci[a][b][v] = 0;
            }
        }
    const T sgn = conjB ? (T)-1 : (T)1;
    gptr<T> pA[L], pB[L];
#pragma unroll
    for (int u = 0; u < L; ++u)
    {
        const int r = tid / KC + u * (256 / KC);
        pA[u] = A + (int64_t)min(m0 + r, M - 1) * K;
        pB[u] = B + (int64_t)min(n0 + r, Nc - 1) * K;
    }
    cpx<T> ra[L], rb_[L];
    auto fetch = [&](int64_t c) {
        const int64_t k = c * KC + kk;
        const bool in = k < K;
#pragma unroll
        for (int u = 0; u < L; ++u)
        {
            ra[u] = pA[u][in ? k : 0];
            rb_[u] = pB[u][in ? k : 0];
            if (!in)
            {
                ra[u] = {0, 0};
                rb_[u] = {0, 0};
            }
            rb_[u].y *= sgn;
        }
    };
    auto put = [&](int b) {
#pragma unroll
        for (int u = 0; u < L; ++u)
        {
            sA[b][tid / KC + u * (256 / KC)][kk] = ra[u];
            sB[b][tid / KC + u * (256 / KC)][kk] = rb_[u];
        }
    };
    if (c0 < c1)
    {
        fetch(c0);
        put(0);
    }
    lds_barrier();
    for (int64_t c = c0; c < c1; ++c)
    {
        const int bf = (int)(c - c0) & 1;
        if (c + 1 < c1) fetch(c + 1);
#pragma unroll
        for (int s = 0; s < KC / 4; ++s)
        {
            const int i = lane & 15, kq = s * 4 + (lane >> 4);
            cpx<T> a[2], b[2];
            a[0] = sA[bf][wr_ * 32 + i][kq];
            a[1] = sA[bf][wr_ * 32 + 16 + i][kq];
            b[0] = sB[bf][wc * 32 + i][kq];
            b[1] = sB[bf][wc * 32 + 16 + i][kq];
#pragma unroll
            for (int rb = 0; rb < 2; ++rb)
#pragma unroll
                for (int cb = 0; cb < 2; ++cb)
                    if (on[rb][cb])
                    {
                        // C += a b: re = ar br - ai bi, im = ar bi + ai br
                        accr[rb][cb] = Mfma<T>::op(a[rb].x, b[cb].x, accr[rb][cb]);
                        acci[rb][cb] = Mfma<T>::op(a[rb].x, b[cb].y, acci[rb][cb]);
                        accr[rb][cb] = Mfma<T>::op(-a[rb].y, b[cb].y, accr[rb][cb]);
                        acci[rb][cb] = Mfma<T>::op(a[rb].y, b[cb].x, acci[rb][cb]);
                    }
        }
        if (c + 1 < c1) put(bf ^ 1);
        lds_barrier();
    }
    for (int rb = 0; rb < 2; ++rb)
        for (int cb = 0; cb < 2; ++cb)
            for (int e = 0; e < 4; ++e)
            {
                const int row = m0 + wr_ * 32 + rb * 16 + Mfma<T>::row(lane, e);
                const int col = n0 + wc * 32 + cb * 16 + (lane & 15);
                if (row < M && col < Nc)
                    part[((int64_t)split * M + row) * Nc + col] = {(double)accr[rb][cb][e],
                                                                   (double)acci[rb][cb][e]};
            }
}
template <typename T>
__global__ __launch_bounds__(256) void k_zgemm_nt(const cpx<T>* __restrict__ A,
                                                  const cpx<T>* __restrict__ B, int M, int Nc,
                                                  int64_t K, int conjB, int64_t chunks_per_split,
                                                  z64* __restrict__ part)
{
    zgemm_nt_body<T>(gptr<T>::of(A), gptr<T>::of(B), M, Nc, K, conjB, chunks_per_split, part);
}

// Reduced-precision projector GEMMs (the FP32 and BF16-split forms of the
// <beta|psi> products, src/nonloc/Vbare_nloc.c:409-418).  beta (phases and
// radial / Y_lm tables in FP64) and the rotated wavefunctions are split into
// NP bf16 pieces per real component, x = x0 + x1 (+ x2), each the
// round-to-nearest of the remaining FP32 residual, stored as planes
// P[piece][re/im][row][k] with k contiguous and zero padded to Kp (a
// multiple of 32) and rows to Rp (a multiple of 64); negim flips the sign of
// the imaginary planes (the conjugate operand).
template <int NP>
__global__ void k_nl_presplit(const z64* __restrict__ X, int R, int64_t K, int Rp, int64_t Kp,
                              int negim, __bf16* __restrict__ out)
{
    const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int r = blockIdx.y;
    if (k >= Kp || r >= Rp) return;
    z64 v = {0, 0};
    if (r < R && k < K) v = X[(int64_t)r * K + k];
    float re = (float)v.x, im = (float)(negim ? -v.y : v.y);
    const int64_t plane = (int64_t)Rp * Kp;
#pragma unroll
    for (int p = 0; p < NP; ++p)
    {
        const __bf16 a = (__bf16)re, b = (__bf16)im;
        out[(2 * p) * plane + (int64_t)r * Kp + k] = a;
        out[(2 * p + 1) * plane + (int64_t)r * Kp + k] = b;
        re -= (float)a;
        im -= (float)b;
    }
}

typedef __bf16 nl_bf16x8 __attribute__((ext_vector_type(8)));
typedef float nl_flt4 __attribute__((ext_vector_type(4)));

__device__ inline nl_bf16x8 nl_neg(nl_bf16x8 x)
{
    typedef unsigned short u16x8 __attribute__((ext_vector_type(8)));
    u16x8 u = __builtin_bit_cast(u16x8, x);
    u ^= (unsigned short)0x8000;
    return __builtin_bit_cast(nl_bf16x8, u);
}

// C[M][N] (partial of split s) = sum_k A[m][k] B[n][k] over the split's k
// range, complex, from the piece planes of k_nl_presplit (B's imaginary
// planes already carry the conjugation sign): Cr = Ar Br - Ai Bi, Ci = Ar Bi
// + Ai Br, each real product as the piece products p1 + p2 < NP (NPROD 3:
// p1 + p2 <= 1) on v_mfma_f32_16x16x32_bf16, FP32 accumulation within the
// split, partials in FP64.  Block 64 x 64, 4 waves of 32 x 32; fragments are
// read straight from global memory (16 bytes per lane: A lane l holds row
// l % 16, k 8 (l / 16) .. + 7; B the same for column l % 16).
template <int NP, int NPROD>
__global__ __launch_bounds__(256) void k_zgemm_nt_bf(const __bf16* __restrict__ Ap,
                                                     const __bf16* __restrict__ Bp, int M,
                                                     int Nc, int Mp, int Np, int64_t Kp,
                                                     int64_t chunks_per_split,
                                                     z64* __restrict__ part)
{
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int ntn = Np / 64;
    const int tm = blockIdx.x / ntn, tn = blockIdx.x % ntn;
    const int m0 = tm * 64 + (wave >> 1) * 32, n0 = tn * 64 + (wave & 1) * 32;
    const int split = blockIdx.y;
    const int64_t nch = Kp / 32;
    const int64_t c0 = (int64_t)split * chunks_per_split;
    const int64_t c1 = (c0 + chunks_per_split < nch) ? c0 + chunks_per_split : nch;
    const int64_t pa = (int64_t)Mp * Kp, pb = (int64_t)Np * Kp;
    nl_flt4 accr[2][2], acci[2][2];
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int b = 0; b < 2; ++b)
        {
            accr[a][b] = (nl_flt4){0.f, 0.f, 0.f, 0.f};
            acci[a][b] = (nl_flt4){0.f, 0.f, 0.f, 0.f};
        }
    const int r = lane & 15, kq = 8 * (lane >> 4);
    for (int64_t c = c0; c < c1; ++c)
    {
        const int64_t k = c * 32 + kq;
        nl_bf16x8 ar[NP][2], ai[NP][2], nai[NP][2], br[NP][2], bi[NP][2];
#pragma unroll
        for (int p = 0; p < NP; ++p)
#pragma unroll
            for (int h = 0; h < 2; ++h)
            {
                const int64_t ra = (int64_t)(m0 + 16 * h + r) * Kp + k;
                const int64_t rb = (int64_t)(n0 + 16 * h + r) * Kp + k;
                ar[p][h] = *reinterpret_cast<const nl_bf16x8*>(Ap + (2 * p) * pa + ra);
                ai[p][h] = *reinterpret_cast<const nl_bf16x8*>(Ap + (2 * p + 1) * pa + ra);
                nai[p][h] = nl_neg(ai[p][h]);
                br[p][h] = *reinterpret_cast<const nl_bf16x8*>(Bp + (2 * p) * pb + rb);
                bi[p][h] = *reinterpret_cast<const nl_bf16x8*>(Bp + (2 * p + 1) * pb + rb);
            }
#pragma unroll
        for (int p1 = 0; p1 < NP; ++p1)
#pragma unroll
            for (int p2 = 0; p2 < NP; ++p2)
            {
                if (p1 + p2 >= NP) continue;
                if (NPROD == 3 && p1 + p2 > 1) continue;
#pragma unroll
                for (int a = 0; a < 2; ++a)
#pragma unroll
                    for (int b = 0; b < 2; ++b)
                    {
                        accr[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ar[p1][a], br[p2][b],
                                                                            accr[a][b], 0, 0, 0);
                        accr[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(nai[p1][a], bi[p2][b],
                                                                            accr[a][b], 0, 0, 0);
                        acci[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ar[p1][a], bi[p2][b],
                                                                            acci[a][b], 0, 0, 0);
                        acci[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ai[p1][a], br[p2][b],
                                                                            acci[a][b], 0, 0, 0);
                    }
            }
    }
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int b = 0; b < 2; ++b)
#pragma unroll
            for (int v = 0; v < 4; ++v)
            {
                const int row = m0 + 16 * a + 4 * (lane >> 4) + v;
                const int col = n0 + 16 * b + r;
                if (row < M && col < Nc)
                    part[((int64_t)split * M + row) * Nc + col] = {(double)accr[a][b][v],
                                                                   (double)acci[a][b][v]};
            }
}
