// conv.hpp -- local e-ph part in the sphere form: dV_nu psi_k,n transformed
// to the k+q sphere and contracted with psi_k+q there, as elphLocal does
// (src/fft/convolution.c:13-189, src/dvloc/compute_Vbare_loc.c:286-342):
//
//   g[nu][n][m] = (1/N) sum_{sigma, G in sphere} conj(psi_kq,m,sigma(G))
//                                        FFT[(dV_nu psi_k,n)_sigma](G)
//
// By Parseval this equals the sum over the box (contract.hpp), and costs
// 5 N log2 N + 8 npw nb instead of 8 N nb operations per (nu, n): at 96^3
// points, npw 36,800 and 128 bands a seventh.
//
// Only what the spheres touch is transformed, and the planes stay in LDS:
//   k_sph_mask / _scan / _gather : a rotated sphere as sticks along x (one
//                per occupied (Gy, Gz), their Gx as bit masks) and its
//                coefficients in stick order, for both sides of a pair
//   k_box_x, k_box_plane : psi_k(r): sticks along x, then per x plane y and
//                z in LDS, written once
//   k_conv_plane : per x plane, dV psi formed while it is loaded, z
//                transform of its rows (keeping the Gz of the sphere), y
//                transform of the kept columns (keeping the sticks)
//   k_conv_x   : x transform of the sticks (keeping their Gx)
//   k_sph_gemm : the product over the sphere on MFMA
// A line is N = R1 x R2 points (radix.hpp): one LDS exchange per axis.
//
// LDS layouts: an exchange row of a line holds [R2][R1 | 1] (odd strides:
// the column-wise stores and row-wise loads spread over the banks); the
// plane between the z and y steps holds, per kept Gz, y as [R1][R2 | 1],
// transformed in place (a thread writes back the addresses it read).
#pragma once

#include <algorithm>

#include "common.hpp"
#include "mfma.hpp"
#include "radix.hpp"

#define SPH_MAXN 256 // longest axis (bit masks of 8 words, byte ranks)

// one side (iBZ k, symmetry, umklapp vector) of a pair as a sphere
struct SphSide
{
    const z64* wfc;
    const double* gvec;
    int npw, ld; // plane waves, row length of coef (multiple of 16)
    SideGeom geo;
    int* idx;        // (npw) box index or -1
    z64* ph;         // (npw) translation phase
    unsigned* mask;  // (Nz, Ny, words) Gx bits of every (Gz, Gy)
    int* smap;       // (nzk, Ny) stick number or -1
    short* zc;       // (Nz) kept column of Gz or -1
    int* off;        // (sticks) first coefficient
    unsigned* smask; // (sticks, words) Gx bits
    int* cnt;        // kept columns, sticks, coefficients
    void* coef;      // (sets, ld) coefficients in stick order
    void* line;      // k side: (sets, Nx, sticks) after the x step
    void* box;       // k side: (sets, N)
};

// box index, translation phase and Gx bits of every plane wave (k_gindex)
static __global__ void k_sph_mask(const SphSide* __restrict__ sides, int Nx, int Ny, int Nz, int words,
                           int* __restrict__ err)
{
    const SphSide& sd = sides[blockIdx.y];
    const int g = blockIdx.x * blockDim.x + threadIdx.x;
    if (g >= sd.npw) return;
    const auto gv = g_of(sd.gvec + 3 * (int64_t)g);
    const double G[3] = {gv[0], gv[1], gv[2]};
    const int N[3] = {Nx, Ny, Nz};
    int gi[3], bad = 0;
    double Gr[3];
    for (int i = 0; i < 3; ++i)
    {
        const double c = G[0] * sd.geo.M[3 * i] + G[1] * sd.geo.M[3 * i + 1] +
                         G[2] * sd.geo.M[3 * i + 2] + sd.geo.G0c[i];
        Gr[i] = rint(c);
        const int v = (int)Gr[i];
        const int b = v < 0 ? v + N[i] : v;
        if (b < 0 || b >= N[i]) bad = 1;
        gi[i] = b;
    }
    if (bad)
    {
        atomicOr(err, 1);
        g_of(sd.idx)[g] = -1;
        return;
    }
    g_of(sd.idx)[g] = (gi[0] * Ny + gi[1]) * Nz + gi[2];
    const double kd = sd.geo.kc[0] * sd.geo.tauc[0] + sd.geo.kc[1] * sd.geo.tauc[1] +
                      sd.geo.kc[2] * sd.geo.tauc[2];
    const double gd =
        Gr[0] * sd.geo.tauc[0] + Gr[1] * sd.geo.tauc[1] + Gr[2] * sd.geo.tauc[2];
    double s1, c1, s2, c2;
    sincos(-2.0 * LELPH_RPI * kd, &s1, &c1);
    sincos(-2.0 * LELPH_RPI * gd, &s2, &c2);
    gptr<double>::of(sd.ph).set(g, cmul(z64{c1, s1}, z64{c2, s2}));
    atomicOr(&sd.mask[((int64_t)gi[2] * Ny + gi[1]) * words + (gi[0] >> 5)],
             1u << (gi[0] & 31));
}

// exclusive scan of (a, b) over a block of 1024 threads; tot: block totals
__device__ inline void sph_scan2(int& a, int& b, int* wa, int* wb, int& ta, int& tb)
{
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    int ia = a, ib = b;
    for (int d = 1; d < 64; d <<= 1)
    {
        const int xa = __shfl_up(ia, d), xb = __shfl_up(ib, d);
        if (lane >= d)
        {
            ia += xa;
            ib += xb;
        }
    }
    __syncthreads();
    if (lane == 63)
    {
        wa[wave] = ia;
        wb[wave] = ib;
    }
    __syncthreads();
    int oa = 0, ob = 0;
    ta = tb = 0;
    for (int w = 0; w < 16; ++w)
    {
        if (w < wave)
        {
            oa += wa[w];
            ob += wb[w];
        }
        ta += wa[w];
        tb += wb[w];
    }
    a = oa + ia - a;
    b = ob + ib - b;
}

// sticks in (Gz, Gy) order, their first coefficients and masks, the kept Gz
// columns.  One block per side; nzk_max, nst_max: what the host sized the
// buffers and launches for (error bit 3 when a sphere exceeds them or two
// plane waves share a box point).
static __global__ __launch_bounds__(1024) void k_sph_scan(const SphSide* __restrict__ sides, int Ny,
                                                   int Nz, int words, int nzk_max, int nst_max,
                                                   int* __restrict__ err)
{
    __shared__ int wa[16], wb[16];
    __shared__ int zf[SPH_MAXN];
    __shared__ short zl[SPH_MAXN];
    const SphSide& sd = sides[blockIdx.x];
    const int tid = threadIdx.x;
    const int cells = Ny * Nz;
    const auto mask = g_of(sd.mask), smask = g_of(sd.smask);
    const auto smap = g_of(sd.smap), off = g_of(sd.off), cnt = g_of(sd.cnt);
    const auto zc = g_of(sd.zc);
    if (tid < SPH_MAXN) zf[tid] = 0;
    __syncthreads();
    for (int c = tid; c < cells; c += 1024)
    {
        unsigned any = 0;
        for (int w = 0; w < words; ++w) any |= mask[(int64_t)c * words + w];
        if (any) zf[c / Ny] = 1;
    }
    __syncthreads();
    int z = tid < Nz ? zf[tid] : 0, dum = 0, nzk, td;
    const int has = z;
    sph_scan2(z, dum, wa, wb, nzk, td);
    if (tid < Nz)
    {
        zl[tid] = has ? (short)z : (short)-1;
        zc[tid] = zl[tid];
    }
    __syncthreads();
    int s0 = 0, p0 = 0;
    for (int c0 = 0; c0 < cells; c0 += 1024)
    {
        const int c = c0 + tid;
        int n = 0;
        if (c < cells)
            for (int w = 0; w < words; ++w) n += __popc(mask[(int64_t)c * words + w]);
        int st = n > 0 ? 1 : 0, po = n, ts, tp;
        sph_scan2(st, po, wa, wb, ts, tp);
        if (c < cells && zl[c / Ny] >= 0 && zl[c / Ny] < nzk_max)
        {
            const int s = s0 + st;
            const bool in = n > 0 && s < nst_max;
            smap[zl[c / Ny] * Ny + c % Ny] = in ? s : -1;
            if (in)
            {
                off[s] = p0 + po;
                for (int w = 0; w < words; ++w)
                    smask[(int64_t)s * words + w] = mask[(int64_t)c * words + w];
            }
        }
        s0 += ts;
        p0 += tp;
        __syncthreads();
    }
    if (tid == 0)
    {
        const bool ok = nzk <= nzk_max && s0 <= nst_max && p0 == sd.npw;
        cnt[0] = ok ? nzk : 0;
        cnt[1] = ok ? s0 : 0;
        cnt[2] = ok ? p0 : 0;
        if (!ok) atomicOr(err, 8);
    }
}

// rank of Gx in a stick, or -1
__device__ inline int sph_rank(const GLOBAL_AS unsigned* m, int gx)
{
    const int w = gx >> 5;
    const unsigned bit = 1u << (gx & 31);
    const unsigned mw = m[w];
    if (!(mw & bit)) return -1;
    int r = __popc(mw & (bit - 1));
    for (int i = 0; i < w; ++i) r += __popc(m[i]);
    return r;
}

// rotated coefficients (su2, translation phase, time-reversal conjugate, as
// k_scatter) in stick order, rounded once to T; the row tail up to ld is
// zero.  blockIdx.y: groups of `per` sets.
template <typename T>
__global__ __launch_bounds__(256) void k_sph_gather(const SphSide* __restrict__ sides,
                                                    int64_t nsets, int nspinor, int Ny, int Nz,
                                                    int words, int per)
{
    const SphSide& sd = sides[blockIdx.z];
    const int g = blockIdx.x * blockDim.x + threadIdx.x;
    if (g >= sd.ld || sd.cnt[1] == 0) return;
    const int64_t npw = sd.npw, ld = sd.ld;
    const int64_t s0 = (int64_t)blockIdx.y * per;
    const int64_t s1 = s0 + per < nsets ? s0 + per : nsets;
    const auto out = gptr<T>::of(sd.coef);
    if (g >= npw)
    {
        for (int64_t r = s0 * nspinor; r < s1 * nspinor; ++r) out.set(r * ld + g, {0, 0});
        return;
    }
    const int id = g_of(sd.idx)[g];
    if (id < 0) return;
    const int gz = id % Nz, gxy = id / Nz, gy = gxy % Ny, gx = gxy / Ny;
    const int st = g_of(sd.smap)[g_of(sd.zc)[gz] * Ny + gy];
    const int64_t p = g_of(sd.off)[st] + sph_rank(g_of(sd.smask) + (int64_t)st * words, gx);
    const z64 ph = gptr<double>::of(sd.ph)[g];
    const bool cj = sd.geo.conj;
    for (int64_t s = s0; s < s1; ++s)
    {
        const auto w = gptr<double>::of(sd.wfc) + s * nspinor * npw;
        const auto o = out + s * nspinor * ld;
        if (nspinor == 1)
        {
            z64 c = cmul(w[g], ph);
            if (cj) c.y = -c.y;
            o.set(p, {(T)c.x, (T)c.y});
        }
        else
        {
            const z64 u = w[g], d = w[npw + g];
            z64 a = cmul(cadd(cmul(u, sd.geo.su2[0]), cmul(d, sd.geo.su2[1])), ph);
            z64 b = cmul(cadd(cmul(u, sd.geo.su2[2]), cmul(d, sd.geo.su2[3])), ph);
            if (cj)
            {
                a.y = -a.y;
                b.y = -b.y;
            }
            o.set(p, {(T)a.x, (T)a.y});
            o.set(ld + p, {(T)b.x, (T)b.y});
        }
    }
}

// ---------------------------------------------------------------------------
// line steps

// Precision of the FP32 form.  The transforms of dV psi are FP32, the psi_k
// boxes FP64 in registers (FP32 between the axes; a twelfth of the pair's
// time) and the sphere product FP64 on MFMA with FP32 operands.  Error of g
// against FP64, 16^3 .. 80^3 and all spins: 0.5 .. 0.9e-7; with FP32 boxes
// and FP32 products added into FP64 every 64 points 2.3 .. 2.6e-7, more than
// the box form's 0.7 .. 1.8e-7.
template <typename T, typename A>
__device__ __forceinline__ cpx<T> to(cpx<A> v)
{
    return {(T)v.x, (T)v.y};
}

// twiddle w_N^(SIGN j k) from the table of e^{+2 pi i t/N}
template <int SIGN>
__device__ __forceinline__ z64 ln_tw(const z64* __restrict__ W, int t)
{
    z64 w = W[t];
    if (SIGN < 0) w.y = -w.y;
    return w;
}

// first step of a line: R1-point transforms of v, twiddled, into an
// exchange row
template <typename T, int SIGN, int R1, typename A>
__device__ __forceinline__ void ln_first(cpx<A>* v, int j, const z64* __restrict__ W,
                                         cpx<T>* row)
{
    Rdft<A, SIGN, R1>::run(v);
    cpx<T>* o = row + j * (R1 | 1);
    o[0] = to<T>(v[0]);
#pragma unroll
    for (int k = 1; k < R1; ++k) o[k] = to<T>(cmul(v[k], to<A>(ln_tw<SIGN>(W, j * k))));
}

// second step: point k1 + R1 k2 of the line in v[k2]
template <typename T, int SIGN, int R1, int R2, typename A>
__device__ __forceinline__ void ln_second(const cpx<T>* row, int k1, cpx<A>* v)
{
#pragma unroll
    for (int j = 0; j < R2; ++j) v[j] = to<A>(row[j * (R1 | 1) + k1]);
    Rdft<A, SIGN, R2>::run(v);
}

// exchange row of a line, in elements: [R2][R1 | 1]
constexpr int ln_row(int R1, int R2) { return R2 * (R1 | 1); }
// the same for the x steps, whose lanes run over lines (odd)
constexpr int ln_xrow(int R1, int R2) { return (R2 * (R1 | 1)) | 1; }
// y line of a kept column in the plane buffer
constexpr int ln_prow(int R1, int R2) { return R1 * (R2 | 1) + 1; }

// Position of point z inside a row of a box or potential that the plane
// kernels read.  A lane loads points j + R2 i for all i: in FP32 two of them
// (i, i + 1) lie together, so that it loads 16 bytes at a time as in FP64
// (96 x 96 planes: 384 -> 192 load instructions per plane, 19 address cycles
// each).
template <typename T>
__host__ __device__ inline int ln_pos(int z, int R1, int R2)
{
    if (sizeof(T) == 8) return z;
    const int i = z / R2, j = z - i * R2;
    return i == R1 - 1 && R1 % 2 ? z : (i >> 1) * 2 * R2 + 2 * j + (i & 1);
}

// points j + R2 i of a row, in ln_pos order
template <int R1, int R2>
__device__ __forceinline__ void ln_load(cpx<double>* x, gptr<double> row, int j)
{
#pragma unroll
    for (int i = 0; i < R1; ++i) x[i] = row[j + R2 * i];
}
template <int R1, int R2>
__device__ __forceinline__ void ln_load(cpx<float>* x, gptr<float> row, int j)
{
    typedef float v4 __attribute__((ext_vector_type(4), aligned(8)));
#pragma unroll
    for (int i = 0; i + 1 < R1; i += 2)
    {
        const v4 v = *(const GLOBAL_AS v4*)(row.p + 2 * j + R2 * i);
        x[i] = {v.x, v.y};
        x[i + 1] = {v.z, v.w};
    }
    if (R1 % 2) x[R1 - 1] = row[j + R2 * (R1 - 1)];
}

// ---------------------------------------------------------------------------
// psi_k(r)

struct BoxArgs
{
    int Nx, Ny, Nz, words;
    int64_t nrows; // sets x spinors
    int nzk_max, nst_max, rows_per_block;
};

// sticks -> x lines: line[row][x][stick].  Block: a tile of sticks, a group
// of rows.
template <typename T, int R1, int R2, int TS, int NT>
__device__ inline void box_x_body(const SphSide& sd, const BoxArgs& a, int tile, int64_t row0,
                                  const z64* __restrict__ W, char* smem)
{
    constexpr int N = R1 * R2, SR = ln_xrow(R1, R2);
    cpx<T>* S = reinterpret_cast<cpx<T>*>(smem);
    unsigned char* rk = reinterpret_cast<unsigned char*>(S + TS * SR);
    int* so = reinterpret_cast<int*>(rk + ((TS * N + 15) & ~15));
    const int nst = sd.cnt[1];
    const int s0 = tile * TS;
    if (s0 >= nst) return;
    const int tid = threadIdx.x;
    for (int f = tid; f < TS * N; f += NT)
    {
        const int s = f / N, gx = f - s * N;
        const int r = s0 + s < nst ? sph_rank(g_of(sd.smask) + (int64_t)(s0 + s) * a.words, gx) : -1;
        rk[f] = (unsigned char)(r < 0 ? 255 : r);
    }
    if (tid < TS) so[tid] = s0 + tid < nst ? g_of(sd.off)[s0 + tid] : 0;
    __syncthreads();
    const int64_t r1 = row0 + a.rows_per_block < a.nrows ? row0 + a.rows_per_block : a.nrows;
    for (int64_t row = row0; row < r1; ++row)
    {
        const auto c = gptr<T>::of(sd.coef) + row * sd.ld;
        const auto out = gptr<T>::of(sd.line) + row * N * nst;
        for (int t = tid; t < TS * R2; t += NT)
        {
            const int s = t / R2, j = t - s * R2;
            z64 v[R1];
#pragma unroll
            for (int i = 0; i < R1; ++i)
            {
                const int r = rk[s * N + j + R2 * i];
                v[i] = r == 255 ? z64{0, 0} : to<double>(c[so[s] + r]);
            }
            ln_first<T, 1, R1>(v, j, W, S + s * SR);
        }
        __syncthreads();
        for (int t = tid; t < TS * R1; t += NT)
        {
            const int s = t % TS, k1 = t / TS;
            z64 v[R2];
            ln_second<T, 1, R1, R2>(S + s * SR, k1, v);
            if (s0 + s < nst)
#pragma unroll
                for (int k2 = 0; k2 < R2; ++k2)
                    out.set((int64_t)(k1 + R1 * k2) * nst + s0 + s, to<T>(v[k2]));
        }
        __syncthreads();
    }
}

// Orders the LDS accesses of one wave (they execute in order; this keeps the
// compiler from moving them across): the exchange between the two steps of a
// line stays inside a wave, so no block barrier is needed for it.
__device__ __forceinline__ void wave_order()
{
    __builtin_amdgcn_wave_barrier();
    asm volatile("" ::: "memory");
}

// rows (lines) that one wave takes through both steps at a time
constexpr int ln_rows(int R2) { return 64 / R2; }

// first y step of columns c0 .. of the plane buffer, in place; all lanes
// compute, those past the last column store nothing
template <typename A, typename T, int SIGN, int R1, int R2, typename TW>
__device__ __forceinline__ void plane_y_first(cpx<T>* P, int c0, int nzk, const TW& tw, int r,
                                              int j)
{
    constexpr int P2 = R2 | 1, PR = ln_prow(R1, R2);
    cpx<T>* b = P + min(c0 + r, nzk - 1) * PR + j;
    cpx<A> v[R1];
#pragma unroll
    for (int i = 0; i < R1; ++i) v[i] = to<A>(b[i * P2]);
    Rdft<A, SIGN, R1>::run(v);
#pragma unroll
    for (int k = 1; k < R1; ++k) v[k] = cmul(v[k], to<A>(tw(j, k)));
    if (r < ln_rows(R2) && c0 + r < nzk)
#pragma unroll
        for (int k = 0; k < R1; ++k) b[k * P2] = to<T>(v[k]);
    wave_order();
}

// twiddles of a lane's j: from the table, or held in registers
template <int SIGN>
struct LnTable
{
    const z64* W;
    __device__ __forceinline__ z64 operator()(int j, int k) const
    {
        return ln_tw<SIGN>(W, j * k);
    }
};
template <int R2, typename T>
struct LnLds // copied to LDS, [k][j]
{
    const cpx<T>* tw;
    __device__ __forceinline__ cpx<T> operator()(int j, int k) const { return tw[k * R2 + j]; }
};
struct LnHeld
{
    const z64* tw;
    __device__ __forceinline__ z64 operator()(int, int k) const { return tw[k]; }
};

// y transform of the kept columns of the plane buffer; second step's point
// y = k1 + R1 k2 back to [k1][k2] of the column
template <typename T, int SIGN, int R1, int R2, int NW>
__device__ inline void plane_y_lds(cpx<T>* P, int nzk, const z64* __restrict__ W, int tid)
{
    constexpr int LC = ln_rows(R2), P2 = R2 | 1, PR = ln_prow(R1, R2);
    const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int j = lane % R2, r = lane / R2, k1 = lane % R1, rd = lane / R1;
    for (int c0 = wave * LC; c0 < nzk; c0 += NW * LC)
    {
        plane_y_first<double, T, SIGN, R1, R2>(P, c0, nzk, LnTable<SIGN>{W}, r, j);
        cpx<T>* b = P + min(c0 + rd, nzk - 1) * PR + k1 * P2;
        z64 v[R2];
#pragma unroll
        for (int i = 0; i < R2; ++i) v[i] = to<double>(b[i]);
        Rdft<double, SIGN, R2>::run(v);
        wave_order();
        if (rd < LC && c0 + rd < nzk)
#pragma unroll
            for (int i = 0; i < R2; ++i) b[i] = to<T>(v[i]);
        wave_order();
    }
}

// forward y transform of the kept columns, out to the sticks
template <typename T, int R1, int R2, typename TW>
__device__ inline void plane_y_out(cpx<T>* P, int nzk, const TW& tw, const unsigned short* sl,
                                   gptr<T> out, int NW, int tid)
{
    constexpr int LC = ln_rows(R2), P2 = R2 | 1, PR = ln_prow(R1, R2), N = R1 * R2;
    const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int j = lane % R2, r = lane / R2, k1 = lane % R1, rd = lane / R1;
    for (int c0 = wave * LC; c0 < nzk; c0 += NW * LC)
    {
        plane_y_first<T, T, -1, R1, R2>(P, c0, nzk, tw, r, j);
        const int c = min(c0 + rd, nzk - 1);
        const cpx<T>* b = P + c * PR + k1 * P2;
        const unsigned short* sm = sl + c * N + k1;
        cpx<T> v[R2];
#pragma unroll
        for (int i = 0; i < R2; ++i) v[i] = b[i];
        Rdft<T, -1, R2>::run(v);
        if (rd < LC && c0 + rd < nzk)
#pragma unroll
            for (int k = 0; k < R2; ++k)
            {
                const int st = sm[R1 * k];
                if (st != 0xffff) out.set(st, v[k]);
            }
        wave_order();
    }
}

// operands of dV psi on one plane: one potential and one psi, or (TWO) the
// two terms of a spinor component under a 2x2 potential
template <typename T>
struct ConvSrc
{
    gptr<T> p0, v0, p1, v1;
};

// FP64 lines exchange their real and imaginary parts one after the other
// through the same rows: half the LDS, so that the rows of 8 waves (41 KB) fit
// beside a 96 x 96 plane buffer (80 KB) and its tables.
template <typename T>
constexpr bool ln_split()
{
    return sizeof(T) == 8;
}
// bytes of an exchange row
template <typename T>
constexpr int ln_row_bytes(int R1, int R2)
{
    return ln_row(R1, R2) * (int)sizeof(T) * (ln_split<T>() ? 1 : 2);
}

// rows of exchange space per wave: lanes beyond the last whole line (64 not a
// multiple of R2) write a row of their own that nobody reads
constexpr int ln_space(int R2) { return ln_rows(R2) + (64 % R2 ? 1 : 0); }

// Bytes from the start of the exchange rows that ln_exchange reads: lanes past
// the last line (R1 < R2: more of them in the second step) read on beyond the
// rows of their wave, values that are not stored.  A block has at least that
// much LDS; only planes of a few kept columns have less by themselves.
static inline size_t ln_reach(int R1, int R2, int NW, int row_bytes)
{
    const size_t last = (size_t)(63 / R1) * ln_row(R1, R2) + (R2 - 1) * (R1 | 1) + R1; // of 8 bytes
    return (size_t)(NW - 1) * ln_space(R2) * row_bytes + 8 * last;
}

// The exchange of a wave's lines between their two steps: x (twiddled) of
// lane (row r, j) to v of lane (row rd, k1).  All lanes take part, so there
// is no branch to carry registers over: rows past LR hold or read values
// that are not stored.
template <typename T, int R1, int R2, typename A>
__device__ __forceinline__ void ln_exchange(const cpx<A>* x, cpx<A>* v, char* Sw, int r, int j,
                                            int rd, int k1)
{
    constexpr int SR = ln_row(R1, R2);
    if constexpr (ln_split<T>())
    {
        T* S = reinterpret_cast<T*>(Sw);
        T* o = S + r * SR + j * (R1 | 1);
        const T* in = S + rd * SR + k1;
#pragma unroll
        for (int k = 0; k < R1; ++k) o[k] = x[k].x;
        wave_order();
#pragma unroll
        for (int i = 0; i < R2; ++i) v[i].x = in[i * (R1 | 1)];
        wave_order();
#pragma unroll
        for (int k = 0; k < R1; ++k) o[k] = x[k].y;
        wave_order();
#pragma unroll
        for (int i = 0; i < R2; ++i) v[i].y = in[i * (R1 | 1)];
        wave_order();
    }
    else
    {
        cpx<T>* S = reinterpret_cast<cpx<T>*>(Sw);
        cpx<T>* o = S + r * SR + j * (R1 | 1);
        const cpx<T>* in = S + rd * SR + k1;
#pragma unroll
        for (int k = 0; k < R1; ++k) o[k] = {(T)x[k].x, (T)x[k].y};
        wave_order();
#pragma unroll
        for (int i = 0; i < R2; ++i) v[i] = {(A)in[i * (R1 | 1)].x, (A)in[i * (R1 | 1)].y};
        wave_order();
    }
}

// Forward z rows of dV psi of one plane (any Ny): each of the NW waves takes
// LR rows at a time through both steps, the next rows' psi loaded before the
// second step of the current ones.
template <typename T, bool TWO, int R1, int R2>
__device__ inline void plane_z_rows(const ConvSrc<T>& q, int Ny, const LnLds<R2, T>& tw, char* S, cpx<T>* P, int prow, const unsigned short* yad,
                                    const short* zc, int NW, int tid)
{
    constexpr int LR = ln_rows(R2), N = R1 * R2, M = TWO ? 2 : 1;
    const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int j = lane % R2, r = lane / R2, k1 = lane % R1, rd = lane / R1;
    char* Sw = S + wave * ln_space(R2) * ln_row_bytes<T>(R1, R2);
    if (wave * LR >= Ny) return;
    cpx<T> p[M][R1];
    auto row_of = [&](int y) { return min(y + r, Ny - 1) * N; };
    auto fetch = [&](int y) {
        ln_load<R1, R2>(p[0], q.p0 + row_of(y), j);
        if constexpr (TWO)
            ln_load<R1, R2>(p[1], q.p1 + row_of(y), j);
    };
    fetch(wave * LR);
    for (int y0 = wave * LR; y0 < Ny; y0 += NW * LR)
    {
        cpx<T> x[R1], v[R2];
        if constexpr (TWO)
        {
            cpx<T> e[2][R1]; // no registers to load these ahead
            ln_load<R1, R2>(e[0], q.v0 + row_of(y0), j);
            ln_load<R1, R2>(e[1], q.v1 + row_of(y0), j);
#pragma unroll
            for (int i = 0; i < R1; ++i) x[i] = cadd(cmul(e[0][i], p[0][i]), cmul(e[1][i], p[1][i]));
        }
        else
        {
            ln_load<R1, R2>(x, q.v0 + row_of(y0), j);
#pragma unroll
            for (int i = 0; i < R1; ++i) x[i] = cmul(x[i], p[0][i]);
        }
        Rdft<T, -1, R1>::run(x);
#pragma unroll
        for (int k = 1; k < R1; ++k) x[k] = cmul(x[k], tw(j, k));
        if (y0 + NW * LR < Ny) fetch(y0 + NW * LR);
        ln_exchange<T, R1, R2>(x, v, Sw, r, j, rd, k1);
        Rdft<T, -1, R2>::run(v);
        if (rd < LR && y0 + rd < Ny)
        {
            cpx<T>* o = P + yad[y0 + rd];
#pragma unroll
            for (int k = 0; k < R2; ++k)
            {
                const int c = zc[k1 + R1 * k];
                if (c >= 0) o[c * prow] = v[k];
            }
        }
    }
}

// backward z rows of the plane: kept columns -> box plane
template <typename T, int R1, int R2, int NW>
__device__ inline void plane_z_backward(const cpx<T>* P, int prow, const unsigned short* yad,
                                        const short* zc, int Ny, const z64* __restrict__ W,
                                        char* S, gptr<T> out, int tid)
{
    constexpr int LR = ln_rows(R2), N = R1 * R2;
    const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int j = lane % R2, r = lane / R2, k1 = lane % R1, rd = lane / R1;
    char* Sw = S + wave * ln_space(R2) * ln_row_bytes<T>(R1, R2);
    for (int y0 = wave * LR; y0 < Ny; y0 += NW * LR)
    {
        z64 x[R1], v[R2];
        const cpx<T>* p = P + yad[min(y0 + r, Ny - 1)];
#pragma unroll
        for (int i = 0; i < R1; ++i)
        {
            const int c = zc[j + R2 * i];
            x[i] = to<double>(p[max(c, 0) * prow]);
            if (c < 0) x[i] = {0, 0};
        }
        Rdft<double, 1, R1>::run(x);
#pragma unroll
        for (int k = 1; k < R1; ++k) x[k] = cmul(x[k], ln_tw<1>(W, j * k));
        ln_exchange<T, R1, R2>(x, v, Sw, r, j, rd, k1);
        Rdft<double, 1, R2>::run(v);
        if (rd < LR && y0 + rd < Ny)
        {
            const auto o = out + (int64_t)(y0 + rd) * N;
#pragma unroll
            for (int k = 0; k < R2; ++k) o.set(ln_pos<T>(k1 + R1 * k, R1, R2), to<T>(v[k]));
        }
    }
}

// row groups of a square plane per wave
constexpr int sq_groups(int R1, int R2, int NW)
{
    return (R1 * R2 + NW * ln_rows(R2) - 1) / (NW * ln_rows(R2));
}
// twiddles in LDS instead of 4 (R1 - 1) registers
constexpr bool sq_tw_lds(int R1) { return R1 >= 7; }
// row groups of a plane whose dV stays in registers over the sets: in FP32
// what fits in 40 of them (72^3, 64 bands, 4 pairs: 13.6 -> 13.1 ms; 96^3,
// 128 bands: no difference, 19.8 ms per pair either way); in FP64 none (64
// registers of it made the transforms spill: 31.9 -> 34.1 ms per pair)
template <typename T>
constexpr int sq_keep(int R1, int R2, int NW)
{
    const int fit = sizeof(T) == 8 ? 0 : 40 / (R1 * (int)sizeof(cpx<T>) / 4);
    const int g = sq_groups(R1, R2, NW);
    return fit < g ? fit : g;
}

// FP32 potential with its rows in ln_pos order
template <typename T>
__global__ void k_conv_dv32(const z64* __restrict__ s, cpx<T>* __restrict__ d, int64_t n, int Nz,
                            int R1, int R2)
{
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= n) return;
    const int64_t row = t / Nz;
    const int z = (int)(t - row * Nz);
    d[row * Nz + ln_pos<T>(z, R1, R2)] = {(T)s[t].x, (T)s[t].y};
}

struct ConvPair
{
    const void* box;  // psi_k(r), (sets, N)
    const void* dv;   // (nm, nmag, N)
    int side;         // k+q side
    void* line;       // (modes, sets of a launch, Nx, sticks) after the y step
    void* c;          // (modes of a block, sets, ld) on the sphere
};

struct ConvArgs
{
    int Nx, Ny, Nz, words;
    int vc, v0, nv;   // first mode that c holds, first and number of this launch
    int s0, ns;       // first set (spin, band, spinor) and number of this launch
    int nspin, nb, nspinor, nmag;
    int nzk_max, nst_max;
    int sper;         // sets per block of the plane kernels
    int rows_per_block;
};

// LDS of a plane block: exchange rows, plane buffer, y addresses, kept
// columns, twiddles of both axes
struct PlaneLds
{
    int rows;  // bytes of the exchange rows
    int prow;  // elements of a plane column
    int tw;    // offset of the twiddles
    size_t bytes;
};

template <typename T>
static inline PlaneLds plane_lds(int R1y, int R2y, int R1z, int R2z, int nzk, int NT)
{
    PlaneLds l;
    l.rows = ((NT / 64) * ln_space(R2z) * ln_row_bytes<T>(R1z, R2z) + 15) & ~15;
    l.prow = ln_prow(R1y, R2y);
    l.tw = (int)(((size_t)l.rows + sizeof(cpx<T>) * (size_t)nzk * l.prow +
                  2 * (size_t)(R1y * R2y + R1z * R2z + nzk * R1y * R2y) + 15) &
                 ~(size_t)15);
    l.bytes = std::max((size_t)l.tw + sizeof(cpx<T>) * (size_t)(R1y * R2y + R1z * R2z),
                       ln_reach(R1z, R2z, NT / 64, ln_row_bytes<T>(R1z, R2z)));
    return l;
}

// the same of k_conv_square: exchange rows, plane buffer, sticks, twiddles
template <typename T>
static inline size_t square_lds(int R1, int R2, int NW, int nzk)
{
    auto up = [](size_t n) { return (n + 15) & ~(size_t)15; };
    const size_t rb = (size_t)ln_row_bytes<T>(R1, R2), item = sizeof(cpx<T>);
    return std::max(up(NW * ln_space(R2) * rb) + up(item * nzk * ln_prow(R1, R2)) +
                        up(2 * (size_t)nzk * R1 * R2) + (sq_tw_lds(R1) ? item * R1 * R2 : 0),
                    ln_reach(R1, R2, NW, (int)rb));
}

// tables of a plane block: address of y inside a column, column of Gz
__device__ inline void plane_tables(const GLOBAL_AS short* zc, int Ny, int Nz, bool sub,
                                    int R1y, int R2y, unsigned short* yad, short* zl)
{
    for (int y = threadIdx.x; y < Ny; y += blockDim.x)
        yad[y] = (unsigned short)(sub ? (y % R1y) * (R2y | 1) + y / R1y
                                      : (y / R2y) * (R2y | 1) + y % R2y);
    for (int z = threadIdx.x; z < Nz; z += blockDim.x) zl[z] = zc[z];
}

// x lines of the sticks -> coefficients on the k+q sphere
template <typename T, int R1, int R2, int TS, int NT>
__device__ inline void conv_x_body(const ConvPair& pr, const SphSide& sd, const ConvArgs& a,
                                   const z64* __restrict__ W, int tile, int64_t row0,
                                   char* smem)
{
    constexpr int N = R1 * R2, SR = ln_xrow(R1, R2);
    cpx<T>* S = reinterpret_cast<cpx<T>*>(smem);
    unsigned char* rk = reinterpret_cast<unsigned char*>(S + TS * SR);
    int* so = reinterpret_cast<int*>(rk + ((TS * N + 15) & ~15));
    const int nst = sd.cnt[1];
    const int s0 = tile * TS;
    if (s0 >= nst) return;
    const int tid = threadIdx.x;
    for (int f = tid; f < TS * N; f += NT)
    {
        const int s = f / N, gx = f - s * N;
        const int r = s0 + s < nst ? sph_rank(g_of(sd.smask) + (int64_t)(s0 + s) * a.words, gx) : -1;
        rk[f] = (unsigned char)(r < 0 ? 255 : r);
    }
    if (tid < TS) so[tid] = s0 + tid < nst ? g_of(sd.off)[s0 + tid] : 0;
    __syncthreads();
    const int64_t nsets = (int64_t)a.nspin * a.nb * a.nspinor;
    const int64_t nrows = (int64_t)a.nv * a.ns;
    const int64_t r1 = row0 + a.rows_per_block < nrows ? row0 + a.rows_per_block : nrows;
    for (int64_t row = row0; row < r1; ++row)
    {
        const auto in = gptr<T>::of(pr.line) + (row * N * nst + s0);
        const auto c = gptr<T>::of(pr.c) +
                       ((a.v0 - a.vc + row / a.ns) * nsets + a.s0 + row % a.ns) * sd.ld;
        for (int t = tid; t < TS * R2; t += NT)
        {
            const int s = t % TS, j = t / TS;
            cpx<T> v[R1];
#pragma unroll
            for (int i = 0; i < R1; ++i)
                v[i] = s0 + s < nst ? in[(int64_t)(j + R2 * i) * nst + s] : cpx<T>{0, 0};
            ln_first<T, -1, R1>(v, j, W, S + s * SR);
        }
        __syncthreads();
        for (int t = tid; t < TS * R1; t += NT)
        {
            const int s = t / R1, k1 = t - s * R1;
            cpx<T> v[R2];
            ln_second<T, -1, R1, R2>(S + s * SR, k1, v);
#pragma unroll
            for (int k2 = 0; k2 < R2; ++k2)
            {
                const int r = rk[s * N + k1 + R1 * k2];
                if (r != 255) c.set(so[s] + r, to<T>(v[k2]));
            }
        }
        __syncthreads();
    }
}

// ---------------------------------------------------------------------------
// Plane kernels.  The z and y lengths are chosen at run time among the
// compiled ones (a uniform switch per step; each case has its radices as
// constants).  CLS 0: first factors up to 10 and second up to 12 (lengths to
// 120 with few registers), CLS 1: the longer ones.  Square planes of one
// component have kernels of their own (k_conv_square).

constexpr int rx_class(int R1, int R2) { return R1 <= 10 && R2 <= 12 ? 0 : 1; }

struct PlaneArgs
{
    int s_bytes, prow, tw; // of PlaneLds
    int R1y, R2y, R2z;
};

// block -> (x, inner, outer): all blocks of an x plane on one XCD (block b
// runs on XCD b % 8), so that its psi and dV planes are shared in that L2
__device__ inline bool plane_decode(int Nx, int inner, int& x, int& in, int& outer)
{
    const int64_t b = blockIdx.x;
    const int nxg = (Nx + 7) / 8;
    int64_t r = b >> 3;
    in = (int)(r % inner);
    r /= inner;
    x = (int)(r % nxg) * 8 + (int)(b & 7);
    outer = (int)(r / nxg);
    return x < Nx;
}

// What a block of the plane kernels works on: one x plane, one mode, a range
// of sets.  Blocks that run together on an XCD are the modes of a launch
// times a few ranges at one x, so its 4 MB L2 holds their dV planes and each
// psi plane is fetched once for all the modes (a loop over modes instead,
// one psi plane per block, misses on 214 of the 295 KB that a 96 x 96 plane
// loads in FP64).
template <typename T, bool TWO>
struct PlaneJob
{
    gptr<T> psi, dv;       // this plane of box 0, of the mode's first component
    int64_t N;
    int t0, t1;            // sets
    int nzk, nst, nspinor, per_spin;
    const GLOBAL_AS int* smap;
    const GLOBAL_AS short* zc;
    gptr<T> out;           // sticks of set t0
    int64_t outs;          // elements between sets
    __device__ bool init(const ConvPair* pairs, const SphSide* sides, const ConvArgs& a)
    {
        const int nr = (a.ns + a.sper - 1) / a.sper;
        int x, in, ip;
        if (!plane_decode(a.Nx, a.nv * nr, x, in, ip)) return false;
        const int vl = in % a.nv, rg = in / a.nv;
        const ConvPair& pr = pairs[ip];
        const SphSide& sd = sides[pr.side];
        nzk = sd.cnt[0];
        nst = sd.cnt[1];
        if (nst == 0) return false;
        smap = g_of(sd.smap);
        zc = g_of(sd.zc);
        const int64_t pl = (int64_t)a.Ny * a.Nz;
        N = a.Nx * pl;
        nspinor = a.nspinor;
        per_spin = a.nmag == 2 ? a.nb * a.nspinor : 0; // sets per spin-resolved potential
        psi = gptr<T>::of(pr.box) + x * pl;
        dv = gptr<T>::of(pr.dv) + ((int64_t)(a.v0 + vl) * a.nmag * N + x * pl);
        t0 = a.s0 + rg * a.sper;
        t1 = a.s0 + min((rg + 1) * a.sper, a.ns);
        outs = (int64_t)a.Nx * nst;
        out = gptr<T>::of(pr.line) + (((int64_t)vl * a.ns + (t0 - a.s0)) * a.Nx + x) * nst;
        return true;
    }
    __device__ ConvSrc<T> src(int set) const
    {
        ConvSrc<T> q;
        if constexpr (TWO)
        {
            // 2x2 spinor potential (src/fft/convolution.c:322-352)
            const int sp = set & 1;
            q.p0 = psi + (int64_t)(set - sp) * N;
            q.p1 = q.p0 + N;
            q.v0 = dv + 2 * sp * N;
            q.v1 = q.v0 + N;
        }
        else
        {
            q.p0 = psi + (int64_t)set * N;
            q.v0 = per_spin && set >= per_spin ? dv + N : dv;
            q.p1 = q.p0;
            q.v1 = q.v0;
        }
        return q;
    }
};

// stick numbers of the kept columns as 16-bit LDS entries (0xffff: none)
__device__ inline void plane_sticks(const GLOBAL_AS int* smap, int n, unsigned short* sl)
{
    for (int f = threadIdx.x; f < n; f += blockDim.x) sl[f] = (unsigned short)smap[f];
}

// most threads of a plane block: what the registers of the longest factors of
// a class leave room for
template <typename T, bool TWO>
constexpr int plane_threads(int cls)
{
    return cls == 0 ? (sizeof(T) == 8 ? (TWO ? 256 : 512) : 768) : 256;
}

// any compiled (Ny, Nz).  Twiddles in LDS: read from the table per line they
// were a third of the address cycles (36^3 spinor, FP32: 1.58 -> 1.41 ms per
// 8 pairs; 45 x 108 planes, FP64: 1 %).  Loading dV a group ahead beside psi
// gains nothing here and costs 5 % in k_conv_square in FP64.
template <typename T, bool TWO, int CLS>
__global__ __launch_bounds__((plane_threads<T, TWO>(CLS))) void k_conv_plane(
    const ConvPair* __restrict__ pairs, const SphSide* __restrict__ sides, ConvArgs a,
    PlaneArgs pa, const z64* __restrict__ Wy, const z64* __restrict__ Wz)
{
    extern __shared__ __attribute__((aligned(16))) char cv_smem[];
    const int NW = blockDim.x >> 6;
    PlaneJob<T, TWO> jb;
    if (!jb.init(pairs, sides, a)) return;
    const int Ny = a.Ny, Nz = a.Nz;
    cpx<T>* P = reinterpret_cast<cpx<T>*>(cv_smem + pa.s_bytes);
    unsigned short* yad = reinterpret_cast<unsigned short*>(P + a.nzk_max * pa.prow);
    short* zl = reinterpret_cast<short*>(yad + Ny);
    unsigned short* sl = reinterpret_cast<unsigned short*>(zl + Nz);
    cpx<T>* twy = reinterpret_cast<cpx<T>*>(cv_smem + pa.tw);
    cpx<T>* twz = twy + Ny;
    for (int f = threadIdx.x; f < Ny; f += blockDim.x)
        twy[f] = to<T>(ln_tw<-1>(Wy, (f / pa.R2y) * (f % pa.R2y)));
    for (int f = threadIdx.x; f < Nz; f += blockDim.x)
        twz[f] = to<T>(ln_tw<-1>(Wz, (f / pa.R2z) * (f % pa.R2z)));
    plane_tables(jb.zc, Ny, Nz, false, pa.R1y, pa.R2y, yad, zl);
    plane_sticks(jb.smap, jb.nzk * Ny, sl);
    __syncthreads();
    for (int t = jb.t0; t < jb.t1; ++t)
    {
        // opaque per set, or the compiler would hoist the addresses and
        // twiddles of every length's case out of this loop and spill them
        int tid = threadIdx.x;
        asm volatile("" : "+v"(tid));
        const ConvSrc<T> q = jb.src(t);
        switch (Nz)
        {
#define CV_CASE(L, A, B)                                                                          \
    case L:                                                                                       \
        if constexpr (rx_class(A, B) <= CLS)                                                      \
            plane_z_rows<T, TWO, A, B>(q, Ny, LnLds<B, T>{twz}, cv_smem, P, pa.prow, yad, zl, NW, \
                                       tid);                                                      \
        break;
            RX_LENGTHS(CV_CASE)
#undef CV_CASE
            default: break;
        }
        lds_barrier();
        const gptr<T> out = jb.out + (t - jb.t0) * jb.outs;
        switch (Ny)
        {
#define CV_CASE(L, A, B)                                                                          \
    case L:                                                                                       \
        if constexpr (rx_class(A, B) <= CLS)                                                      \
            plane_y_out<T, A, B>(P, jb.nzk, LnLds<B, T>{twy}, sl, out, NW, tid);                  \
        break;
            RX_LENGTHS(CV_CASE)
#undef CV_CASE
            default: break;
        }
        lds_barrier();
    }
}

// square planes, Ny = Nz = R1 R2: dV stays in registers over the sets of the
// block as far as it fits (sq_keep), the next rows' psi (the next set's first
// rows at the end) are loaded before the second step of the current ones and
// stay in flight over the y transform.
// (FP32: registers for three waves per SIMD)
template <typename T, int R1, int R2, int NW>
__global__ __launch_bounds__(64 * NW, (sizeof(T) == 4 ? 3 : 1)) void k_conv_square(
    const ConvPair* __restrict__ pairs, const SphSide* __restrict__ sides, ConvArgs a,
    const z64* __restrict__ W)
{
    extern __shared__ __attribute__((aligned(16))) char cv_smem[];
    constexpr int N = R1 * R2, LR = ln_rows(R2), PR = ln_prow(R1, R2);
    constexpr int G = sq_groups(R1, R2, NW), P2 = R2 | 1;
    constexpr int SB = (NW * ln_space(R2) * ln_row_bytes<T>(R1, R2) + 15) & ~15;
    PlaneJob<T, false> jb;
    if (!jb.init(pairs, sides, a)) return;
    cpx<T>* P = reinterpret_cast<cpx<T>*>(cv_smem + SB);
    unsigned short* sl = reinterpret_cast<unsigned short*>(P + a.nzk_max * PR);
    plane_sticks(jb.smap, jb.nzk * N, sl);
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int j = lane % R2, r = lane / R2, k1 = lane % R1, rd = lane / R1;
    char* Sw = cv_smem + wave * ln_space(R2) * ln_row_bytes<T>(R1, R2);
    // column offsets of the kept Gz, two to a register
    unsigned po[(R2 + 1) / 2] = {};
#pragma unroll
    for (int k = 0; k < R2; ++k)
    {
        const int c = jb.zc[k1 + R1 * k];
        po[k / 2] |= (c >= 0 ? (unsigned)(c * PR) : 0xffffu) << (16 * (k & 1));
    }
    // twiddles of this lane's j, for both axes: in registers, or where those
    // are short (FP64) in LDS
    constexpr bool TL = sq_tw_lds(R1), TZ = sizeof(T) == 4;
    z64 tw[TL ? 1 : R1];
    cpx<T> tz[TZ ? R1 : 1];
    cpx<T>* twl = reinterpret_cast<cpx<T>*>(
        cv_smem + SB + ((sizeof(cpx<T>) * (size_t)a.nzk_max * PR + 15) & ~(size_t)15) +
        ((2 * (size_t)a.nzk_max * N + 15) & ~(size_t)15));
    if constexpr (TL)
    {
        for (int f = threadIdx.x; f < N; f += 64 * NW)
            twl[f] = to<T>(ln_tw<-1>(W, (f / R2) * (f % R2)));
        lds_barrier();
    }
    else
#pragma unroll
        for (int k = 1; k < R1; ++k) tw[k] = ln_tw<-1>(W, j * k);
    if constexpr (TZ)
#pragma unroll
        for (int k = 1; k < R1; ++k) tz[k] = to<T>(ln_tw<-1>(W, j * k));
    auto twid = [&]() {
        if constexpr (TL)
            return LnLds<R2, T>{twl};
        else
            return LnHeld{tw};
    };
    auto row_of = [&](int g) {
        return min((g * NW + wave) * LR + r, N - 1) * N;
    };
    constexpr int KG = sq_keep<T>(R1, R2, NW);
    cpx<T> p[R1], d[KG > 0 ? KG : 1][R1];
    auto load = [&](cpx<T>* x, gptr<T> src) { ln_load<R1, R2>(x, src, j); };
    ConvSrc<T> q = jb.src(jb.t0);
    gptr<T> dv = q.v0;
    load(p, q.p0 + row_of(0));
#pragma unroll
    for (int g = 0; g < KG; ++g) load(d[g], dv + row_of(g));
    for (int t = jb.t0; t < jb.t1; ++t)
    {
        const ConvSrc<T> qn = jb.src(t + 1 < jb.t1 ? t + 1 : t);
#pragma unroll
        for (int g = 0; g < G; ++g)
        {
            const int y0 = (g * NW + wave) * LR;
            if (y0 < N) // uniform over the wave
            {
                cpx<T> x[R1], v[R2];
                if (g >= KG) load(x, dv + row_of(g));
#pragma unroll
                for (int i = 0; i < R1; ++i) x[i] = cmul(g < KG ? d[g < KG ? g : 0][i] : x[i], p[i]);
                Rdft<T, -1, R1>::run(x);
#pragma unroll
                for (int k = 1; k < R1; ++k) 
                    if constexpr (TZ)
                        x[k] = cmul(x[k], tz[k]);
                    else
                        x[k] = cmul(x[k], to<T>(twid()(j, k)));
                // the next rows that this wave has, or the next set's first
                const bool more = g + 1 < G && y0 + NW * LR < N;
                load(p, (more ? q.p0 : qn.p0) + row_of(more ? g + 1 : 0));
                ln_exchange<T, R1, R2>(x, v, Sw, r, j, rd, k1);
                Rdft<T, -1, R2>::run(v);
                if (rd < LR && y0 + rd < N)
                {
                    const int y = y0 + rd;
                    cpx<T>* o = P + (y / R2) * P2 + y % R2;
#pragma unroll
                    for (int k = 0; k < R2; ++k)
                    {
                        const unsigned c = k & 1 ? po[k / 2] >> 16 : po[k / 2] & 0xffffu;
                        if (c != 0xffffu) o[c] = v[k];
                    }
                }
            }
        }
        if (qn.v0.p != dv.p)
        {
            // the other spin's potential from here on
            dv = qn.v0;
#pragma unroll
            for (int g = 0; g < KG; ++g) load(d[g], dv + row_of(g));
        }
        q = qn;
        lds_barrier();
        plane_y_out<T, R1, R2>(P, jb.nzk, twid(), sl, jb.out, NW, threadIdx.x);
        jb.out = jb.out + jb.outs;
        lds_barrier();
    }
}

// psi_k(r): per x plane the sticks into the plane buffer, y in place, z rows
// out.  Block: (x, row, side).
template <typename T, int CLS, int NT>
__global__ __launch_bounds__(NT) void k_box_plane(const SphSide* __restrict__ sides, BoxArgs a,
                                                  PlaneArgs pa, const z64* __restrict__ Wy,
                                                  const z64* __restrict__ Wz)
{
    extern __shared__ __attribute__((aligned(16))) char cv_smem[];
    int x, row, ks;
    if (!plane_decode(a.Nx, (int)a.nrows, x, row, ks)) return;
    const SphSide& sd = sides[ks];
    const int nzk = sd.cnt[0], nst = sd.cnt[1];
    if (nst == 0) return;
    const int Ny = a.Ny, Nz = a.Nz, tid = threadIdx.x;
    cpx<T>* P = reinterpret_cast<cpx<T>*>(cv_smem + pa.s_bytes);
    unsigned short* yad = reinterpret_cast<unsigned short*>(P + a.nzk_max * pa.prow);
    short* zl = reinterpret_cast<short*>(yad + Ny);
    plane_tables(g_of(sd.zc), Ny, Nz, true, pa.R1y, pa.R2y, yad, zl);
    const auto in = gptr<T>::of(sd.line) + ((int64_t)row * a.Nx + x) * nst;
    const auto smap = g_of(sd.smap);
    const int P2 = pa.R2y | 1;
    for (int f = tid; f < nzk * Ny; f += NT)
    {
        const int c = f / Ny, y = f - c * Ny;
        const int s = smap[f];
        P[c * pa.prow + (y / pa.R2y) * P2 + y % pa.R2y] = s >= 0 ? in[s] : cpx<T>{0, 0};
    }
    __syncthreads();
    switch (Ny)
    {
#define CV_CASE(L, A, B)                                                                          \
    case L:                                                                                       \
        if constexpr (rx_class(A, B) <= CLS)                                                      \
        {                                                                                         \
            plane_y_lds<T, 1, A, B, NT / 64>(P, nzk, Wy, tid);                                    \
        }                                                                                         \
        break;
        RX_LENGTHS(CV_CASE)
#undef CV_CASE
        default: break;
    }
    lds_barrier();
    const auto out = gptr<T>::of(sd.box) + ((int64_t)row * a.Nx + x) * Ny * Nz;
    switch (Nz)
    {
#define CV_CASE(L, A, B)                                                                          \
    case L:                                                                                       \
        if constexpr (rx_class(A, B) <= CLS)                                                      \
            plane_z_backward<T, A, B, NT / 64>(P, pa.prow, yad, zl, Ny, Wz, cv_smem, out, tid);   \
        break;
        RX_LENGTHS(CV_CASE)
#undef CV_CASE
        default: break;
    }
}

// sticks per tile of the x kernels: rows of 256 bytes
template <typename T>
constexpr int x_tile()
{
    return 256 / (int)sizeof(cpx<T>);
}
#define X_THREADS 256

template <typename T>
static inline size_t x_lds(int R1, int R2)
{
    constexpr int TS = x_tile<T>();
    return sizeof(cpx<T>) * (size_t)(TS * ln_xrow(R1, R2)) + ((TS * R1 * R2 + 15) & ~15) +
           sizeof(int) * TS;
}

template <typename T, int CLS>
__global__ __launch_bounds__(X_THREADS) void k_conv_x(const ConvPair* __restrict__ pairs,
                                                      const SphSide* __restrict__ sides,
                                                      ConvArgs a, const z64* __restrict__ W)
{
    extern __shared__ __attribute__((aligned(16))) char cv_smem[];
    const ConvPair& pr = pairs[blockIdx.z];
    const SphSide& sd = sides[pr.side];
    switch (a.Nx)
    {
#define CV_CASE(L, A, B)                                                                          \
    case L:                                                                                       \
        if constexpr (rx_class(A, B) <= CLS)                                                      \
            conv_x_body<T, A, B, x_tile<T>(), X_THREADS>(                                         \
                pr, sd, a, W, blockIdx.x, (int64_t)blockIdx.y * a.rows_per_block, cv_smem);       \
        break;
        RX_LENGTHS(CV_CASE)
#undef CV_CASE
        default: break;
    }
}

template <typename T, int CLS>
__global__ __launch_bounds__(X_THREADS) void k_box_x(const SphSide* __restrict__ sides, BoxArgs a,
                                                     const z64* __restrict__ W)
{
    extern __shared__ __attribute__((aligned(16))) char cv_smem[];
    const SphSide& sd = sides[blockIdx.z];
    switch (a.Nx)
    {
#define CV_CASE(L, A, B)                                                                          \
    case L:                                                                                       \
        if constexpr (rx_class(A, B) <= CLS)                                                      \
            box_x_body<T, A, B, x_tile<T>(), X_THREADS>(                                          \
                sd, a, blockIdx.x, (int64_t)blockIdx.y * a.rows_per_block, W, cv_smem);           \
        break;
        RX_LENGTHS(CV_CASE)
#undef CV_CASE
        default: break;
    }
}

// ---------------------------------------------------------------------------
// g[nu][is][n][m] = scale sum_{sigma, p} C[nu][is][n][sigma][p]
//                                       conj(W[is][m][sigma][p])
// Rows r = (nu, n), columns m; 4 waves of RB x CB blocks of 16 x 16, WR x WC
// of them.  Chunks of 16 points are loaded a chunk ahead into registers and
// double buffered in LDS (one barrier per chunk).  FP32 operands are
// multiplied and summed in FP64 too: half the MFMA rate, 0.3 of 3.4 ms for a
// 72^3 pair of 64 bands, and the largest error of the FP32 form gone (see
// above).  blockIdx.y: K split (partials in FP64, summed in fixed order by
// k_reduce_parts; one split writes g itself), blockIdx.z: (pair, spin).
#define SG_KC 16
template <typename T, int RB, int CB, int WR, int WC>
__global__ __launch_bounds__(256) void k_sph_gemm(const ConvPair* __restrict__ pairs,
                                                  const SphSide* __restrict__ sides, int nm,
                                                  int nspin, int nb, int nspinor, int nsplit,
                                                  int npairs, double scale,
                                                  z64* __restrict__ out)
{
    typedef typename Mfma<double>::acc acc_t;
    constexpr int MB = 16 * RB * WR, NB = 16 * CB * WC, LD = SG_KC + 1;
    constexpr int LA = MB * SG_KC / 256, LB = (NB * SG_KC + 255) / 256;
    __shared__ cpx<T> sA[2][MB][LD];
    __shared__ cpx<T> sB[2][NB][LD];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int ip = blockIdx.z / nspin, is = blockIdx.z % nspin;
    const ConvPair& pr = pairs[ip];
    const SphSide& sd = sides[pr.side];
    const int ntm = (nb + NB - 1) / NB;
    const int m0 = (blockIdx.x % ntm) * NB, r0 = (blockIdx.x / ntm) * MB;
    const int M = nm * nb, npw = sd.npw;
    const int64_t ld = sd.ld;
    const int nck = (npw + SG_KC - 1) / SG_KC, tot = nck * nspinor;
    const int cps = (tot + nsplit - 1) / nsplit;
    const int c0 = blockIdx.y * cps, c1 = min(c0 + cps, tot);
    const int wr = wave / WC, wc = wave % WC;
    const auto C = gptr<T>::of(pr.c), W = gptr<T>::of(sd.coef);
    const int kk = tid % SG_KC;
    gptr<T> pA[LA], pB[LB];
#pragma unroll
    for (int u = 0; u < LA; ++u)
    {
        const int r = min(r0 + tid / SG_KC + u * (256 / SG_KC), M - 1);
        const int v = r / nb, n = r - v * nb;
        pA[u] = C + (((int64_t)(v * nspin + is) * nb + n) * nspinor * ld + kk);
    }
#pragma unroll
    for (int u = 0; u < LB; ++u)
    {
        const int m = min(m0 + tid / SG_KC + u * (256 / SG_KC), nb - 1);
        pB[u] = W + (((int64_t)is * nb + m) * nspinor * ld + kk);
    }
    acc_t accr[RB][CB], acci[RB][CB];
#pragma unroll
    for (int a = 0; a < RB; ++a)
#pragma unroll
        for (int b = 0; b < CB; ++b)
#pragma unroll
            for (int v = 0; v < 4; ++v)
            {
                accr[a][b][v] = 0;
                acci[a][b][v] = 0;
            }
    cpx<T> ra[LA], rb_[LB];
    auto fetch = [&](int c) {
        const int sp = c / nck, k = (c - sp * nck) * SG_KC;
        const int64_t o = (int64_t)sp * ld + k;
        const bool in = k + kk < npw;
#pragma unroll
        for (int u = 0; u < LA; ++u)
        {
            ra[u] = pA[u][in ? o : 0];
            if (!in) ra[u] = {0, 0};
        }
#pragma unroll
        for (int u = 0; u < LB; ++u)
        {
            rb_[u] = pB[u][in ? o : 0];
            if (!in) rb_[u] = {0, 0};
        }
    };
    auto put = [&](int b) {
#pragma unroll
        for (int u = 0; u < LA; ++u) sA[b][tid / SG_KC + u * (256 / SG_KC)][kk] = ra[u];
#pragma unroll
        for (int u = 0; u < LB; ++u)
        {
            const int m = tid / SG_KC + u * (256 / SG_KC);
            if (NB * SG_KC % 256 == 0 || m < NB) sB[b][m][kk] = rb_[u];
        }
    };
    if (c0 < c1)
    {
        fetch(c0);
        put(0);
    }
    lds_barrier();
    for (int c = c0; c < c1; ++c)
    {
        const int b = (c - c0) & 1;
        if (c + 1 < c1) fetch(c + 1);
#pragma unroll
        for (int s = 0; s < SG_KC / 4; ++s)
        {
            const int i = lane & 15, kq = s * 4 + (lane >> 4);
            z64 fa[RB], fb[CB];
#pragma unroll
            for (int a = 0; a < RB; ++a) fa[a] = to<double>(sA[b][(wr * RB + a) * 16 + i][kq]);
#pragma unroll
            for (int q = 0; q < CB; ++q) fb[q] = to<double>(sB[b][(wc * CB + q) * 16 + i][kq]);
#pragma unroll
            for (int a = 0; a < RB; ++a)
#pragma unroll
                for (int q = 0; q < CB; ++q)
                {
                    accr[a][q] = Mfma<double>::op(fa[a].x, fb[q].x, accr[a][q]);
                    acci[a][q] = Mfma<double>::op(fa[a].y, fb[q].x, acci[a][q]);
                }
#pragma unroll
            for (int a = 0; a < RB; ++a)
#pragma unroll
                for (int q = 0; q < CB; ++q)
                {
                    accr[a][q] = Mfma<double>::op(fa[a].y, fb[q].y, accr[a][q]);
                    acci[a][q] = Mfma<double>::op(-fa[a].x, fb[q].y, acci[a][q]);
                }
        }
        if (c + 1 < c1) put(b ^ 1);
        lds_barrier();
    }
    const int64_t gsz = (int64_t)nm * nspin * nb * nb;
    z64* o = out + ((int64_t)(nsplit > 1 ? blockIdx.y * npairs : 0) + ip) * gsz;
    const double sc = nsplit > 1 ? 1.0 : scale;
#pragma unroll
    for (int a = 0; a < RB; ++a)
#pragma unroll
        for (int q = 0; q < CB; ++q)
#pragma unroll
            for (int e = 0; e < 4; ++e)
            {
                const int r = r0 + (wr * RB + a) * 16 + Mfma<double>::row(lane, e);
                const int m = m0 + (wc * CB + q) * 16 + (lane & 15);
                if (r < M && m < nb)
                {
                    const int v = r / nb, n = r - v * nb;
                    o[((int64_t)(v * nspin + is) * nb + n) * nb + m] = {
                        sc * accr[a][q][e], sc * acci[a][q][e]};
                }
            }
}
