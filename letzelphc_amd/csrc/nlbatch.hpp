// nlbatch.hpp -- the non-local part of many pairs at once (add_elphNonLocal,
// src/nonloc/Vbare_nloc.c:397-558): every (iBZ k, symmetry) side that the
// pairs touch is projected once, <beta_K|psi> of all sides in three launches
// (k_nl_sides, k_nl_gemm, k_nl_reduce), then the K/K' sums and the mode
// rotation of all pairs in one launch each.  A side serves as k+q of one pair
// and as k of another: its K' projections are read from the K ones, bbKp =
// diag(1, -1, -1, -1) conj(bbK) row by row of four, exact (the K' projectors
// are the conjugates of the K ones, the K-weighted rows with the opposite
// sign, psi enters conjugated the other way).
//
// A pair on its own took 10 to 13 launches; 64 pairs of a 24^3 cell 2.35 ms
// of them, 0.2 ms now (all of g: 3.2 -> 0.62 ms).  Included by lelph_hip.hip.
#pragma once

struct NlKey
{
    const double* gvec;
    const z64* wfc;
    const double* Fk;
    int64_t npw;
    NlSide sd;
    void* wr;   // (ncol, npw) rotated psi
    void* beta; // (rows, npw)
    z64* part;  // (nsplit, rows, ncol)
    z64* bb;    // (rows, ncol)
    int64_t cps;
    int nsplit;
};

// Rotated psi (blockIdx.y < ngy: sets in groups of spy) and projectors
// (blockIdx.y - ngy: NL_PROJ of an atom, beta[(a*pmax + p)*4 + x][G] = F_l(K)
// e^{-2 pi i K.tau_a} Y_lm(K), and K-weighted) of one side (blockIdx.z).  The
// phase and the direction of K are formed once per thread (with one projector
// per thread they were most of its time); tables of them would cost a launch.
#define NL_PROJ 4
template <typename T>
__global__ __launch_bounds__(128) void k_nl_sides(
    const NlKey* __restrict__ keys, int64_t nsets, int nspinor, int spy, int ngy, NlProj pj,
    const int* __restrict__ plist, const int* __restrict__ atype, const double* __restrict__ apos,
    const double* __restrict__ Fsign)
{
    const NlKey& k = keys[blockIdx.z];
    const int64_t npw = k.npw, g = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (g >= npw) return;
    const NlSide& sd = k.sd;
    const auto gv = g_of(k.gvec);
    const double t[3] = {sd.k[0] + gv[3 * g], sd.k[1] + gv[3 * g + 1], sd.k[2] + gv[3 * g + 2]};
    double K[3];
    for (int i = 0; i < 3; ++i)
        K[i] = sd.S[3 * i] * t[0] + sd.S[3 * i + 1] * t[1] + sd.S[3 * i + 2] * t[2];
    double s, c;
    if ((int)blockIdx.y < ngy)
    {
        sincos(-2.0 * LELPH_RPI * (K[0] * sd.tau[0] + K[1] * sd.tau[1] + K[2] * sd.tau[2]), &s, &c);
        const z64 ph = {c, s};
        const int64_t s0 = (int64_t)blockIdx.y * spy;
        const int64_t s1 = s0 + spy < nsets ? s0 + spy : nsets;
        for (int64_t st = s0; st < s1; ++st)
        {
            const auto w = gptr<double>::of(k.wfc) + st * nspinor * npw;
            const auto o = gptr<T>::of(k.wr) + st * nspinor * npw;
            if (nspinor == 1)
            {
                const z64 v = cmul(w[g], ph);
                o.set(g, {(T)v.x, (T)v.y});
            }
            else
            {
                const z64 u = w[g], d = w[npw + g];
                const z64 a = cmul(cadd(cmul(u, sd.su2[0]), cmul(d, sd.su2[1])), ph);
                const z64 b = cmul(cadd(cmul(u, sd.su2[2]), cmul(d, sd.su2[3])), ph);
                o.set(g, {(T)a.x, (T)a.y});
                o.set(npw + g, {(T)b.x, (T)b.y});
            }
        }
        return;
    }
    const int npg = (pj.pmax + NL_PROJ - 1) / NL_PROJ, yb = blockIdx.y - ngy, a = yb / npg;
    const int p0 = (yb % npg) * NL_PROJ, p1 = min(p0 + NL_PROJ, pj.pmax);
    const int ty = atype[a];
    const double* tau = apos + 3 * a;
    sincos(-2.0 * LELPH_RPI * (K[0] * tau[0] + K[1] * tau[1] + K[2] * tau[2]), &s, &c);
    const YlmDir dir(K);
    for (int p = p0; p < p1; ++p)
    {
        const int ap = a * pj.pmax + p;
        const int* e = plist + 3 * ap;
        const auto b = gptr<T>::of(k.beta) + (int64_t)ap * 4 * npw;
        if (e[0] < 0)
        {
            for (int x = 0; x < 4; ++x) b.set((int64_t)x * npw + g, {0, 0});
            continue;
        }
        const int lidx = e[0], l = e[1];
        const double f =
            g_of(k.Fk)[((int64_t)lidx * pj.ntype + ty) * npw + g] * d_Ylm(l, e[2] - l * l - l, dir);
        const z64 b0 = {f * c, f * s};
        const double sg = Fsign[lidx * pj.ntype + ty];
        b.set(g, {(T)b0.x, (T)b0.y});
        for (int x = 0; x < 3; ++x)
        {
            const double kx = K[x] * sg;
            b.set((int64_t)(x + 1) * npw + g, {(T)(b0.x * kx), (T)(b0.y * kx)});
        }
    }
}

// the projector GEMMs of all sides: blockIdx.y split, blockIdx.z side
template <typename T>
__global__ __launch_bounds__(256) void k_nl_gemm(const NlKey* __restrict__ keys, int M, int Nc)
{
    const NlKey& k = keys[blockIdx.z];
    if ((int)blockIdx.y >= k.nsplit) return;
    zgemm_nt_body<T>(gptr<T>::of(k.beta), gptr<T>::of(k.wr), M, Nc, k.npw, k.sd.conj_w, k.cps,
                     k.part);
}

__global__ __launch_bounds__(256) void k_nl_reduce(const NlKey* __restrict__ keys, int64_t count)
{
    const NlKey& k = keys[blockIdx.y];
    reduce_body(gptr<double>::of(k.part), k.nsplit, count, 1.0, gptr<double>::of(k.bb));
}

// ebuf[pair][a][x][s][n][m] = sum f (K3_x[m] Kp0[n] + K0[m] Kp3_x[n]) over
// the projectors of an atom (sum_VNL_KKp); bb rows (a*pmax+p)*4+x, columns
// (s*nb + b)*nspinor + sigma.  blockIdx.y: pair, kk its two sides (k+q, k).
__global__ __launch_bounds__(256) void k_nl_kkp(
    const z64* __restrict__ bb, const int* __restrict__ kk, int64_t bbs, NlProj pj,
    const int* __restrict__ plist, const int* __restrict__ atype,
    const double* __restrict__ socfac,   // (nltimesj, ntype)
    const z64* __restrict__ fco,         // packed f coefficients or null
    const int64_t* __restrict__ fco_off, // (nltimesj*ntype) offsets or -1
    int nspin, int nb, int nspinor, z64* __restrict__ ebuf)
{
    const int64_t per_a = (int64_t)3 * nspin * nb * nb;
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= (int64_t)pj.natom * per_a) return;
    const z64* bbK = bb + kk[2 * blockIdx.y] * bbs;
    const z64* bbKp = bb + kk[2 * blockIdx.y + 1] * bbs;
    const int a = (int)(t / per_a);
    int64_t r = t - a * per_a;
    const int x = (int)(r / ((int64_t)nspin * nb * nb));
    r -= (int64_t)x * nspin * nb * nb;
    const int s = (int)(r / ((int64_t)nb * nb));
    r -= (int64_t)s * nb * nb;
    const int n = (int)(r / nb), m = (int)(r % nb);
    const int ty = atype[a];
    const int64_t ncol = (int64_t)nspin * nb * nspinor;
    z64 acc = {0, 0};
    for (int p1 = 0; p1 < pj.pmax; ++p1)
    {
        const int* e1 = plist + 3 * (a * pj.pmax + p1);
        if (e1[0] < 0) continue;
        const z64* K0 = bbK + ((int64_t)(a * pj.pmax + p1) * 4 + 0) * ncol;
        const z64* K3 = bbK + ((int64_t)(a * pj.pmax + p1) * 4 + 1 + x) * ncol;
        for (int p2 = 0; p2 < pj.pmax; ++p2)
        {
            const int* e2 = plist + 3 * (a * pj.pmax + p2);
            if (e2[0] != e1[0]) continue;
            const int lidx = e1[0], l = e1[1];
            const int64_t off = fco_off ? fco_off[lidx * pj.ntype + ty] : -1;
            if (off < 0 && p1 != p2) continue;
            const z64* Kp0 = bbKp + ((int64_t)(a * pj.pmax + p2) * 4 + 0) * ncol;
            const z64* Kp3 = bbKp + ((int64_t)(a * pj.pmax + p2) * 4 + 1 + x) * ncol;
            const int m1 = e1[2] - l * l, m2 = e2[2] - l * l;
            for (int s1 = 0; s1 < nspinor; ++s1)
                for (int s2 = 0; s2 < nspinor; ++s2)
                {
                    z64 f;
                    if (off >= 0)
                        f = fco[off + ((int64_t)(2 * l + 1) * m1 + m2) * nspinor * nspinor +
                                nspinor * s1 + s2];
                    else
                        f = {s1 == s2 ? socfac[lidx * pj.ntype + ty] : 0.0, 0.0};
                    if (f.x == 0.0 && f.y == 0.0) continue;
                    const int64_t cm = ((int64_t)s * nb + m) * nspinor + s1;
                    const int64_t cn = ((int64_t)s * nb + n) * nspinor + s2;
                    const z64 q0 = {Kp0[cn].x, -Kp0[cn].y}, q3 = {-Kp3[cn].x, Kp3[cn].y};
                    acc = cadd(acc, cmul(f, cadd(cmul(K3[cm], q0), cmul(K0[cm], q3))));
                }
        }
    }
    ebuf[(int64_t)blockIdx.y * pj.natom * per_a + t] = acc;
}

// g[pair][v][s][n][m] += pre * sum_j eig[v][j] ebuf[pair][j][s][n][m], j = (a, x).
// Four modes per thread: ebuf passes through L2 a quarter as often.
#define NL_MODES 4
__global__ __launch_bounds__(256) void k_nl_mode(const z64* __restrict__ ebuf,
                                                 const z64* __restrict__ eig, int nm, int n3a,
                                                 int64_t es, z64 pre, z64* __restrict__ g)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= es) return;
    const int v0 = blockIdx.y * NL_MODES;
    const z64* e = ebuf + (int64_t)blockIdx.z * n3a * es + i;
    z64 acc[NL_MODES];
#pragma unroll
    for (int u = 0; u < NL_MODES; ++u) acc[u] = {0, 0};
#pragma unroll 4
    for (int j = 0; j < n3a; ++j)
    {
        const z64 x = e[(int64_t)j * es];
#pragma unroll
        for (int u = 0; u < NL_MODES; ++u)
            acc[u] = cadd(acc[u], cmul(eig[(int64_t)min(v0 + u, nm - 1) * n3a + j], x));
    }
    z64* o = g + ((int64_t)blockIdx.z * nm + v0) * es + i;
#pragma unroll
    for (int u = 0; u < NL_MODES; ++u)
        if (v0 + u < nm) o[u * es] = cadd(o[u * es], cmul(pre, acc[u]));
}
