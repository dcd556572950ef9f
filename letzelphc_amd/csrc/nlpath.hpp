// nlpath.hpp -- host side of the non-local part (nlbatch.hpp), included by
// lelph_hip.hip.
#pragma once

// scratch of a set of sides whose projections are formed together
#define NL_SCRATCH_BYTES ((size_t)1 << 30)
// pairs whose sides are projected ahead of them, and the projections' bytes
#define NL_WINDOW_PAIRS 256
#define NL_WINDOW_BYTES ((size_t)1 << 30)
// sets of a block row of k_nl_sides
#define NL_SPY 16

struct NlDims
{
    int rows = 0;
    int64_t ncol = 0, es = 0;
    bool f32 = false, split = false;
    explicit NlDims(const lelph_ctx* c)
    {
        const lelph_lattice& L = c->lat;
        const int prec = effective_precision(c);
        rows = L.natom * c->pmax * 4;
        ncol = (int64_t)L.nspin * L.nbnds * L.nspinor;
        es = (int64_t)L.nspin * L.nbnds * L.nbnds;
        // bf16 contexts: FP32 operands on FP32 MFMA by default (closer than
        // the bf16 pieces: 1.3-1.9e-7 against 2.1-2.6e-7 of the non-local
        // part alone, and 0.16 against 0.46 ms at 128 bands); nl_form 1: bf16
        // pieces, 3 of them and 6 products for both split precisions (the
        // 2-piece form left 8.5e-6)
        split = (prec == LELPH_BF16X3 || prec == LELPH_BF16X6) && c->tune.nl_form == 1;
        f32 = prec != LELPH_FP64 && !split;
    }
};

// pairs per window: of `step` pairs at a time
static int64_t nl_window(const lelph_ctx* c, int64_t step, int64_t npairs)
{
    const NlDims d(c);
    const int64_t per = 2 * (int64_t)sizeof(z64) * d.rows * d.ncol;
    const int64_t fit = std::min<int64_t>(NL_WINDOW_PAIRS, (int64_t)NL_WINDOW_BYTES / std::max<int64_t>(per, 1));
    return std::min(npairs, std::max<int64_t>(1, fit / step) * step);
}

// one side's <beta|psi> projector GEMM into out (rows, ncol) from the beta /
// psi pieces of k_nl_presplit on BF16 MFMA (NP pieces, NPROD products),
// FP64 split-K partials and a fixed-order FP64 reduction
template <int NP, int NPROD>
static int nl_gemm_split(NlBufs& b, const z64* A, const z64* B, int rows, int64_t ncol,
                         int64_t npw, int conjB, z64* part, int64_t cps, int nsplit, z64* out,
                         hipStream_t st)
{
    const int Mp = (int)(cdiv(rows, 64) * 64), Np = (int)(cdiv(ncol, 64) * 64);
    const int64_t Kp = cdiv(npw, 32) * 32;
    hipLaunchKernelGGL((k_nl_presplit<NP>), dim3((unsigned)cdiv(Kp, 256), (unsigned)Mp), dim3(256),
                       0, st, A, rows, npw, Mp, Kp, 0, b.splitA.as<__bf16>());
    hipLaunchKernelGGL((k_nl_presplit<NP>), dim3((unsigned)cdiv(Kp, 256), (unsigned)Np), dim3(256),
                       0, st, B, (int)ncol, npw, Np, Kp, conjB, b.splitB.as<__bf16>());
    const int64_t tiles = (int64_t)(Mp / 64) * (Np / 64);
    hipLaunchKernelGGL((k_zgemm_nt_bf<NP, NPROD>), dim3((unsigned)tiles, (unsigned)nsplit),
                       dim3(256), 0, st, b.splitA.as<__bf16>(), b.splitB.as<__bf16>(), rows,
                       (int)ncol, Mp, Np, Kp, cps, part);
    HIP_TRY(hipGetLastError());
    return reduce_parts(part, nsplit, (int64_t)rows * ncol, 1.0, out, st);
}

static int nl_check(const lelph_ctx* c, const NlWindow& w)
{
    for (const auto& k : w.keys)
        if (!c->wf[k[0]].wfc || !c->wf[k[0]].Fk) return LELPH_ERR_STATE;
    return LELPH_OK;
}

// the GEMM splits of a window's sides and the bytes it takes
struct NlLayout
{
    std::vector<int64_t> cps;
    std::vector<int> nsplit;
    size_t side_max = 0; // scratch of a side
    int per = 1;         // sides formed together
    size_t side = 0, bb = 0, splitA = 0, splitB = 0;
    NlLayout(const lelph_ctx* c, const NlDims& d, const NlWindow& w)
    {
        const size_t nk = w.keys.size(), item = d.f32 ? sizeof(c32) : sizeof(z64);
        const int64_t count = d.rows * d.ncol;
        const int64_t tiles = cdiv(d.rows, GZ_MB) * cdiv(d.ncol, GZ_NB);
        int64_t npw_max = 0;
        cps.resize(nk);
        nsplit.resize(nk);
        for (size_t i = 0; i < nk; ++i)
        {
            const int64_t npw = c->wf[w.keys[i][0]].npw;
            pick_splits(tiles, cdiv(npw, d.split ? 32 : CT_KC), count, &cps[i], &nsplit[i]);
            npw_max = std::max(npw_max, npw);
            const size_t one = item * (size_t)npw * (d.ncol + d.rows) +
                               sizeof(z64) * (size_t)(nsplit[i] * count) + 64;
            side_max = std::max(side_max, (one + 255) & ~(size_t)255);
        }
        per = (int)std::max<size_t>(1, std::min<size_t>(nk, NL_SCRATCH_BYTES / side_max));
        side = side_max * per;
        bb = sizeof(z64) * nk * (size_t)count;
        if (d.split)
        {
            const int64_t Kp = cdiv(npw_max, 32) * 32;
            splitA = sizeof(__bf16) * 6 * (size_t)(cdiv(d.rows, 64) * 64 * Kp);
            splitB = sizeof(__bf16) * 6 * (size_t)(cdiv(d.ncol, 64) * 64 * Kp);
        }
    }
    int ensure(NlBufs& b, hipStream_t st) const
    {
        LELPH_TRY(buf_grow(b.side, side, b.fixed, st));
        LELPH_TRY(buf_grow(b.bb, bb, b.fixed, st));
        LELPH_TRY(buf_grow(b.splitA, splitA, b.fixed, st));
        return buf_grow(b.splitB, splitB, b.fixed, st);
    }
};

// Sizes b for all of these windows, for good: their descriptors, which hold
// its addresses, are run again by a captured pass.
static int nl_reserve(const lelph_ctx* c, NlBufs& b, const std::vector<NlWindow>& win,
                      hipStream_t st)
{
    const NlDims d(c);
    for (const NlWindow& w : win)
    {
        LELPH_TRY(nl_check(c, w));
        LELPH_TRY(NlLayout(c, d, w).ensure(b, st));
    }
    b.fixed = true;
    return LELPH_OK;
}

// <beta_K|psi> of the window's sides into b.bb on stream st.  upload: the
// descriptors are copied over (a captured pass finds them there).  Nothing
// of an earlier window may still run on another stream than st.
template <typename T>
static int nl_sides_t(lelph_ctx* c, NlBufs& b, DBuf& desc, const NlWindow& w, bool upload,
                      hipStream_t st)
{
    const lelph_lattice& L = c->lat;
    const NlDims d(c);
    const int64_t nsb = (int64_t)L.nspin * L.nbnds, count = d.rows * d.ncol;
    const int nk = (int)w.keys.size();
    LELPH_TRY(nl_check(c, w));
    const NlLayout lay(c, d, w);
    const size_t side_max = lay.side_max;
    const int per = lay.per;
    std::vector<NlKey> hk((size_t)nk);
    for (int i = 0; i < nk; ++i)
    {
        const DevWfc& v = c->wf[w.keys[i][0]];
        const lelph_symmetry& S = c->syms[w.keys[i][1]];
        NlKey& k = hk[i];
        k = NlKey{};
        k.gvec = v.gvec;
        k.wfc = v.wfc;
        k.Fk = v.Fk;
        k.npw = v.npw;
        k.cps = lay.cps[i];
        k.nsplit = lay.nsplit[i];
        std::memcpy(k.sd.S, S.Rmat, sizeof(k.sd.S));
        std::memcpy(k.sd.k, c->kpt_ibz.data() + 3 * w.keys[i][0], sizeof(k.sd.k));
        std::memcpy(k.sd.tau, S.tau, sizeof(k.sd.tau));
        k.sd.conj_w = S.time_rev ? 0 : 1; // 'C' unless time reversed (Vbare_nloc.c:397-407)
        LELPH_TRY(su2mat(S.Rmat, L.nspinor, S.time_rev, k.sd.su2));
    }
    LELPH_TRY(lay.ensure(b, st));
    for (int i = 0; i < nk; ++i)
    {
        NlKey& k = hk[i];
        char* p = b.side.as<char>() + side_max * (i % per);
        k.part = reinterpret_cast<z64*>(p);
        p += sizeof(z64) * (size_t)(k.nsplit * count);
        k.wr = p;
        p += sizeof(cpx<T>) * (size_t)k.npw * d.ncol;
        k.beta = p;
        k.bb = b.bb.as<z64>() + i * count;
    }
    const size_t nb_k = sizeof(NlKey) * (size_t)nk, nb_kk = sizeof(int) * w.kk.size();
    if (upload)
    {
        LELPH_TRY(buf_grow(desc, nb_k + nb_kk, false, st));
        std::vector<char> host(nb_k + nb_kk);
        std::memcpy(host.data(), hk.data(), nb_k);
        std::memcpy(host.data() + nb_k, w.kk.data(), nb_kk);
        HIP_TRY(hipMemcpyAsync(desc.p, host.data(), host.size(), hipMemcpyHostToDevice, st));
    }
    b.kk = reinterpret_cast<const int*>(desc.as<char>() + nb_k);
    const NlProj pj{L.natom, c->pmax, c->ntype};
    const unsigned ngy = (unsigned)cdiv(nsb, NL_SPY);
    for (int k0 = 0; k0 < nk; k0 += per)
    {
        const int n = std::min(per, nk - k0);
        int64_t npw = 0;
        int ns = 0;
        for (int i = k0; i < k0 + n; ++i)
        {
            npw = std::max(npw, hk[i].npw);
            ns = std::max(ns, hk[i].nsplit);
        }
        const NlKey* dk = desc.as<NlKey>() + k0;
        hipLaunchKernelGGL(k_nl_sides<T>,
                           dim3((unsigned)cdiv(npw, 128), ngy + L.natom * (unsigned)cdiv(c->pmax, NL_PROJ),
                                (unsigned)n),
                           dim3(128), 0, st, dk, nsb, L.nspinor, NL_SPY, (int)ngy, pj, c->d_plist,
                           c->d_atype, c->d_apos, c->d_Fsign);
        HIP_TRY(hipGetLastError());
        if (d.split)
        {
            for (int i = k0; i < k0 + n; ++i)
                LELPH_TRY((nl_gemm_split<3, 6>(b, static_cast<z64*>(hk[i].beta),
                                               static_cast<z64*>(hk[i].wr), d.rows, d.ncol,
                                               hk[i].npw, hk[i].sd.conj_w, hk[i].part, hk[i].cps,
                                               hk[i].nsplit, hk[i].bb, st)));
            continue;
        }
        hipLaunchKernelGGL(k_nl_gemm<T>,
                           dim3((unsigned)(cdiv(d.rows, GZ_MB) * cdiv(d.ncol, GZ_NB)),
                                (unsigned)ns, (unsigned)n),
                           dim3(256), 0, st, dk, d.rows, (int)d.ncol);
        hipLaunchKernelGGL(k_nl_reduce, dim3((unsigned)cdiv(count, RP_ELEMS), (unsigned)n),
                           dim3(256), 0, st, dk, count);
        HIP_TRY(hipGetLastError());
    }
    return LELPH_OK;
}

static int nl_sides(lelph_ctx* c, NlBufs& b, DBuf& desc, const NlWindow& w, bool upload,
                      hipStream_t st)
{
    if (!c->dv_set) return LELPH_ERR_STATE;
    return NlDims(c).f32 ? nl_sides_t<float>(c, b, desc, w, upload, st)
                         : nl_sides_t<double>(c, b, desc, w, upload, st);
}

// elements of a pair's K/K' sums
static int64_t nl_sum_size(const lelph_ctx* c)
{
    const lelph_lattice& L = c->lat;
    return (int64_t)L.natom * 3 * L.nspin * L.nbnds * L.nbnds;
}

// per-atom K/K' sums of pairs p0 .. p0 + n - 1 of the window
static int nl_sums(lelph_ctx* c, NlBufs& b, int64_t p0, int64_t n, z64* ebuf, hipStream_t st)
{
    const lelph_lattice& L = c->lat;
    const NlDims d(c);
    const int64_t ne = nl_sum_size(c);
    hipLaunchKernelGGL(k_nl_kkp, dim3((unsigned)cdiv(ne, 256), (unsigned)n), dim3(256), 0, st,
                       b.bb.as<z64>(), b.kk + 2 * p0, (int64_t)d.rows * d.ncol,
                       NlProj{L.natom, c->pmax, c->ntype}, c->d_plist, c->d_atype, c->d_socfac,
                       c->d_fco, c->has_fco ? c->d_fco_off : nullptr, L.nspin, L.nbnds, L.nspinor,
                       ebuf);
    HIP_TRY(hipGetLastError());
    return LELPH_OK;
}

// the cart -> mode rotation of those pairs, accumulated into their g (n
// consecutive matrices): g += -2 pi i e^2 eig ebuf (Vbare_nloc.c:541-558)
static int nl_modes(lelph_ctx* c, const z64* ebuf, int64_t n, z64* g, hipStream_t st)
{
    const lelph_lattice& L = c->lat;
    const int64_t es = (int64_t)L.nspin * L.nbnds * L.nbnds;
    const z64 pre = {0.0, -2 * LELPH_RPI * LELPH_E2};
    const int64_t one = nl_sum_size(c), gsz = (int64_t)L.nmodes * es;
    for (int64_t p = 0; p < n; p += 32768) // grid limit
        hipLaunchKernelGGL(k_nl_mode,
                           dim3((unsigned)cdiv(es, 256), (unsigned)cdiv(L.nmodes, NL_MODES),
                                (unsigned)std::min<int64_t>(32768, n - p)),
                           dim3(256), 0, st, ebuf + p * one, c->eig_d.as<z64>(), L.nmodes,
                           3 * L.natom, es, pre, g + p * gsz);
    HIP_TRY(hipGetLastError());
    return LELPH_OK;
}

// sums and modes of pairs p0 .. p0 + n - 1 of the current window into their g
// (n consecutive matrices) on stream st, which waits for `after` (the pairs'
// local part) before it touches g
static int nl_add(lelph_ctx* c, NlBufs& b, int64_t p0, int64_t n, z64* g, hipStream_t st,
                  hipEvent_t after)
{
    LELPH_TRY(buf_grow(b.ebuf, sizeof(z64) * (size_t)(nl_sum_size(c) * n), false, st));
    LELPH_TRY(nl_sums(c, b, p0, n, b.ebuf.as<z64>(), st));
    if (after) HIP_TRY(hipStreamWaitEvent(st, after, 0));
    return nl_modes(c, b.ebuf.as<z64>(), n, g, st);
}
