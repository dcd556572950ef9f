// convpath.hpp -- host side of the sphere form (conv.hpp): buffers, launch
// shapes and the sequence of one group of (k, k+q) pairs.  Included by
// lelph_hip.hip after the context.
//
// A group of pairs goes through every step in one launch each, so a batch of
// small cells costs a dozen launches and not a dozen per pair; the pairs of
// a large cell go one by one, in chunks of modes whose x lines stay in the
// last-level cache between the plane and the x step.
#pragma once

// sizes and launch shapes of a context's grid, from its spheres' radius
struct ConvGeo
{
    bool f32 = false, two = false;
    int r1[3], r2[3], xcls;
    int words;
    int nzk, nst, npw, ld; // bounds over the context's spheres
    int64_t nrows;         // sets x spinors
    PlaneShape conv, box;
    bool square; // the planes have a kernel of their own
    size_t sqlds;
    size_t xlds;
    int nsplit;
};

// bytes of line buffers (the planes' output) that a launch may fill.  More
// than the 256 MB last-level cache on purpose: fewer, longer launches and
// more sets per psi plane outweigh what the x step finds cached (4 pairs of
// 96^3, 128 bands, FP64: 153 ms with 128 MB, 133 with 512, 128 with 1024, 126
// with 2048; 36 of a 45x45x108 slab 20.2, 14.9, 13.9, 13.6)
static const int64_t CONV_LINE_BYTES = 1024ll << 20;
// modes of a launch that share a psi plane in L2 (96^3 in FP64: 4 costs 5 %,
// 16 2 %; 72^3 in FP32: 1 % either way), sets that a block takes in turn (96^3:
// 32 cost 3 %, the blocks of one psi plane drift apart and miss, 4 cost 2 % in
// starting blocks; 72^3 in FP32: 32 gain 2 to 3 %, 4 cost 8 %)
static const int CONV_MODES = 8, CONV_SETS = 8;
static const int64_t CONV_GROUP_BYTES = 2ll << 30;
// bytes of a pair's coefficients on the k+q sphere, all sets of a block of
// modes (144^3, 96 atoms, 480 bands would take 336 GB at once).  Beyond the
// 96^3 cell's 3.6 GB: a block reads the psi boxes again.
static const int64_t CONV_C_BYTES = 4ll << 30;
static const int CONV_GROUP_PAIRS = 256;

// threads of the blocks over planes: as many waves as leave the fewest idle
// rows and columns in their rounds, within `most` and 160 KB of LDS
static bool conv_plane_shape(const ConvGeo& g, size_t item, int most, bool any, PlaneShape* s)
{
    const int Ny = g.r1[1] * g.r2[1];
    s->cls = std::max(rx_class(g.r1[1], g.r2[1]), rx_class(g.r1[2], g.r2[2]));
    double best = -1;
    for (int nw = 4; nw <= most / 64; nw += any ? 1 : 4)
    {
        const PlaneLds l =
            item == sizeof(z64)
                ? plane_lds<double>(g.r1[1], g.r2[1], g.r1[2], g.r2[2], g.nzk, 64 * nw)
                : plane_lds<float>(g.r1[1], g.r2[1], g.r1[2], g.r2[2], g.nzk, 64 * nw);
        if (l.bytes > 160 * 1024) break;
        // rounds of a wave over the rows and the columns, against the waves
        // that a CU holds (by registers 8 in FP64 and 12 in FP32, or what
        // the LDS allows)
        const double rounds = 2.0 * cdiv(Ny, nw * ln_rows(g.r2[2])) +
                              (double)cdiv(g.nzk, nw * ln_rows(g.r2[1]));
        const int blocks = (int)std::min<size_t>(160 * 1024 / l.bytes,
                                                 std::max(1, (item == sizeof(z64) ? 8 : 12) / nw));
        const double score = blocks / rounds;
        if (score > best * 1.001)
        {
            best = score;
            s->nt = 64 * nw;
            s->lds = l;
        }
    }
    return best > 0;
}

// false where the sphere form does not apply: an axis length without a
// compiled two-factor form or a plane that does not fit in LDS
static bool conv_geo(const lelph_ctx* c, ConvGeo* g)
{
    const lelph_lattice& L = c->lat;
    g->f32 = c->precision != LELPH_FP64;
    g->two = L.nspinor == 2 && L.nmag == 4;
    double rmax = 0;
    int64_t npw = 0;
    for (const DevWfc& w : c->wf)
    {
        rmax = std::max(rmax, w.rmax);
        npw = std::max(npw, w.npw);
    }
    if (!npw || npw > 0x3fffffff) return false;
    for (int i = 0; i < 3; ++i)
        if (!rx_factors(L.fft_dims[i], &g->r1[i], &g->r2[i])) return false;
    g->xcls = rx_class(g->r1[0], g->r2[0]);
    g->words = (int)cdiv(L.fft_dims[0], 32);
    // |G_i| spans at most 2 |a_i| max|k + G| in crystal units, whatever the
    // rotation and the umklapp vector
    int ext[3];
    for (int i = 0; i < 3; ++i)
    {
        const double* a = L.alat_vec;
        const double len = sqrt(a[i] * a[i] + a[3 + i] * a[3 + i] + a[6 + i] * a[6 + i]);
        ext[i] = (int)std::min<double>((double)L.fft_dims[i], floor(2 * rmax * len + 1e-6) + 1);
    }
    g->npw = (int)npw;
    g->ld = (int)(cdiv(npw, 16) * 16);
    g->nzk = ext[2];
    g->nst = (int)std::min<int64_t>((int64_t)ext[1] * ext[2], npw);
    g->nrows = (int64_t)L.nspin * L.nbnds * L.nspinor;
    if (g->nrows > 65535 || (int64_t)L.nmodes * g->nrows > 0x3fffffff) return false;
    const size_t item = g->f32 ? sizeof(c32) : sizeof(z64);
    const int cls = std::max(rx_class(g->r1[1], g->r2[1]), rx_class(g->r1[2], g->r2[2]));
    const int most = g->f32 ? (g->two ? plane_threads<float, true>(cls)
                                      : plane_threads<float, false>(cls))
                            : (g->two ? plane_threads<double, true>(cls)
                                      : plane_threads<double, false>(cls));
    if (!conv_plane_shape(*g, item, most, true, &g->conv)) return false;
    g->square = !g->two && rx_square(L.fft_dims[1], L.fft_dims[2]);
    if (g->square)
    {
        const int r1 = g->r1[1], r2 = g->r2[1];
        g->sqlds = g->f32 ? square_lds<float>(r1, r2, rx_square_waves<float>(r1 * r2), g->nzk)
                          : square_lds<double>(r1, r2, rx_square_waves<double>(r1 * r2), g->nzk);
        g->square = g->sqlds <= 160 * 1024;
    }
    if (!conv_plane_shape(*g, item, cls == 0 ? 512 : 256, false, &g->box)) return false;
    g->xlds = g->f32 ? x_lds<float>(g->r1[0], g->r2[0]) : x_lds<double>(g->r1[0], g->r2[0]);
    if (g->xlds > 160 * 1024) return false;
    // K splits of the sphere product: enough blocks for one pair alone, at
    // least 8 chunks each; from the shape only, so that a pair's sums do not
    // depend on what it is batched with
    const int64_t tiles = sph_gemm_tiles(L.nmodes, L.nbnds) * L.nspin;
    const int64_t chunks = cdiv(npw, SG_KC) * L.nspinor;
    g->nsplit = (int)std::max<int64_t>(1, std::min<int64_t>(cdiv(1024, tiles), chunks / 8));
    return true;
}

// pairs that go through the steps together, the modes and sets of a plane
// launch, and the modes of a block: transformed to the sphere, then contracted
struct ConvGroup
{
    int np, nv, ns, nm;
};

static ConvGroup conv_group(const lelph_ctx* c, const ConvGeo& g, int64_t npairs)
{
    const lelph_lattice& L = c->lat;
    const int64_t item = g.f32 ? sizeof(c32) : sizeof(z64);
    const int64_t one = item * L.fft_dims[0] * g.nst; // lines of one mode and set
    const int64_t gsz = (int64_t)L.nmodes * L.nspin * L.nbnds * L.nbnds;
    const int64_t pair = item * g.nrows * (c->nf + L.fft_dims[0] * (int64_t)g.nst +
                                           (int64_t)(L.nmodes + 2) * g.ld) +
                         (int64_t)sizeof(z64) * g.nsplit * gsz;
    const int64_t room = std::max<int64_t>(1, CONV_LINE_BYTES / one); // (mode, set) lines
    int64_t p = std::min<int64_t>(npairs, CONV_GROUP_PAIRS);
    p = std::min(p, std::max<int64_t>(1, room / (L.nmodes * g.nrows)));
    p = std::min(p, std::max<int64_t>(1, CONV_GROUP_BYTES / pair));
    p = std::min<int64_t>(p, 65535 / std::max(1, L.nspin) / 2);
    ConvGroup r;
    r.np = (int)std::max<int64_t>(1, p);
    int64_t nm = L.nmodes; // several pairs: all modes are within a group's bytes
    if (r.np == 1)
    {
        nm = std::max<int64_t>(1, CONV_C_BYTES / (item * g.nrows * g.ld));
        if (nm > CONV_MODES) nm -= nm % CONV_MODES;
        nm = std::min<int64_t>(nm, L.nmodes);
    }
    // one pair: up to 8 modes share a psi plane, the sets fill the rest
    int64_t nv = nm, ns = g.nrows;
    if (nv * ns * r.np > room)
    {
        nv = std::min<int64_t>(nm, CONV_MODES);
        nv = std::max<int64_t>(1, std::min(nv, room));
        ns = std::max<int64_t>(1, std::min<int64_t>(g.nrows, room / nv));
        if (ns == g.nrows) nv = std::max<int64_t>(1, std::min<int64_t>(nm, room / ns));
    }
    nv = std::max<int64_t>(1, std::min<int64_t>(nv, 500000 / ns)); // grid rows
    r.nv = (int)nv;
    r.ns = (int)ns;
    r.nm = (int)nm;
    return r;
}

// the FP32 potential with its rows in the plane kernels' order
static int conv_ensure_dv32(lelph_ctx* c, const ConvGeo& g)
{
    if (c->cv_dv32_valid) return LELPH_OK;
    const int64_t n = (int64_t)c->lat.nmodes * c->lat.nmag * c->nf;
    LELPH_TRY(c->cv_dv32.ensure(sizeof(c32) * n));
    hipLaunchKernelGGL(k_conv_dv32<float>, dim3((unsigned)cdiv(n, 256)), dim3(256), 0, c->stream,
                       c->dv64.as<z64>(), c->cv_dv32.as<c32>(), n, (int)c->lat.fft_dims[2],
                       g.r1[2], g.r2[2]);
    HIP_TRY(hipGetLastError());
    c->cv_dv32_valid = true;
    return LELPH_OK;
}

// bytes of a group's buffers and of their parts: np pairs, ns sides (a k+q
// one per pair, the distinct k ones)
struct ConvLayout
{
    size_t n_mask, o_ph, s_ph, s_idx, s_smap, s_zc, s_off, per; // maps of a side
    size_t s_coef, s_line, s_box;                               // of a side
    size_t s_cl, s_c;                                           // of a pair
    size_t map, coef, line, box, c, part;
    static size_t up(size_t n) { return (n + 255) & ~(size_t)255; }
    ConvLayout(const lelph_ctx* ctx, const ConvGeo& g, const ConvGroup& gr, int np, int ns)
    {
        const lelph_lattice& L = ctx->lat;
        const size_t Nx = (size_t)L.fft_dims[0], Ny = (size_t)L.fft_dims[1];
        const size_t Nz = (size_t)L.fft_dims[2], item = g.f32 ? sizeof(c32) : sizeof(z64);
        n_mask = up(4 * Ny * Nz * g.words);
        o_ph = up(n_mask * (size_t)ns);
        s_ph = up(sizeof(z64) * g.npw);
        s_idx = up(4 * (size_t)g.npw);
        s_smap = up(4 * (size_t)g.nzk * Ny);
        s_zc = up(2 * Nz);
        s_off = up(4 * (size_t)g.nst);
        per = s_ph + s_idx + s_smap + s_zc + s_off + up(4 * (size_t)g.nst * g.words) + 256;
        const size_t row = item * (size_t)g.nrows;
        s_coef = row * g.ld;
        s_line = row * Nx * g.nst;
        s_box = row * (size_t)ctx->nf;
        s_cl = item * (size_t)gr.ns * gr.nv * Nx * g.nst;
        s_c = s_coef * gr.nm;
        map = o_ph + per * ns;
        coef = s_coef * ns;
        line = std::max(s_line * (ns - np), s_cl * np);
        box = s_box * (ns - np);
        c = s_c * np;
        const size_t gsz = (size_t)gr.nm * L.nspin * L.nbnds * L.nbnds; // of a block
        part = g.nsplit > 1 ? sizeof(z64) * (size_t)g.nsplit * np * gsz : 0;
    }
    size_t bytes() const { return map + coef + line + box + c + part; }
    int ensure(ConvBufs& b, hipStream_t st) const
    {
        LELPH_TRY(buf_grow(b.map, map, b.fixed, st));
        LELPH_TRY(buf_grow(b.coef, coef, b.fixed, st));
        LELPH_TRY(buf_grow(b.line, line, b.fixed, st));
        LELPH_TRY(buf_grow(b.box, box, b.fixed, st));
        LELPH_TRY(buf_grow(b.c, c, b.fixed, st));
        return buf_grow(b.part, part, b.fixed, st);
    }
};

// Sizes b for every group of these pairs, for good: their descriptors, which
// hold its addresses, are run again by a captured pass.
static int conv_reserve(lelph_ctx* c, const ConvGeo& g, const ConvGroup& gr, ConvBufs& b,
                        const std::vector<lelph_pair>& pairs, hipStream_t st)
{
    for (size_t p0 = 0; p0 < pairs.size(); p0 += gr.np)
    {
        const size_t p1 = std::min(pairs.size(), p0 + gr.np);
        std::vector<std::array<int, 2>> k;
        for (size_t i = p0; i < p1; ++i) k.push_back({pairs[i].ik, pairs[i].ksym});
        std::sort(k.begin(), k.end());
        const int nk = (int)(std::unique(k.begin(), k.end()) - k.begin());
        const int np = (int)(p1 - p0);
        LELPH_TRY(ConvLayout(c, g, gr, np, np + nk).ensure(b, st));
    }
    b.fixed = true;
    return LELPH_OK;
}

// local part of `np` pairs into g (device, np * gsz contiguous) on stream
// st.  ev: [1] boxes built, [2] products done, or NULL.  desc: the group's
// descriptors, uploaded unless they are there already (a captured pass).
template <typename T>
static int conv_local(lelph_ctx* c, const ConvGeo& geo, ConvBufs& b, DBuf& desc, bool upload,
                      const double* qpt, const lelph_pair* pairs, int np, const ConvGroup& gr,
                      z64* g, hipStream_t st, hipEvent_t* ev)
{
    const lelph_lattice& L = c->lat;
    const int nv = gr.nv, nset = gr.ns;
    const int Nx = (int)L.fft_dims[0], Ny = (int)L.fft_dims[1], Nz = (int)L.fft_dims[2];
    const int nmag_eff = (L.nspinor == 1 && L.nmag == 4) ? 1 : L.nmag;
    // sides: every pair's k+q sphere, then the distinct k ones
    std::vector<SphSide> sides((size_t)np);
    std::vector<ConvPair> cp((size_t)np);
    std::vector<int> kside((size_t)np);
    std::vector<std::pair<int64_t, int>> keys;
    for (int i = 0; i < np; ++i)
    {
        const lelph_pair& p = pairs[i];
        if (p.ik < 0 || p.ikq < 0 || p.ik >= (int)c->wf.size() || p.ikq >= (int)c->wf.size())
            return LELPH_ERR_ARG;
        if (p.ksym < 0 || p.kqsym < 0 || p.ksym >= L.nsym || p.kqsym >= L.nsym)
            return LELPH_ERR_ARG;
        if (!c->wf[p.ik].wfc || !c->wf[p.ikq].wfc) return LELPH_ERR_STATE;
        SideGeom gk;
        LELPH_TRY(local_geometry(c, qpt, p.ikq, p.ik, p.kqsym, p.ksym, &sides[i].geo, &gk));
        sides[i].wfc = c->wf[p.ikq].wfc;
        sides[i].gvec = c->wf[p.ikq].gvec;
        sides[i].npw = (int)c->wf[p.ikq].npw;
        const int64_t key = (int64_t)p.ik * L.nsym + p.ksym;
        int at = -1;
        for (const auto& k : keys)
            if (k.first == key) at = k.second;
        if (at < 0)
        {
            at = (int)sides.size();
            keys.push_back({key, at});
            SphSide s{};
            s.geo = gk;
            s.wfc = c->wf[p.ik].wfc;
            s.gvec = c->wf[p.ik].gvec;
            s.npw = (int)c->wf[p.ik].npw;
            sides.push_back(s);
        }
        kside[i] = at;
    }
    const int ns = (int)sides.size(), nk = ns - np;
    const ConvLayout lay(c, geo, gr, np, ns);
    LELPH_TRY(lay.ensure(b, st));
    char* mp = b.map.as<char>();
    for (int i = 0; i < ns; ++i)
    {
        SphSide& s = sides[i];
        s.ld = (int)(cdiv(s.npw, 16) * 16);
        s.mask = reinterpret_cast<unsigned*>(mp + lay.n_mask * i);
        char* m = mp + lay.o_ph + lay.per * i;
        s.cnt = reinterpret_cast<int*>(m + lay.per - 256);
        s.ph = reinterpret_cast<z64*>(m);
        s.idx = reinterpret_cast<int*>(m += lay.s_ph);
        s.smap = reinterpret_cast<int*>(m += lay.s_idx);
        s.zc = reinterpret_cast<short*>(m += lay.s_smap);
        s.off = reinterpret_cast<int*>(m += lay.s_zc);
        s.smask = reinterpret_cast<unsigned*>(m += lay.s_off);
        s.coef = b.coef.as<char>() + lay.s_coef * i;
        s.line = i < np ? nullptr : b.line.as<char>() + lay.s_line * (i - np);
        s.box = i < np ? nullptr : b.box.as<char>() + lay.s_box * (i - np);
    }
    for (int i = 0; i < np; ++i)
    {
        cp[i].box = sides[kside[i]].box;
        cp[i].dv = geo.f32 ? c->cv_dv32.p : c->dv64.p;
        cp[i].side = i;
        cp[i].line = b.line.as<char>() + lay.s_cl * i;
        cp[i].c = b.c.as<char>() + lay.s_c * i;
    }
    const size_t n_s = ConvLayout::up(sizeof(SphSide) * ns);
    std::vector<char> hd(n_s + sizeof(ConvPair) * np);
    std::memcpy(hd.data(), sides.data(), sizeof(SphSide) * ns);
    std::memcpy(hd.data() + n_s, cp.data(), sizeof(ConvPair) * np);
    if (upload)
    {
        LELPH_TRY(desc.ensure(hd.size()));
        HIP_TRY(hipMemcpyAsync(desc.p, hd.data(), hd.size(), hipMemcpyHostToDevice, st));
    }
    const SphSide* ds = desc.as<SphSide>();
    const ConvPair* dp = reinterpret_cast<const ConvPair*>(desc.as<char>() + n_s);
    const z64 *Wx = axis_tw<double>(c->ax[0]), *Wy = axis_tw<double>(c->ax[1]),
              *Wz = axis_tw<double>(c->ax[2]);

    LELPH_TRY(zero_async(mp, lay.n_mask * ns, st));
    LELPH_TRY(conv_maps_launch(ns, geo.npw, st, ds, Nx, Ny, Nz, geo.words, geo.nzk, geo.nst,
                               c->d_err));
    const int64_t nsets = (int64_t)L.nspin * L.nbnds;
    const int gper = 16;
    LELPH_TRY(conv_gather_launch<T>(dim3((unsigned)cdiv(geo.ld, 256),
                                         (unsigned)cdiv(nsets, gper), (unsigned)ns),
                                    st, ds, nsets, L.nspinor, Ny, Nz, geo.words, gper));
    // psi_k boxes
    const unsigned tiles = (unsigned)cdiv(geo.nst, x_tile<T>());
    BoxArgs ba{Nx, Ny, Nz, geo.words, geo.nrows, geo.nzk, geo.nst, 1};
    ba.rows_per_block =
        (int)std::max<int64_t>(1, std::min<int64_t>(8, geo.nrows * tiles * nk / 2048));
    LELPH_TRY(conv_box_x_launch<T>(
        geo.xcls, geo.xlds,
        dim3(tiles, (unsigned)cdiv(geo.nrows, ba.rows_per_block), (unsigned)nk), st, ds + np, ba,
        Wx));
    const int64_t nx8 = 8 * cdiv(Nx, 8);
    PlaneArgs pb{geo.box.lds.rows, geo.box.lds.prow, geo.box.lds.tw,
                 geo.r1[1], geo.r2[1], geo.r2[2]};
    LELPH_TRY(conv_box_plane_launch<T>(geo.box, nx8 * geo.nrows * nk, st, ds + np, ba, pb, Wy,
                                       Wz));
    c->box_sides += nk;
    if (ev) HIP_TRY(hipEventRecord(ev[1], st));
    // dV psi to the sphere, a chunk of modes at a time
    PlaneArgs pc{geo.conv.lds.rows, geo.conv.lds.prow, geo.conv.lds.tw,
                 geo.r1[1], geo.r2[1], geo.r2[2]};
    const int64_t es = (int64_t)L.nspin * L.nbnds * L.nbnds;
    for (int m0 = 0; m0 < L.nmodes; m0 += gr.nm)
    {
        const int nm = std::min(gr.nm, L.nmodes - m0);
        const int64_t nvs = cdiv(nm, nv);
        for (int64_t vs = 0; vs < nvs * cdiv(geo.nrows, nset); ++vs)
        {
            // sets outside, modes inside: the psi boxes of the sets stay cached
            ConvArgs a{};
            a.Nx = Nx;
            a.Ny = Ny;
            a.Nz = Nz;
            a.words = geo.words;
            a.vc = m0;
            a.v0 = m0 + (int)(vs % nvs) * nv;
            a.nv = std::min(nv, m0 + nm - a.v0);
            a.s0 = (int)(vs / nvs) * nset;
            a.ns = (int)std::min<int64_t>(nset, geo.nrows - a.s0);
            a.nspin = L.nspin;
            a.nb = L.nbnds;
            a.nspinor = L.nspinor;
            a.nmag = nmag_eff;
            a.nzk_max = geo.nzk;
            a.nst_max = geo.nst;
            const int64_t planes = (int64_t)a.ns * Nx * a.nv * np;
            a.sper = (int)std::max<int64_t>(1, std::min<int64_t>(CONV_SETS, planes / 1024));
            const int64_t blocks = nx8 * a.nv * cdiv(a.ns, a.sper) * np;
            if (geo.square)
                LELPH_TRY(conv_square_launch<T>(geo.sqlds, blocks, st, dp, ds, a, Wz));
            else
                LELPH_TRY(
                    conv_plane_launch<T>(geo.two, geo.conv, blocks, st, dp, ds, a, pc, Wy, Wz));
            const int64_t rows = (int64_t)a.ns * a.nv;
            a.rows_per_block =
                (int)std::max<int64_t>(1, std::min<int64_t>(8, rows * tiles * np / 4096));
            LELPH_TRY(conv_x_launch<T>(geo.xcls, geo.xlds,
                                       dim3(tiles, (unsigned)cdiv(rows, a.rows_per_block),
                                            (unsigned)np),
                                       st, dp, ds, a, Wx));
        }
        z64* gm = g + m0 * es; // fewer than all modes: of a single pair
        LELPH_TRY(sph_gemm_launch<T>(geo.nsplit, np, st, dp, ds, nm, L.nspin, L.nbnds,
                                     L.nspinor, 1.0 / (double)c->nf,
                                     geo.nsplit > 1 ? b.part.as<z64>() : gm));
        if (ev && m0 + nm == L.nmodes) HIP_TRY(hipEventRecord(ev[2], st));
        if (geo.nsplit > 1)
            LELPH_TRY(reduce_parts(b.part.as<z64>(), geo.nsplit, nm * es * np,
                                   1.0 / (double)c->nf, gm, st));
    }
    return LELPH_OK;
}

// internal status: a sphere that this form does not take (two plane waves
// on one box point); the caller goes on in the box form
#define LELPH_CONV_REDO 1001

// Sticks per (Gy, Gz) of the plane up to which conv_use's constants hold: a
// sphere of half a grid's length across takes (1/2 + 1/N)^2 of them.
static const double CONV_ORDINARY = 0.34;

// The same question for spheres that fill more of the box than that.  The
// sphere form keeps more columns, sticks and plane waves there: at 60^3, 64
// bands, 18 modes, FP32, a sphere of 0.47, 0.60, 0.76, 0.93 of an axis takes
// 3.7, 5.2, 7.7, 11.7 ps against the box form's 7.0.  Both forms in ps per
// pair, fitted to 1900 timings (12^3 to 80^3, slabs, 4 to 128 bands, spheres
// of 0.47 to 0.93, one to four pairs, all spins; rms 6 to 15 %): launches,
// psi boxes per row and point, the rest per mode, row and point.  With
// conv_use's constants alone 160 of them took the sphere form at up to 2.3
// times the box form's time; 25 do with this, at up to 1.25.
static bool conv_dense(const lelph_ctx* c, const ConvGeo& g, int prec, double box, double fs)
{
    const lelph_lattice& L = c->lat;
    const double rows = (double)c->nf * L.nspin * L.nspinor * L.nbnds, work = rows * L.nmodes;
    const double fp = (double)g.npw / (double)c->nf;
    double tb;
    if (prec == LELPH_FP64)
        tb = g.two ? 14 * rows + (box + 3.2) * work : 28 * rows + (box + 1.8) * work;
    else if (prec == LELPH_FP32)
        tb = 21 * rows + (g.two ? 1.95 : 1.0) * box * work;
    else if (prec == LELPH_BF16X6)
        tb = g.two ? 21 * rows + (1.7 * box + 0.7) * work : 28 * rows + box * work;
    else
        tb = 28 * rows + 0.8 * box * work;
    double ts; // without the sticks' and the product's share
    if (g.f32)
        ts = g.two ? 14 * rows + 2.7 * work : (g.square ? 23 : 26) * rows;
    else
        ts = g.two ? 54 * rows + 4.5 * work
                   : g.square ? 28 * rows + 1.2 * work : 45 * rows;
    const double stick = g.f32 ? (g.two ? 8.3 : g.square ? 7.2 : 9.7)
                               : (g.two ? 14.8 : g.square ? 12.2 : 17.7);
    return 40e6 + ts + (stick * fs + 0.18 * fp * L.nbnds) * work < 95e6 + tb;
}

// Whether the local part runs in the sphere form.  Per set, mode and grid
// point the box form costs 8 nb operations, the sphere form a transform
// whatever nb is; in picoseconds, all steps of the local part:
//   box, FP32    0.093 per band, bands padded to 16; FP64 0.19, with the
//                padding of its tile; bf16x6 5.4 per tile of 128 x 64; bf16x3
//                on the producer/consumer kernel 2.65 at 128 bands
//   sphere       square planes 3.3 + 0.011 nb (FP32), 5.6 (FP64), others
//                4.5 + 0.011 nb and 6.0; a 2x2 spinor potential 5.2 and 14
//                (box form 2.2 x)
// Fitted to the first kernels of the sphere form.  Measured since, 96^3, 128
// bands, 48 modes, per pair: FP64 29.4 ms (5.4 ps) against 133.5 (24.6) in the
// box form, FP32 19.9 (3.7) against 58.9 (10.8), bf16x6 31.7 (5.8), bf16x3
// 16.1 (3.0).  So the rule stays with the box form a little longer than it
// needs to: in 26 of 322 timings of spheres of half an axis (FP32 at 16 and 32
// bands on 36^3 to 80^3, FP64 at 16) the sphere form would take 0.5 to 0.97 of
// the time; it takes none where the box form is more than 2 % faster.
// Below 2e7 points x rows, where the box form's time is launches, the sphere
// form wins by taking all pairs of a group together.
static bool conv_use(const lelph_ctx* c, ConvGeo* g)
{
    if (c->local_form == LELPH_FORM_BOX || c->conv_off || !conv_geo(c, g)) return false;
    // one pair's buffers in half of the memory: three boxes' worth where the
    // sphere fills the box, the box form takes two
    if (ConvLayout(c, *g, conv_group(c, *g, 1), 1, 2).bytes() > c->mem_total / 2) return false;
    if (c->local_form == LELPH_FORM_SPHERE) return true;
    const lelph_lattice& L = c->lat;
    const int prec = effective_precision(c), nb = L.nbnds;
    const double work = (double)c->nf * L.nmodes * L.nspin * L.nspinor * nb; // points x rows
    double box, sphere;
    if (prec == LELPH_FP64)
    {
        const int* s = CT_SHAPES[ct_auto(L.nmodes, nb, false) - 1];
        box = 0.19 * (double)(cdiv(L.nmodes, s[0]) * s[0]) / L.nmodes *
              (double)(cdiv(nb, s[1]) * s[1]) / nb * (double)(cdiv(nb, s[2]) * s[2]);
        sphere = g->two ? 14.0 : g->square ? 5.6 : 6.0;
    }
    else
    {
        sphere = (g->two ? 5.2 : g->square ? 3.3 : 4.5) + 0.011 * nb;
        if (prec == LELPH_FP32)
            box = 0.093 * (double)(cdiv(nb, 16) * 16) * (double)(cdiv(nb, 16) * 16) / nb;
        else if (prec == LELPH_BF16X6)
            box = 5.4 * (double)(cdiv(nb, 128) * 128) * (double)(cdiv(nb, 64) * 64) /
                  (128.0 * nb);
        else
            box = 2.65 * (double)(cdiv(nb, 16) * 16) * (double)(cdiv(nb, 128) * 128) /
                  (128.0 * nb);
    }
    // below 2e7 the box product of a pair takes less than some 100 us; all
    // pairs of a group in one launch each then save more than it costs (64
    // pairs of 24^3, 8 bands: 6.6 -> 0.6 ms; a single pair, 16 bands: 0.157
    // against 0.168 ms of local part)
    if (work >= 2e7 && sphere >= box * (g->two && prec != LELPH_BF16X6 ? 2.2 : 1)) return false;
    const double fs = (double)g->nst / (double)(L.fft_dims[1] * L.fft_dims[2]);
    return fs <= CONV_ORDINARY || conv_dense(c, *g, prec, box, fs);
}

// the potential in the precision that the sphere form reads
static int conv_prepare(lelph_ctx* c, const ConvGeo& geo)
{
    if (!c->dv_set) return LELPH_ERR_STATE;
    if (c->lat.nmag == 2 && (c->lat.nspin != 2 || c->lat.nspinor != 1)) return LELPH_ERR_ARG;
    return geo.f32 ? conv_ensure_dv32(c, geo) : LELPH_OK;
}

static int conv_group_local(lelph_ctx* c, const ConvGeo& geo, const ConvGroup& gr, ConvBufs& b,
                            DBuf& desc, bool upload, const double* qpt, const lelph_pair* pairs,
                            int np, z64* g, hipStream_t st, hipEvent_t* ev)
{
    return geo.f32
               ? conv_local<float>(c, geo, b, desc, upload, qpt, pairs, np, gr, g, st, ev)
               : conv_local<double>(c, geo, b, desc, upload, qpt, pairs, np, gr, g, st, ev);
}
