"""Multi-cell batches of more pairs than one group or window takes (256): the
later ones need larger buffers than the first, whose descriptors the replayed
graph reads again.  The first 256 pairs are one pair repeated (two sides, one
psi_k box), the others touch every k.  A cell in the sphere form per precision
and one in the box form (an axis of 13 points); every replay bit-identical to
lelph_gkq_batch, with work of the contexts in between."""
import numpy as np
import pytest

from letzelphc_amd import lelph, synth

from .util import say

pytestmark = pytest.mark.gpu

WINDOW = 256
CELLS = [
    ("sphere_fp64", dict(nbnds=2), "fp64"),
    ("sphere_fp32_spin2", dict(nbnds=3, nspin=2, nmag=2), "fp32"),
    ("box_fp64", dict(nbnds=2, fft=(13, 12, 12)), "fp64"),
]


def sides(pairs):
    return {(p[0], p[2]) for p in pairs} | {(p[1], p[3]) for p in pairs}


def test_later_groups_are_larger():
    jobs = []
    try:
        for name, kw, prec in CELLS:
            s = synth.tiny(kgrid=(4, 4, 2), syms="id", **kw)
            ctx = lelph.Context(s, prec)
            ctx.set_dvscf(s.qpts[0], s.eigvec(0), s.dvscf(0), kernel="dfpt")
            every = synth.kq_pairs(s, 0)
            pairs = [every[0]] * WINDOW + every
            assert len(sides(pairs[WINDOW:])) > len(sides(pairs[:WINDOW]))
            jobs.append((ctx, s.qpts[0], pairs))
        say("case: multi-cell batch, later groups larger: "
            + ", ".join(f"{c[0]} ({len(j[2])} pairs)" for c, j in zip(CELLS, jobs)))
        m = lelph.MultiBatch(jobs)
        try:
            refs = [ctx.gkq_batch(p, qpt=q) for ctx, q, p in jobs]
            for rep in range(3):
                for (name, *_), g, r in zip(CELLS, m.run(), refs):
                    assert np.array_equal(g, r), (rep, name)
                ctx, q, pairs = jobs[rep]
                ctx.gkq(*pairs[-1], qpt=q)
        finally:
            m.close()
    finally:
        for ctx, _, _ in jobs:
            ctx.close()
