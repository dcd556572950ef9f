"""Spheres that the sphere form of the local part does not take: two plane
waves G and G - N b_1 on one box point, with the same coefficients (the box
form stores one over the other).  Every entry point finds that out on the
device and repeats the work in the box form: g bit-identical to a context
pinned to it.  New wavefunctions bring the sphere form back, and nothing of it
reaches calls that have no local part."""
import copy

import numpy as np
import pytest

from letzelphc_amd import lelph, synth

from .util import say

pytestmark = pytest.mark.gpu

IK = 3


def aliased(s, ik=IK, with_fk=True):
    """s with the first plane wave of positive G_1 of wavefunction ik twice"""
    s = copy.copy(s)
    s.wfcs = list(s.wfcs)
    w = copy.copy(s.wfcs[ik])
    i = int(np.flatnonzero(w.gint[:, 0] > 0)[0])
    n = np.array([s.fft_dims[0], 0, 0])
    w.gint = np.vstack([w.gint, w.gint[i] - n])
    w.gvec = np.vstack([w.gvec, w.gvec[i] - n[0] * s.blat[:, 0] / (2 * synth.RPI)])
    w.wfc = np.ascontiguousarray(np.concatenate([w.wfc, w.wfc[..., i:i + 1]], axis=-1))
    w.Fk = np.ascontiguousarray(np.concatenate([w.Fk, w.Fk[..., i:i + 1]], axis=-1))
    if not with_fk:
        w.Fk = None
    s.wfcs[ik] = w
    return s


def context(s, prec, form="auto"):
    ctx = lelph.Context(s, prec)
    ctx.set_dvscf(s.qpts[0], s.eigvec(0), s.dvscf(0), kernel="dfpt")
    ctx.set_local_form(form)
    return ctx


KINDS = {
    "plain": dict(nbnds=3),
    "spin2": dict(nbnds=2, nspin=2, nmag=2),
    "spinor_nmag4": dict(nbnds=2, nspinor=2, nmag=4),
}


@pytest.mark.parametrize("kind", list(KINDS))
@pytest.mark.parametrize("prec", ["fp64", "fp32"])
def test_repeated_in_the_box_form(kind, prec):
    clean = synth.tiny(syms="id", **KINDS[kind])
    s = aliased(clean)
    pairs = synth.kq_pairs(s, 0)
    touched = next(p for p in pairs if IK in p[:2])
    say(f"case: aliased sphere {kind} {prec}")
    box = context(s, prec, "box")
    ref = box.gkq_batch(pairs, qpt=s.qpts[0])
    one = {p: box.gkq(*p, qpt=s.qpts[0]) for p in pairs}
    box.close()
    good = context(clean, prec)
    want = good.gkq_batch(pairs, qpt=s.qpts[0])
    for call in ("gkq", "batch", "compute", "multi"):
        ctx = context(s, prec)
        try:
            assert ctx.local_form() == "sphere"
            if call == "gkq":
                free = next(p for p in pairs if IK not in p[:2])
                ctx.gkq(*free, qpt=s.qpts[0])
                assert ctx.local_form() == "sphere"
                assert np.array_equal(ctx.gkq(*touched, qpt=s.qpts[0]), one[touched])
            elif call == "batch":
                assert np.array_equal(ctx.gkq_batch(pairs, qpt=s.qpts[0]), ref)
            elif call == "compute":
                assert np.array_equal(ctx.compute_elphq(s.qpts[0]), ref)
            else:
                m = lelph.MultiBatch([(good, s.qpts[0], pairs), (ctx, s.qpts[0], pairs)])
                try:
                    for _ in range(3):
                        a, b = m.run()
                        assert np.array_equal(a, want) and np.array_equal(b, ref)
                        good.gkq(*touched, qpt=s.qpts[0])
                finally:
                    m.close()
            assert ctx.local_form() == "box" and good.local_form() == "sphere"
            w = clean.wfcs[IK]
            ctx.upload_wfc(IK, w.wfc, w.gvec, w.Fk)
            assert ctx.local_form() == "sphere"
            # the K splits of the product follow the largest sphere, now the
            # clean system's again
            assert np.array_equal(ctx.gkq_batch(pairs, qpt=s.qpts[0]), want)
        finally:
            ctx.close()
    good.close()


@pytest.mark.parametrize("call", ["gkq", "batch"])
def test_failed_call_leaves_nothing_behind(call):
    """no projector tables: the local part meets the sphere, then the call
    fails; the next one is told nothing of it"""
    s = aliased(synth.tiny(nbnds=3, syms="id"), with_fk=False)
    pairs = synth.kq_pairs(s, 0)
    touched = next(p for p in pairs if IK in p[:2])
    say(f"case: aliased sphere, call without projector tables, {call}")
    ctx = context(s, "fp64")
    try:
        with pytest.raises(lelph.LelphError) as e:
            if call == "gkq":
                ctx.gkq(*touched, qpt=s.qpts[0])
            else:
                ctx.gkq_batch(pairs, qpt=s.qpts[0])
        assert e.value.status == 6
        ctx.set_dvscf(s.qpts[0], s.eigvec(0), s.dvscf(0), kernel="dfpt")
        box = context(s, "fp64", "box")
        assert np.array_equal(ctx.elph_local(*touched), box.elph_local(*touched))
        box.close()
    finally:
        ctx.close()
