"""Spheres that the sphere form of the local part does not take: two plane
waves G and G - N b_1 on one box point, with the same coefficients (the box
form stores one over the other).  Every entry point finds that out on the
device and repeats the work in the box form: g bit-identical to a context
pinned to it, and nothing of it reaches calls that have no local part."""
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
