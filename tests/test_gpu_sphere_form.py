"""The sphere form of the local part (transforms of dV psi to the k+q sphere,
csrc/conv.hpp) against the FP64 oracle at the sizes where its layouts can go
wrong: odd and unequal axes, lines of every factor class (products of 2, 3, 5
and 7; both factors small, one of 15 to 18), planes with a kernel of their own
and planes without, row counts that leave a wave's last rows idle, spheres
that fill most of the box, rotated and time-reversed sides with an umklapp
vector, both spins, spinors with and without the 2x2 potential.  Lengths
without a two-factor form (11, 13, 22) run in the box form and must agree
just as well.

Bars: the FP64 form differs from the oracle by rounding of the same sums
(1e-10, as everywhere); FP32 transforms of N points carry some
log2(N) * 6e-8 per coefficient, averaged over the sphere (1e-6)."""
import ctypes

import numpy as np
import pytest

from letzelphc_amd import lelph, synth
from oracle import oracle as O

from .util import rel_err, say

pytestmark = pytest.mark.gpu

GRIDS = [
    (12, 12, 12), (15, 16, 18), (16, 15, 15), (14, 21, 20), (25, 12, 27), (28, 18, 24),
    (12, 30, 30), (32, 14, 35), (12, 42, 16), (18, 45, 45), (12, 12, 54), (12, 56, 56),
    (63, 12, 12), (12, 14, 70), (12, 75, 12), (12, 81, 14), (12, 96, 96), (12, 14, 108),
    (12, 126, 12), (12, 12, 135), (144, 12, 14), (12, 160, 12), (12, 14, 216), (225, 12, 12),
    (12, 12, 240), (13, 12, 12), (12, 22, 12), (12, 12, 26),
]


@pytest.mark.parametrize("fft", GRIDS)
def test_grids(fft):
    # the cubic cell stretched so that every axis holds the sphere
    s = synth.tiny(nbnds=5, fft=fft, kgrid=(2, 2, 2), syms="cubic" if fft[0] == fft[1] else "id",
                   ecut=5.0)
    o = O.OracleSystem(s)
    dv = o.dv_total(0)
    pairs = synth.kq_pairs(s, 0)
    pick = [pairs[i] for i in (0, 3, len(pairs) - 1)]
    ref = np.stack([o.add_nonlocal(0, *p, o.elph_local(0, *p, dv)) for p in pick])
    errs = {}
    ctx = lelph.Context(s, "fp64")
    try:
        ctx.set_dvscf(s.qpts[0], s.eigvec(0), s.dvscf(0), kernel="dfpt")
        for prec in ("fp64", "fp32"):
            ctx.set_precision(prec)
            assert ctx.local_form() == ("box" if {13, 22, 26} & set(fft) else "sphere")
            errs[prec] = rel_err(ctx.gkq_batch(pick, qpt=s.qpts[0]), ref)
    finally:
        ctx.close()
    say(f"case: sphere form {fft}: {errs}")
    assert errs["fp64"] < 1e-10 and errs["fp32"] < 1e-6


# square planes that GRIDS leaves out
SQUARES = [18, 20, 24, 25, 27, 28, 32, 36, 40, 42, 48, 50, 54, 60, 64, 70, 72, 75, 80, 81, 84, 90,
           100, 108, 120]


@pytest.mark.parametrize("n", SQUARES)
def test_square_planes(n):
    s = synth.tiny(nbnds=4, fft=(12, n, n), kgrid=(2, 2, 1), syms="trev", ecut=6.0,
                   q=(0.5, 0.0, 0.0))
    o = O.OracleSystem(s)
    dv = o.dv_total(0)
    pairs = synth.kq_pairs(s, 0)
    pick = [pairs[0], pairs[-1]]
    ref = np.stack([o.elph_local(0, *p, dv) for p in pick])
    errs = {}
    ctx = lelph.Context(s, "fp64")
    try:
        ctx.set_local_form("sphere")
        ctx.set_dvscf(s.qpts[0], s.eigvec(0), s.dvscf(0), kernel="dfpt")
        for prec in ("fp64", "fp32"):
            ctx.set_precision(prec)
            assert ctx.local_form() == "sphere"
            errs[prec] = rel_err(ctx.gkq_batch(pick, non_loc=False, qpt=s.qpts[0]), ref)
    finally:
        ctx.close()
    say(f"case: square planes {n}: {errs}")
    assert errs["fp64"] < 1e-10 and errs["fp32"] < 1e-6


SPIN = {
    "spin2": dict(nspin=2, nmag=2),
    "spinor_nmag1": dict(nspinor=2, nmag=1),
    "spinor_nmag4": dict(nspinor=2, nmag=4),
}


@pytest.mark.parametrize("case", list(SPIN))
@pytest.mark.parametrize("nb", [1, 17, 33, 49])
@pytest.mark.parametrize("fft", [(16, 16, 16), (16, 15, 18)])
def test_bands_and_spin(case, nb, fft):
    """column tiles of the sphere product (16, 32, 48, 64) and their
    remainders, with the spin layouts"""
    s = synth.tiny(nbnds=nb, fft=fft, ecut=14.0, kgrid=(2, 2, 1), syms="id", q=(0.5, 0.0, 0.0),
                   **SPIN[case])
    o = O.OracleSystem(s)
    dv = o.dv_total(0)
    pairs = synth.kq_pairs(s, 0)
    ref = np.stack([o.elph_local(0, *p, dv) for p in pairs[:2]])
    errs = {}
    ctx = lelph.Context(s, "fp64")
    try:
        ctx.set_dvscf(s.qpts[0], s.eigvec(0), s.dvscf(0), kernel="dfpt")
        for prec in ("fp64", "fp32"):
            ctx.set_precision(prec)
            assert ctx.local_form() == "sphere"
            one = np.stack([ctx.elph_local(*p) for p in pairs[:2]])
            bat = ctx.gkq_batch(pairs, non_loc=False, qpt=s.qpts[0])[:2]
            # a pair's sums do not depend on what it is batched with
            assert np.array_equal(one, bat)
            errs[prec] = rel_err(one, ref)
    finally:
        ctx.close()
    say(f"case: sphere form {case} nb {nb} {fft}: {errs}")
    assert errs["fp64"] < 1e-10 and errs["fp32"] < 1e-6


def test_blocks_of_modes():
    """A pair whose coefficients on the sphere, 24 modes x 256 bands x 46,000
    plane waves, exceed the 4 GB kept of them: transformed and contracted in
    two blocks of modes (16 and 8: 2.9 GB beside the boxes, lines and maps, not
    4.3).  Against the box form, another sum of the same terms (1e-12; the
    oracle takes minutes), alone and in a batch of two."""
    free_total = (ctypes.c_size_t * 2)()

    def free():
        # the HIP runtime that the library is linked to
        assert lelph.lib().hipMemGetInfo(free_total, ctypes.byref(free_total, 8)) == 0
        return free_total[0] / 2 ** 30

    s = synth.make_system("blocks", 11, 16.0 * np.eye(3),
                          [[x, y, z] for x in (0, 0.5) for y in (0, 0.5) for z in (0, 0.5)],
                          [0] * 8, [3.0], (48, 48, 48), (2, 1, 1), 77.0, 256,
                          [(np.eye(3), np.zeros(3), 0)], 0, [(0.5, 0.0, 0.0)])
    assert 16 * s.nmodes * s.nbnds * min(w.npw for w in s.wfcs) > 4 << 30
    pairs = synth.kq_pairs(s, 0)
    g = {}
    ctx = lelph.Context(s, "fp64")
    try:
        ctx.set_dvscf(s.qpts[0], s.eigvec(0), s.dvscf(0), kernel="dfpt")
        for form in ("box", "sphere"):
            ctx.set_local_form(form)
            before = free()
            g[form] = np.stack([ctx.elph_local(*p) for p in pairs])
            used = before - free()
        say(f"case: sphere form in blocks of modes: {used:.2f} GB of buffers")
        assert used < 5.2
        assert np.array_equal(ctx.gkq_batch(pairs, non_loc=False, qpt=s.qpts[0]), g["sphere"])
    finally:
        ctx.close()
    err = rel_err(g["sphere"], g["box"])
    say(f"  npw {[w.npw for w in s.wfcs]}, against the box form {err:.2e}")
    assert err < 1e-12


# (points per axis, bands): where spheres that fill the box make the sphere
# form the slower one (a sphere of 0.92 of an axis; 1.3 to 1.9 times the box
# form's time when it was taken there all the same)
DENSE = [((48, 48, 48), 32, "fp64"), ((48, 48, 48), 64, "fp32"), ((45, 45, 108), 32, "fp64"),
         ((48, 60, 72), 8, "fp64"), ((48, 60, 72), 64, "bf16x6")]


@pytest.mark.parametrize("fft,nb,prec", DENSE)
def test_spheres_that_fill_the_box(fft, nb, prec):
    """the box form by itself for a dense sphere, the sphere form for one of
    half an axis, and both forms of the dense one agree"""
    used, g = {}, {}
    for frac in (0.235, 0.46):
        gmax = frac * 3.0 * 2 * np.pi  # points per bohr: 3
        s = synth.make_system("dense", 5, np.diag(np.array(fft) / 3.0),
                              [[0, 0, 0], [0.5, 0.5, 0.5], [0.5, 0.0, 0.5], [0.0, 0.5, 0.5]],
                              [0] * 4, [3.0], fft, (2, 1, 1), gmax ** 2, nb,
                              [(np.eye(3), np.zeros(3), 0)], 0, [(0.5, 0.0, 0.0)])
        ctx = lelph.Context(s, prec)
        try:
            used[frac] = ctx.local_form()
            if frac > 0.4:
                ctx.set_dvscf(s.qpts[0], s.eigvec(0), s.dvscf(0), kernel="dfpt")
                pair = synth.kq_pairs(s, 0)[0]
                for form in ("auto", "sphere"):
                    ctx.set_local_form(form)
                    g[form] = ctx.elph_local(*pair)
        finally:
            ctx.close()
    err = rel_err(g["sphere"], g["auto"])
    say(f"case: dense sphere {fft} nb {nb} {prec}: {used}, the forms {err:.2e} apart")
    assert used == {0.235: "sphere", 0.46: "box"}
    assert err < (1e-12 if prec == "fp64" else 1e-6)
