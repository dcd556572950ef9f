"""Work that is formed for many pairs or points at once: the non-local sides
of a batch (csrc/nlbatch.hpp), the split-K sums, the D matrices and the staged
copy of large results, at the sizes where they can go wrong: one band, tiles
with a remainder, more than one tile, sides shared by several pairs, a result
above the staging threshold whose last chunk is partial.

Bars: batch and single pair are the same operations in the same order, the
staged copy moves bytes (both bit-identical); against the FP64 oracle 1e-10,
and 1e-6 for FP32 operands (sums of npw products of 6e-8 each)."""
import ctypes

import numpy as np
import pytest

from letzelphc_amd import abi, lelph, synth
from oracle import oracle as O

from .util import rel_err, say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nb", [1, 17, 70])
@pytest.mark.parametrize("syms", ["id", "cubic"])
def test_nonlocal_sides(nb, syms):
    s = synth.tiny(nbnds=nb, fft=(20, 20, 20), kgrid=(2, 2, 2), syms=syms, ecut=22.0)
    o = O.OracleSystem(s)
    pairs = synth.kq_pairs(s, 0)
    pick = [0, len(pairs) // 2, len(pairs) - 1]
    dv = o.dv_total(0)
    ref = np.stack([o.add_nonlocal(0, *pairs[i], o.elph_local(0, *pairs[i], dv)) for i in pick])
    errs = {}
    ctx = lelph.Context(s, "fp64")
    try:
        ctx.set_dvscf(s.qpts[0], s.eigvec(0), s.dvscf(0), kernel="dfpt")
        for prec in ("fp64", "fp32"):
            ctx.set_precision(prec)
            full = ctx.gkq_batch(pairs, qpt=s.qpts[0])
            for i in pick:
                assert np.array_equal(full[i], ctx.gkq(*pairs[i], qpt=s.qpts[0])), (prec, i)
            errs[prec] = rel_err(full[pick], ref)
    finally:
        ctx.close()
    say(f"case: non-local sides nb {nb} {syms}: {errs}")
    assert errs["fp64"] < 1e-10 and errs["fp32"] < 1e-6


def test_staged_results():
    s = synth.tiny(fft=(16, 18, 20), with_wfc=False)
    rng = np.random.default_rng(3)
    dims = (s.nmodes, s.nmag) + tuple(s.fft_dims)
    one = 16 * int(np.prod(dims))
    nq = (16 << 20) // one + 3
    ctx = lelph.Context(s, "fp64")
    try:
        ctx.interp_begin((2, 1, 1), masses=np.linspace(1.5, 2.5, s.natom))
        for q in ([0.0, 0.0, 0.0], [0.5, 0.0, 0.0]):
            e, _ = np.linalg.qr(rng.standard_normal((s.nmodes,) * 2)
                                + 1j * rng.standard_normal((s.nmodes,) * 2))
            ctx.interp_add_coarse(q, e, rng.standard_normal(dims) * (1 + 0.5j))
        ctx.interp_finish()
        fine = rng.uniform(-0.5, 0.5, (nq, 3))
        whole = ctx.interp_dvscf(fine)
        parts = np.concatenate([ctx.interp_dvscf(f) for f in np.array_split(fine, 5)])
    finally:
        ctx.close()
    say(f"case: staged results {whole.nbytes} bytes")
    assert whole.nbytes % (2 << 20) and np.array_equal(whole, parts)


class DeviceArray:
    """device memory of the HIP runtime that the library is linked to"""

    def __init__(self, a):
        self.hip, self.a, self.p = lelph.lib(), a, ctypes.c_void_p()
        assert self.hip.hipMalloc(ctypes.byref(self.p), ctypes.c_size_t(a.nbytes)) == 0
        assert self.hip.hipMemcpy(self.p, a.ctypes.data_as(ctypes.c_void_p),
                                  ctypes.c_size_t(a.nbytes), 1) == 0

    def ptr(self):
        return ctypes.cast(self.p, abi.c_double_p)

    def back(self):
        assert self.hip.hipMemcpy(self.a.ctypes.data_as(ctypes.c_void_p), self.p,
                                  ctypes.c_size_t(self.a.nbytes), 2) == 0
        return self.a

    def free(self):
        self.hip.hipFree(self.p)


def test_device_memory_of_the_caller():
    """a large result into device memory, a G list from it: what the copy
    engine reads and writes, the host's own code must not touch"""
    s = synth.tiny(nbnds=3, fft=(16, 18, 20))
    pair = synth.kq_pairs(s, 0)[1]
    dims = (s.nmodes, s.nmag) + tuple(s.fft_dims)
    nq = (16 << 20) // (16 * int(np.prod(dims))) + 2
    say(f"case: device memory of the caller, {nq} potentials")
    rng = np.random.default_rng(4)
    ctx = lelph.Context(s, "fp64")
    dev = []
    try:
        ctx.set_dvscf(s.qpts[0], s.eigvec(0), s.dvscf(0), kernel="dfpt")
        g = ctx.gkq(*pair, qpt=s.qpts[0])
        w = s.wfcs[pair[1]]
        dev.append(DeviceArray(np.ascontiguousarray(w.gvec)))
        rc = lelph.lib().lelph_upload_wfc(ctx.h, pair[1], abi.dptr(w.wfc), dev[0].ptr(),
                                          abi.dptr(w.Fk), w.npw)
        assert rc == 0 and np.array_equal(ctx.gkq(*pair, qpt=s.qpts[0]), g)
        ctx.interp_begin((1, 1, 1), masses=np.linspace(1.5, 2.5, s.natom))
        ctx.interp_add_coarse([0.0, 0.0, 0.0], s.eigvec(0), s.dvscf(0))
        ctx.interp_finish()
        fine = np.ascontiguousarray(rng.uniform(-0.5, 0.5, (nq, 3)))
        ref = ctx.interp_dvscf(fine)
        assert ref.nbytes > 16 << 20
        dev.append(DeviceArray(np.zeros_like(ref)))
        rc = lelph.lib().lelph_interp_dvscf(ctx.h, nq, abi.dptr(fine), dev[1].ptr())
        assert rc == 0 and np.array_equal(dev[1].back(), ref)
    finally:
        ctx.close()
        for d in dev:
            d.free()
