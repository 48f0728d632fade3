"""MYHX_CX (complex level matrices) at the edges of its MFMA passes: one-level
operators, tile edges and remainders, k remainders, one, two and four waves
per tile, DEPCX on either outer level, several vectors, with and without an
imaginary diagonal.

Reference: dense complex mode products (numpy); tolerance 1e-12 of the
largest entry, the bound of the other MYHX_CX tests.
"""
import numpy as np
import pytest

from scalit_amd import _lib as L
from scalit_amd import problems as P
from scalit_amd.context import Context

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sN,deps,nvec", [
    ((7,), (), 2),
    ((1, 1), (), 1),
    ((2, 3), (1,), 2),
    ((16, 16), (), 1),
    ((17, 33), (1,), 3),
    ((64, 65), (1,), 1),
    ((129, 40, 2), (2,), 1),       # 48 tiles of four waves, three chunks of k
    ((70, 50, 9), (2,), 2),        # 360 tiles: two waves
    ((20, 24, 48), (1, 2), 4),     # 768 tiles: one wave
    ((6, 5, 4, 7), (1, 3), 3),
    ((3, 2, 130), (2,), 1),
    ((4, 3, 30, 30), (1, 3), 5),   # small levels in many planes: one thread per output
    ((8, 40, 2, 25), (2,), 2),     # and only the level of two points
])
def test_complex_levels(sN, deps, nvec):
    g = P.rng(8)

    def cx(*shape):
        return g.standard_normal(shape) + 1j * g.standard_normal(shape)

    h0, dep, dim = [], [], 1
    for l, n in enumerate(sN):
        h0.append(cx(n, n) / np.sqrt(n))
        dep.append(cx(dim) if l in deps else None)
        dim *= n
    res, ap = g.standard_normal(dim), g.uniform(0, 1, size=dim)
    ctx = Context(sN, [d is not None for d in dep])
    for l, h in enumerate(h0):
        ctx.set_h0_cx(l + 1, h)
        if dep[l] is not None:
            ctx.set_dep_cx(l + 1, dep[l])
    ctx.set_res(res)
    ctx.set_ap(L.AP, ap)
    ctx.set_shift(0.31)
    ctx.set_scx(True)
    x = cx(nvec, dim)
    xd = ctx.to_device_cx(x)
    for ntype, diag in ((L.TA0, res + 0j), (L.TMAP, res - 0.31 - 1j * ap)):
        ref, inner = diag * x, 1
        for h, d in zip(h0, dep):
            z = np.einsum("ij,ajk->aik", h, x.reshape(-1, h.shape[0], inner))
            ref = ref + (z if d is None else z * d).reshape(x.shape)
            inner *= h.shape[0]
        y = Context.from_device_cx(ctx.hx_cx(xd, ntype))
        err = float(np.abs(y - ref).max() / np.abs(ref).max())
        print(sN, ntype, err, flush=True)
        assert err <= 1e-12
    ctx.close()
