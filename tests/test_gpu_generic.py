"""H*X of the generic path (any number of levels and DEP pattern) at the edges
of its first pass, levels 1 and 2 with the diagonal on MFMA tiles: one-point
levels, tile edges and remainders, k remainders, one, two and four waves per
tile, several planes, with and without DEP, nonsymmetric level matrices
forward and adjoint, FP64 / FP32 / BF16 storage, and per-vector shifts.

Reference: dense mode products in FP64 (numpy) of the values the device
holds.  Tolerances relative to the largest entry: FP64 1e-12 (the parity bound
of the other H*X tests), FP32 2e-6 and BF16 storage 2e-2 likewise.
"""
import numpy as np
import pytest
import torch

from scalit_amd import _lib as L
from scalit_amd import problems as P
from scalit_amd.context import Context

pytestmark = pytest.mark.gpu

SHAPES = [
    ((1, 1), (), 1),
    ((2, 3), (1,), 2),
    ((16, 16), (), 1),
    ((17, 33), (1,), 3),
    ((400, 96), (1,), 1),      # four waves per tile
    ((400, 96), (1,), 2),      # two
    ((400, 96), (1,), 5),      # one
    ((5, 130), (), 7),
    ((259, 2), (), 4),
    ((31, 5, 4), (), 2),
    ((20, 18, 7), (1, 2), 9),
    ((6, 5, 4, 7), (1, 3), 3),
    ((4, 3, 17, 5), (2, 3), 2),
    ((3, 2, 200), (2,), 3),
    ((4, 3, 30, 30), (1, 3), 5),   # small levels in many planes: one thread per output
    ((8, 40, 2, 25), (2,), 4),     # and only the level of two points
]


def _operator(sN, deps, seed=3):
    g = P.rng(seed)
    h0, dep, dim = [], [], 1
    for l, n in enumerate(sN):
        h0.append(g.standard_normal((n, n)) / np.sqrt(n))
        dep.append(g.uniform(0.5, 1.5, size=dim) if l in deps else None)
        dim *= n
    res = g.standard_normal(dim)
    ctx = Context(sN, [d is not None for d in dep])
    for l, h in enumerate(h0):
        ctx.set_h0(l + 1, h)
        if dep[l] is not None:
            ctx.set_dep(l + 1, dep[l])
    ctx.set_res(res)
    return ctx, h0, dep, res


def _reference(h0, dep, res, x, shifts, trans=False):
    y = (res[None, :] - np.asarray(shifts).reshape(-1, 1)) * x
    inner = 1
    for h, d in zip(h0, dep):
        n = h.shape[0]
        z = np.einsum("ij,ajk->aik", h.T if trans else h, x.reshape(-1, n, inner))
        if d is not None:
            z = z * d
        y = y + z.reshape(x.shape)
        inner *= n
    return y


def _rel(a, b):
    return float(np.abs(a - b).max() / np.abs(b).max())


@pytest.mark.parametrize("sN,deps,nvec", SHAPES)
def test_generic_levels(sN, deps, nvec):
    L.lib().scalit_debug_force_generic(1)
    try:
        ctx, h0, dep, res = _operator(sN, deps)
        ctx.set_shift(0.37)
        x = P.random_vectors(ctx.N, nvec, 9)
        xd = ctx.to_device(x)
        assert _rel(ctx.hx(xd).cpu().numpy(), _reference(h0, dep, res, x, 0.0)) <= 1e-12
        sh = np.linspace(-0.5, 0.5, nvec)
        assert _rel(ctx.hx(xd, shifts=sh).cpu().numpy(), _reference(h0, dep, res, x, sh)) <= 1e-12
        dx, dv = ctx.hx_adjoint(xd, ctx.to_device(x[::-1].copy()), L.TA1)
        assert _rel(dx.cpu().numpy(), _reference(h0, dep, res, x[::-1], 0.37, True)) <= 1e-12
        for dt, tol in ((torch.float32, 2e-6), (torch.bfloat16, 2e-2)):
            xl = ctx.to_device(x, dt)
            y = ctx.hx_lp(xl, L.TA1).double().cpu().numpy()
            assert _rel(y, _reference(h0, dep, res, xl.double().cpu().numpy(), 0.37)) <= tol, dt
        ctx.close()
    finally:
        L.lib().scalit_debug_force_generic(0)


def test_generic_strided_vectors():
    """Leading dimensions larger than N and a base that is only 8-byte aligned."""
    ctx, h0, dep, res = _operator((37, 21), (1,))
    n, ld = ctx.N, ctx.N + 5
    x = P.random_vectors(n, 3, 11)
    buf = torch.full((3 * ld + 1,), 7.0, dtype=torch.float64, device=ctx.dev)
    out = torch.full((3 * ld + 1,), 5.0, dtype=torch.float64, device=ctx.dev)
    for v in range(3):
        buf[1 + v * ld:1 + v * ld + n] = ctx.to_device(x[v])[0]
    import ctypes as C
    L.check(L.lib().scalit_hx(ctx.handle, L.TA0, 3, C.c_void_p(buf.data_ptr() + 8), ld, C.c_void_p(out.data_ptr() + 8),
                              ld, None, C.c_void_p(torch.cuda.current_stream().cuda_stream)))
    o = out.cpu().numpy()
    ref = _reference(h0, dep, res, x, 0.0)
    for v in range(3):
        assert _rel(o[1 + v * ld:1 + v * ld + n], ref[v]) <= 1e-12
        assert (o[1 + v * ld + n:1 + (v + 1) * ld] == 5.0).all()
    assert o[0] == 5.0
    ctx.close()


@pytest.mark.parametrize("va,vb", [(6, 3), (7, 0), (1, 3)])
@pytest.mark.parametrize("sN,nvec", [((5, 3, 2), 1), ((16, 16, 1), 2), ((17, 33, 7), 3), ((24, 32, 24), 1),
                                     ((30, 20, 33), 4), ((20, 18, 50), 16), ((70, 40, 9), 2)])
def test_three_levels_by_tiles(monkeypatch, sN, nvec, va, vb):
    """The 3-level operator's tile variants: levels 1 and 2 by tiles (6), mode 3
    in the tiles (7), the mode-3 pass by tiles (3); nonsymmetric matrices."""
    monkeypatch.setenv("SCALIT_HX_VARIANT_A", str(va))
    monkeypatch.setenv("SCALIT_HX_VARIANT_B", str(vb))
    ctx, h0, dep, res = _operator(sN, (2,))
    ctx.set_shift(0.37)
    x = P.random_vectors(ctx.N, nvec, 9)
    xd = ctx.to_device(x)
    sh = np.linspace(-0.5, 0.5, nvec)
    assert _rel(ctx.hx(xd, shifts=sh).cpu().numpy(), _reference(h0, dep, res, x, sh)) <= 1e-12
    assert ctx.hx_variant(L.FP64, nvec) == (va, vb)
    dx, _ = ctx.hx_adjoint(xd, xd, L.TA1)
    assert _rel(dx.cpu().numpy(), _reference(h0, dep, res, x, 0.37, True)) <= 1e-12
    for dt, tol in ((torch.float32, 2e-6), (torch.bfloat16, 2e-2)):
        xl = ctx.to_device(x, dt)
        y = ctx.hx_lp(xl, L.TA1).double().cpu().numpy()
        assert _rel(y, _reference(h0, dep, res, xl.double().cpu().numpy(), 0.37)) <= tol, dt
    ctx.close()


@pytest.mark.parametrize("dt", [torch.float64, torch.float32, torch.bfloat16])
@pytest.mark.parametrize("sN,nvec", [((5, 3, 2), 1), ((16, 16, 1), 2), ((17, 33, 7), 3), ((24, 32, 24), 1),
                                     ((20, 18, 50), 16), ((37, 50, 41), 2), ((7, 9, 128), 3)])
def test_three_level_variants_agree(monkeypatch, sN, nvec, dt):
    """Every variant of the 3-level operator that a timing picks from gives the
    same bits for every stored type: the default slab pass with each form of
    pass B, another slab shape, the tile pass with each form, and, in FP64 and
    FP32, mode 3 in the tiles."""
    prob = P.build_problem(*sN, P.gaussian_potential(5), seed=5)
    ref = None
    for va, vb in ((1, 0), (1, 1), (1, 2), (1, 3), (5, 0), (6, 0), (6, 3), (7, 0)):
        if va == 7 and dt == torch.bfloat16:
            continue
        monkeypatch.setenv("SCALIT_HX_VARIANT_A", str(va))
        monkeypatch.setenv("SCALIT_HX_VARIANT_B", str(vb))
        ctx = Context.from_problem(prob, e0=0.01)
        x = ctx.to_device(P.random_vectors(ctx.N, nvec, 9), dt)
        y = ctx.hx(x, L.TA1) if dt == torch.float64 else ctx.hx_lp(x, L.TA1)
        assert ctx.hx_variant({torch.float64: L.FP64, torch.float32: L.FP32, torch.bfloat16: L.BF16}[dt], nvec) == (va, vb)
        ref = y if ref is None else ref
        assert torch.equal(y, ref), (va, vb, int((y != ref).sum()))
        ctx.close()


@pytest.mark.parametrize("sN,nvec,fused", [((24, 32, 24), 1, True), ((12, 14, 10), 120, True), ((32, 32, 56), 4, True),
                                           ((12, 14, 10), 150, False), ((20, 20, 20), 17, False),
                                           ((32, 32, 64), 4, False), ((16, 20, 70), 1, False)])
def test_bf16_variant_by_size(monkeypatch, sN, nvec, fused):
    """BF16 storage: the one-launch operator rounds Y once and the two passes
    twice, so that the sizes and not a timing decide: on either side of the line
    the default call gives the bits of that form."""
    prob = P.build_problem(*sN, P.gaussian_potential(5), seed=5)
    ys = []
    for va in (None, 7 if fused else 1):
        if va is not None:
            monkeypatch.setenv("SCALIT_HX_VARIANT_A", str(va))
            monkeypatch.setenv("SCALIT_HX_VARIANT_B", "0")
        ctx = Context.from_problem(prob, e0=0.01)
        ys.append(ctx.hx_lp(ctx.to_device(P.random_vectors(ctx.N, nvec, 9), torch.bfloat16), L.TA1))
        ctx.close()
    assert torch.equal(*ys)


@pytest.mark.parametrize("sN,nvec,variant", [((24, 32, 24), 1, (7, 0)), ((28, 36, 28), 6, (7, 0)),
                                             ((48, 64, 40), 2, (6, 3)), ((17, 23, 47), 5, (6, 3))])
def test_fp64_variant_by_size(monkeypatch, sN, nvec, variant):
    """The one-launch operator and, on the other side of its line, the tile forms
    of both passes: the slab pass's bits."""
    prob = P.build_problem(*sN, P.gaussian_potential(5), seed=5)
    ys = []
    for va in (None, 1):
        if va is not None:
            monkeypatch.setenv("SCALIT_HX_VARIANT_A", str(va))
            monkeypatch.setenv("SCALIT_HX_VARIANT_B", "0")
        ctx = Context.from_problem(prob, e0=0.01)
        ys.append(ctx.hx(ctx.to_device(P.random_vectors(ctx.N, nvec, 9)), L.TA1))
        if va is None:
            assert ctx.hx_variant(L.FP64, nvec) == variant
        ctx.close()
    assert torch.equal(*ys)


@pytest.mark.parametrize("sN,nvec", [((24, 32, 24), 1), ((37, 50, 41), 2), ((20, 20, 20), 17), ((16, 20, 70), 1)])
def test_captured_call_agrees(sN, nvec):
    """A recorded call of a batch size that was never applied before, which times
    nothing, and an eager call, which may, give the same bits on every replay."""
    prob = P.build_problem(*sN, P.gaussian_potential(5), seed=5)
    ctx, eager = Context.from_problem(prob, e0=0.01), Context.from_problem(prob, e0=0.01)
    x = ctx.to_device(P.random_vectors(ctx.N, nvec, 9))
    y = torch.empty_like(x)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        ctx.hx(x, L.TA1, out=y)
    for _ in range(3):
        y.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(eager.hx(x, L.TA1), y)
    ctx.close()
    eager.close()


@pytest.mark.parametrize("sN,nvec", [((5, 3, 2), 1), ((16, 17, 16), 2), ((24, 32, 24), 3), ((7, 130, 3), 2),
                                     ((70, 40, 9), 1)])
def test_rotations_by_tiles(sN, nvec):
    """P*X with the level >= 2 rotations tile by tile (also past 128 points), on
    seeded orthogonal rotations, against dense products; FP64 1e-12, FP32 1e-5
    (the shift lies below every EIG0, so the divide amplifies nothing)."""
    _check_px(sN, [nvec])


# each row: the sizes of one register form of the level-1 kernel's prefetch, with MFMA
# (8 vectors and more, or more than 256 outputs) and on the vector units
@pytest.mark.parametrize("n1", [20, 64, 65, 80, 81, 96, 97, 111, 112, 113, 128])
def test_px_level1_forms(n1):
    """P*X at the edges of level 1's forms: the largest block of a prefetch and
    one more, past the prefetch (113, 128), and batches on both sides of the MFMA
    rule, with a shift per vector; tolerances as above."""
    _check_px((n1, 3, 2), [1, 2, 3, 4, 5, 7, 8, 17])


def _check_px(sN, batches):
    g = P.rng(4)
    ctx = Context(sN, [False] * len(sN))
    n = ctx.N
    vosb = []
    for l, m in enumerate(sN):
        q = np.linalg.qr(g.standard_normal((ctx.blk[l], m, m)))[0]
        vosb.append(q.transpose(0, 2, 1).reshape(-1))   # column-major blocks
    eig0 = g.uniform(1.0, 2.0, size=n)
    ctx.set_precond(vosb, eig0)
    ctx.set_res(np.zeros(n))
    ctx.set_shift(0.5)

    def rot(z, l, trans):
        q = vosb[l].reshape(ctx.blk[l], sN[l], sN[l]).transpose(0, 2, 1)
        z = z.reshape(-1, ctx.blk[l], sN[l], ctx.dim[l])
        return np.einsum("bji,vbjk->vbik" if trans else "bij,vbjk->vbik", q, z).reshape(-1, n)

    for nvec in batches:
        x = P.random_vectors(n, nvec, 12)
        for sh in (None, np.linspace(-0.5, 0.5, nvec)):
            z = x
            for l in reversed(range(len(sN))):
                z = rot(z, l, True)
            z = z / (eig0 - (0.5 if sh is None else sh[:, None]))
            for l in range(len(sN)):
                z = rot(z, l, False)
            assert _rel(ctx.px(ctx.to_device(x), shifts=sh).cpu().numpy(), z) <= 1e-12, (nvec, sh)
            y = ctx.px_lp(ctx.to_device(x, torch.float32), shifts=sh)
            assert _rel(y.double().cpu().numpy(), z) <= 1e-5, (nvec, sh)
    ctx.close()
