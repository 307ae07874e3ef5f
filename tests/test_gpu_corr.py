"""Source corrections made inside the bulk kernels against the same corrections as launches of their own, bit for bit
(lsf_step, which plans them in, against lsf_step_noalloc, which launches them): modal sources and gathers on points, lines,
planes and scattered nodes, several on the same nodes and more than a kernel takes, on D-form nodes, in single passes,
row kernels of other tile shapes and the kernels of periodic engines (real and complex), past the end of a source's
table; and operations that stay launches (rows outside the stepped box or too thin in theirs, a gather of the field it
writes). Engines of one batch against the same engines alone.
"""

import ctypes

import numpy as np
import pytest
import torch

from tests import cases

pytestmark = pytest.mark.gpu

H, E = 0, 3  # the correction phases


class _Ops:
    """A source that adds the given operations."""

    def __init__(self, ops):
        self.ops = ops

    def bind(self, eng):
        self.bind_native(eng)

    def bind_native(self, eng):
        rng = np.random.default_rng(9)
        cplx = eng.complex
        val = lambda *s: rng.standard_normal(s) + (1j * rng.standard_normal(s) if cplx else 0)  # noqa: E731
        for kind, phase, targets in self.ops:
            fld, t = ("H" if phase == H else "E"), eng.native_index(targets)
            if kind == "modal":
                eng.add_modal(phase, fld, t, 1e-2 * val(len(t), 2), rng.standard_normal((11, 2)))
            elif kind == "gather":
                src = torch.as_tensor(val(50), dtype=eng.E_flat.dtype, device=eng.E_flat.device)
                eng._keep.append(src)
                eng.add_gather(phase, fld, t, src, rng.integers(0, 50, (len(t), 3)), 1e-2 * val(len(t), 3))
            else:  # reads the engine's own E or H
                src = eng.E_flat if kind == "own E" else eng.H_flat
                eng.add_gather(phase, fld, t, src, rng.integers(0, src.numel(), (len(t), 2)), 1e-2 * val(len(t), 2))


def _targets(ns, shape, what, rng, lo=2):
    n = shape
    if what == "point":
        return np.array([ns.flat_index(2, n[0] // 2, n[1] // 2, n[2] // 2, shape)])
    if what == "line":
        return ns.flat_index(0, np.arange(1, n[0] - 1), 2, n[2] - 3, shape)
    if what == "plane":
        i, j = (v.ravel() for v in np.meshgrid(np.arange(1, n[0] - 1), np.arange(1, n[1] - 1), indexing="ij"))
        return np.concatenate([ns.flat_index(c, i, j, n[2] // 2, shape) for c in (0, 1)])
    if what == "edge":  # a node that never steps
        return np.array([ns.flat_index(0, 2, 0, 2, shape), ns.flat_index(0, 2, 2, 2, shape)])
    m = 12 if what == "few" else 3 * int(np.prod(shape)) // 20
    c = rng.integers(0, 3, m)
    p = [rng.integers(lo, v - 2, m) for v in n]
    return np.unique(np.concatenate([ns.flat_index(q, *[x[c == q] for x in p], shape) for q in range(3)]))


def _engine(ns, device, shape, ops, periodic=(False,) * 3, bloch=False, poles=0, tiling=None, fused=None):
    rng = np.random.default_rng(7)
    inv = 1 / rng.choice([1.0, 2.25, 4.0], size=(3,) + shape)
    groups = []
    if poles:
        idx = _targets(ns, shape, "many", rng)
        idx = np.union1d(idx, _targets(ns, shape, "plane", rng))
        inv.reshape(-1)[idx] = 1 / 1.5
        groups = [ns.DispersiveGroup(idx=idx, media=[cases.medium(ns, 1.5, cases.lorentz3(rng, poles))],
                                     frac=np.ones((1, len(idx))), w=None)]
    t = [(k, ph, _targets(ns, shape, what, rng)) for k, ph, what in ops]
    old = ns.Engine.tiling
    ns.Engine.tiling = tiling or old
    try:
        e = cases.make(ns, device, shape=shape, dx=2.0, dt=0.9 * 2.0 / np.sqrt(3), inv_eps=inv, groups=groups,
                       periodic=periodic, bloch=tuple(0.03 if bloch and p else 0.0 for p in periodic),
                       pml=ns.PMLSpec(cells=tuple((0, 0) if p else (2, 2) for p in periodic), kappa_max=2.0),
                       sources=[_Ops(t)], fused=fused)
    finally:
        ns.Engine.tiling = old
    if poles == 0:
        g = torch.Generator(device="cpu").manual_seed(3)
        for F, R in ((e.E, e.RE), (e.H, e.RH)):
            for c in range(3):
                F[c][tuple(R[c])] = torch.randn(F[c][tuple(R[c])].shape, generator=g, dtype=F.dtype).to(F.device)
    return e


LISTS = [[("modal", E, "point")],
         [("modal", E, "plane"), ("gather", H, "plane"), ("gather", E, "plane")],
         [("gather", H, "line"), ("modal", H, "few"), ("modal", E, "line"), ("own H", E, "plane"), ("own E", H, "plane")],
         [("modal", E, "few"), ("modal", E, "point"), ("modal", E, "plane"), ("modal", E, "line"), ("gather", E, "line")],
         [("modal", E, "many"), ("gather", E, "few"), ("own E", E, "point"), ("modal", E, "point")],
         [("modal", E, "edge"), ("modal", E, "plane")]]
FORMS = [dict(), dict(poles=2), dict(fused=False), dict(fused=False, poles=3), dict(tiling=(2, 8, 32, 5)),
         dict(periodic=(True, True, False)), dict(periodic=(True, True, False), bloch=True),
         dict(periodic=(True, True, True), bloch=True), dict(periodic=(True, False, False), bloch=True, tiling=(2, 4, 64, 3)),
         dict(periodic=(True, True, False), bloch=True, poles=1)]


@pytest.mark.parametrize("form", range(len(FORMS)))
@pytest.mark.parametrize("ops", range(len(LISTS)))
def test_corrections_equal_the_launches(gpu, ops, form):
    from lightsmith_amd import _lib
    from tests.test_zz_no_alloc import _bind
    lib, ns = _lib.load(), cases.product_ns()
    noalloc = _bind(lib)
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    for shape in ((17, 12, 15), (66, 9, 11)):
        a, b = (_engine(ns, gpu, shape, LISTS[ops], **FORMS[form]) for _ in range(2))
        for n in (1, 4, 9):  # the tables hold 11 steps
            _lib.check(lib.lsf_step(a._h, n, stream), "lsf_step")
            _lib.check(noalloc(b._h, n, stream), "lsf_step_noalloc")
        torch.cuda.synchronize()
        for q, (x, y) in enumerate(zip(a.state_tensors(), b.state_tensors())):
            assert torch.equal(x, y), (shape, q)
        assert a.E_flat.abs().max() > 0


def test_corrections_in_a_batch(gpu):
    from lightsmith_amd.fdtd.batch import Batch
    ns = cases.product_ns()
    forms = [dict(), dict(poles=2), dict(periodic=(True, True, False), bloch=True)]
    alone = [_engine(ns, gpu, (17, 12, 15), LISTS[q], **f) for q, f in enumerate(forms)]
    mem = [_engine(ns, gpu, (17, 12, 15), LISTS[q], **f) for q, f in enumerate(forms)]
    batch = Batch(mem, schedule=(1, 4, 64, 8, 0))
    for e in alone:
        e.steps(9)
    batch.steps(9)
    torch.cuda.synchronize()
    for a, b in zip(alone, mem):
        for x, y in zip(a.state_tensors(), b.state_tensors()):
            assert torch.equal(x, y)
    batch.close()


@pytest.mark.parametrize("tiling", [(1, 4, 64, 4), (2, 4, 64, 4)])
def test_corrections_of_an_adjoint_engine(gpu, tiling):
    """An adjoint engine's gathers and modal sources run, whatever the tile shape: lsf_step, lsf_step_noalloc and a batch agree."""
    from lightsmith_amd import _lib
    from lightsmith_amd.fdtd.batch import Batch
    from tests.test_zz_no_alloc import _bind
    lib, ns = _lib.load(), cases.product_ns()
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    a, b, m, bare = (_engine(ns, gpu, (17, 12, 15), ops, tiling=tiling, fused=False) for ops in [LISTS[1]] * 3 + [[]])
    for e in (a, b, m, bare):
        _lib.check(lib.lsf_set_adjoint(e._h, 1), "lsf_set_adjoint")
    batch = Batch([m], schedule=tiling + (0,))
    for n in (1, 4):
        a.steps(n)
        bare.steps(n)
        batch.steps(n)
        _lib.check(_bind(lib)(b._h, n, stream), "lsf_step_noalloc")
    torch.cuda.synchronize()
    for x, y, z in zip(a.state_tensors(), b.state_tensors(), m.state_tensors()):
        assert torch.equal(x, y) and torch.equal(x, z)
    assert not torch.equal(a.E_flat, bare.E_flat) and not torch.equal(a.H_flat, bare.H_flat)
    batch.close()
