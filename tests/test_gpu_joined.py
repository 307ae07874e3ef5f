"""Sub-engines whose updates run inside their engine's launches against the row kernels of another tile shape, which join
nothing, bit for bit: sub-engines whose corrections read their engine's field or each other's (these follow it in launches of
their own), alone and in a batch.
"""

import numpy as np
import pytest
import torch

from tests import cases

pytestmark = pytest.mark.gpu

H, E = 0, 3  # the correction phases


def _engine(gpu, links, bloch, tiling, shape=(19, 14, 26)):
    """An engine and two sub-engines. links: (reader, phase, read) gathers; 0 is the engine, 1 and 2 the sub-engines."""
    ns = cases.product_ns()
    old = ns.Engine.tiling
    ns.Engine.tiling = tiling
    try:
        def make(shape, **kw):
            n = int(np.prod(shape))
            return cases.make(ns, gpu, shape=shape, dx=2.0, dt=0.9 * 2.0 / np.sqrt(3), periodic=(True, True, False),
                              inv_eps=1 / np.random.default_rng(n).choice([1.0, 2.25], (3,) + shape),
                              bloch=(0.03, -0.02, 0.0) if bloch else (0.0,) * 3, pml=ns.PMLSpec(cells=((0, 0), (0, 0), (3, 3))), **kw)
        eng = make(shape)
        all_ = [eng] + [make((3 + q, 3, 26), _sub=True, _counter=eng._counter) for q in range(2)]
    finally:
        ns.Engine.tiling = old
    for sub in all_[1:]:
        eng.add_subengine(sub)
    rng = np.random.default_rng(5)
    val = lambda *s: rng.standard_normal(s) + (1j * rng.standard_normal(s) if bloch else 0)  # noqa: E731
    for reader, phase, read in links:
        e, fld = all_[reader], "H" if phase == H else "E"
        src = all_[read].H_flat if phase == H else all_[read].E_flat  # the field that the same half-step updates
        i, j = (v.ravel() for v in np.meshgrid(np.arange(1, e.shape[0] - 1), np.arange(1, e.shape[1] - 1), indexing="ij"))
        t = e.native_index(np.concatenate([ns.flat_index(c, i, j, 11, e.shape) for c in (0, 1)]))
        e.add_gather(phase, fld, t, src, rng.integers(0, src.numel(), (len(t), 5)), 0.05 * val(len(t), 5))
    for q, e in enumerate(all_):
        g = torch.Generator().manual_seed(q)
        for F, R in ((e.E, e.RE), (e.H, e.RH)):
            for c in range(3):
                F[c][tuple(R[c])] = torch.randn(F[c][tuple(R[c])].shape, generator=g, dtype=F.dtype).to(F.device)
    return eng


@pytest.mark.parametrize("bloch", [False, True])
@pytest.mark.parametrize("links", [(), ((0, H, 1), (0, E, 2)), ((1, H, 0),), ((1, E, 0),), ((2, H, 1), (2, E, 1)), ((1, H, 2),),
                                   ((1, E, 2), (2, E, 0))])
def test_sub_engines_that_read_their_engine_or_each_other(gpu, links, bloch):
    from lightsmith_amd.fdtd.batch import Batch
    a, b, m = (_engine(gpu, links, bloch, t) for t in ((1, 4, 64, 4), (2, 4, 64, 4), (1, 4, 64, 4)))
    batch = Batch([m], schedule=(1, 4, 64, 4, 0))
    for e in (a, b, batch):
        e.steps(7)
    torch.cuda.synchronize()
    for q, (x, y, z) in enumerate(zip(a.state_tensors(), b.state_tensors(), m.state_tensors())):
        assert torch.equal(x, y) and torch.equal(x, z), q
    assert a.E_flat.abs().max() > 0 and torch.isfinite(a.E_flat.abs()).all()
    batch.close()


@pytest.mark.parametrize("which", [0, 1])
def test_a_sub_engine_on_the_other_side_of_an_adjoint(gpu, which):
    """A forward sub-engine of an adjoint engine (0) and an adjoint one of a forward engine (1) step their own update."""
    from lightsmith_amd import _lib
    ns, out = cases.product_ns(), []
    for tiling in ((1, 4, 64, 4), (2, 4, 64, 4)):
        old = ns.Engine.tiling
        ns.Engine.tiling = tiling
        try:
            make = lambda s, **kw: cases.make(ns, gpu, shape=s, dx=2.0, dt=0.9 * 2.0 / np.sqrt(3), fused=False,  # noqa: E731
                                              inv_eps=np.full((3,) + s, 1 / 2.25), pml=ns.PMLSpec(cells=((2, 2),) * 3), **kw)
            eng = make((17, 12, 15))
            sub = make((9, 8, 11), _sub=True, _counter=eng._counter)
        finally:
            ns.Engine.tiling = old
        _lib.check(eng.lib.lsf_set_adjoint((eng, sub)[which]._h, 1), "lsf_set_adjoint")
        eng.add_subengine(sub)
        for e in (eng, sub):
            cases.random_fields(e, 3)
        eng.steps(5)
        out.append(eng)
    torch.cuda.synchronize()
    for q, (x, y) in enumerate(zip(*(e.state_tensors() for e in out))):
        assert torch.equal(x, y), q
