"""The lean bulk kernels (real engines without periodic axes at the one-row, four-wavefront tilings) against the row kernels of
another tile shape, bit for bit: row widths and planes around the 63 cells a wavefront owns, z extents around the planes
of a tile, CPML on every axis, on one or on none, with and without kappa, cubic cells and others, dense and indexed
material, D-form nodes (H only), forward and adjoint, and in a batch with a persistent grid.
"""

import numpy as np
import pytest
import torch

from tests import cases

pytestmark = pytest.mark.gpu

SHAPES = [(3, 3, 3), (5, 12, 6), (6, 10, 5), (7, 9, 31), (31, 3, 9), (62, 6, 17), (63, 7, 8), (64, 5, 10), (126, 11, 9),
          (125, 130, 13), (40, 66, 122)]


def _engine(ns, device, shape, pml, kappa, material, adjoint=False, poles=0, dx=2.0, tiling=None, seed=4):
    rng = np.random.default_rng(seed)
    eps = rng.choice([1.0, 2.25, 4.0], size=(3,) + shape) if material == "indexed" else \
        rng.uniform(1, 6, size=(3,) + shape)
    inv, groups = 1 / eps, []
    if poles:
        i, j, k = np.nonzero(rng.random(tuple(n - 2 for n in shape)) < 0.3)
        idx = np.sort(np.concatenate([ns.flat_index(c, i + 1, j + 1, k + 1, shape) for c in range(3)]))
        inv.reshape(-1)[idx] = 1 / 1.5
        groups = [ns.DispersiveGroup(idx=idx, media=[cases.medium(ns, 1.5, cases.lorentz3(rng, poles))],
                                     frac=np.ones((1, len(idx))), w=None)]
    cells = tuple((0, 0) if n < 6 or ax not in pml else (2, 3 if n > 6 else 2) for ax, n in enumerate(shape))
    d = np.broadcast_to(dx, 3)
    old = ns.Engine.tiling
    ns.Engine.tiling = tiling or old
    try:
        e = cases.make(ns, device, shape=shape, dx=dx, dt=0.9 / np.sqrt(sum(1 / v ** 2 for v in d)), inv_eps=inv,
                       groups=groups, pml=ns.PMLSpec(cells=cells, kappa_max=kappa, alpha_max=0.01), material=material,
                       fused=False)
    finally:
        ns.Engine.tiling = old
    if adjoint:
        from lightsmith_amd import _lib
        _lib.check(e.lib.lsf_set_adjoint(e._h, 1), "lsf_set_adjoint")
    cases.random_fields(e, seed + 1)
    return e


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("pml,kappa", [((), 1.0), ((0,), 1.0), ((1,), 2.0), ((2,), 1.0), ((0, 1, 2), 1.0), ((0, 1, 2), 3.0)])
def test_lean_kernels_equal_the_row_kernels(gpu, shape, pml, kappa):
    ns = cases.product_ns()
    for kw in (dict(material="dense"), dict(material="indexed"), dict(material="dense", dx=(2.0, 1.5, 3.0)),
               dict(material="indexed", poles=2), dict(material="dense", adjoint=True),
               dict(material="indexed", adjoint=True, dx=(2.0, 1.5, 3.0))):
        a = _engine(ns, gpu, shape, pml, kappa, **kw)
        b = _engine(ns, gpu, shape, pml, kappa, tiling=(2, 4, 64, 5), **kw)
        a.steps(11)
        b.steps(11)
        for q, (x, y) in enumerate(zip(a.state_tensors(), b.state_tensors())):
            assert torch.equal(x, y), (shape, pml, kappa, kw, q)
        assert torch.isfinite(a.E_flat).all() and a.E_flat.abs().max() > 0


def test_lean_kernels_in_a_persistent_batch(gpu):
    from lightsmith_amd.fdtd.batch import Batch
    ns = cases.product_ns()
    kws = [dict(shape=(40, 66, 22), material="dense"), dict(shape=(63, 7, 8), material="indexed"),
           dict(shape=(31, 20, 9), material="indexed", poles=1), dict(shape=(31, 20, 9), material="dense", adjoint=True)]
    mem, ref = ([_engine(ns, gpu, pml=(0, 1, 2), kappa=2.0, tiling=t, **kw) for kw in kws] for t in (None, (2, 4, 64, 5)))
    for sched in ((1, 4, 64, 8, 0), (1, 4, 32, 8, 16)):
        batch = Batch(mem, schedule=sched)
        batch.steps(7)
        for e in ref:
            e.steps(7)
        for e, m in zip(ref, mem):
            for x, y in zip(e.state_tensors(), m.state_tensors()):
                assert torch.equal(x, y)
        batch.close()
