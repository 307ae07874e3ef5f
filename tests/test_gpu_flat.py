"""The flat bulk kernels (engines with a periodic axis at the one-row, four-wavefront tilings) against the row kernels of
another tile shape, bit for bit, and against the FP64 oracle: row widths around the two-cell lane (odd widths, the
narrowest cell), planes of less and more than one wavefront, every set of periodic axes with CPML on the others, real
and complex fields, dense and indexed material.
"""

import numpy as np
import pytest
import torch

from tests import cases

pytestmark = pytest.mark.gpu

SHAPES = [(3, 3, 40), (4, 7, 23), (5, 12, 21), (33, 13, 18), (50, 31, 20), (65, 9, 17)]
PERIODIC = [(True, True, False), (True, False, False), (False, True, False), (False, False, True), (True, True, True)]


def _engine(ns, device, shape, periodic, bloch, indexed, tiling=None, seed=3):
    rng = np.random.default_rng(seed)
    d = (3.0, 2.5, 2.0)
    eps = rng.choice([1.0, 2.25, 4.0], size=(3,) + shape) if indexed else rng.uniform(1, 6, size=(3,) + shape)
    cells = tuple((0, 0) if p or n < 9 else (2, 3) for p, n in zip(periodic, shape))
    kpar = tuple(k if p and bloch else 0.0 for k, p in zip((0.05, -0.03, 0.04), periodic))
    kw = dict(shape=shape, dx=d, dt=0.9 / np.sqrt(sum(1 / v ** 2 for v in d)), inv_eps=1 / eps, periodic=periodic,
              bloch=kpar, pml=ns.PMLSpec(cells=cells, kappa_max=2.0, alpha_max=0.01))
    old = ns.Engine.tiling if tiling else None
    if tiling:
        ns.Engine.tiling = tiling
    try:
        e = cases.make(ns, device, **kw)
    finally:
        if tiling:
            ns.Engine.tiling = old
    rng = np.random.default_rng(seed + 1)
    for F, R in ((e.E, e.RE), (e.H, e.RH)):
        for c in range(3):
            n = tuple(r.stop - r.start for r in R[c])
            v = rng.standard_normal(n) + (1j * rng.standard_normal(n) if any(kpar) else 0)
            F[c][tuple(R[c])] = torch.as_tensor(v, dtype=F.dtype, device=F.device) if hasattr(F, "cpu") else v
    return e


@pytest.mark.parametrize("bloch", [False, True])
@pytest.mark.parametrize("periodic", PERIODIC)
@pytest.mark.parametrize("shape", SHAPES)
def test_flat_kernels_equal_the_row_kernels(gpu, shape, periodic, bloch):
    for indexed in (False, True):
        a = _engine(cases.product_ns(), gpu, shape, periodic, bloch, indexed)
        b = _engine(cases.product_ns(), gpu, shape, periodic, bloch, indexed, tiling=(2, 4, 64, 5))
        a.steps(30)
        b.steps(30)
        for x, y in zip(a.state_tensors(), b.state_tensors()):
            assert torch.equal(x, y), (shape, periodic, bloch, indexed)


@pytest.mark.parametrize("periodic", PERIODIC)
def test_flat_kernels_match_the_oracle(gpu, periodic):
    shape = (33, 13, 18)
    o = _engine(cases.oracle_ns(), None, shape, periodic, True, False)
    g = _engine(cases.product_ns(), gpu, shape, periodic, True, False)
    o.run(60)
    g.steps(60)
    m = cases.real_mask(shape, periodic)
    (Eo, Ho), (Eg, Hg) = cases.fields(o), cases.fields(g)
    eE, eH = cases.rel_l2(Eg, Eo, m), cases.rel_l2(Hg, Ho, m)
    print(f"{periodic}: rel L2 E {eE:.2e} H {eH:.2e}")
    assert eE < 1e-5 and eH < 1e-5  # the parity tolerance of float32 fields (tests/test_gpu_parity.py)
