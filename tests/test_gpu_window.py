"""Launches past the memory-side cache, whose tiles the XCDs take by windows: grids whose tile counts are no multiple of a
window, stepped by passes, lean, row, flat and adjoint kernels, against kernels of another tile shape (another number of
tiles), bit for bit."""

import numpy as np
import pytest
import torch

from tests import cases
from tests.test_gpu_flat import _engine as flat_engine
from tests.test_gpu_lean import _engine as lean_engine

pytestmark = pytest.mark.gpu


def _same(engines, steps=3):
    for e in engines:
        e.steps(steps)
    torch.cuda.synchronize()
    ref = engines[0].state_tensors()
    assert engines[0].E_flat.abs().max() > 0
    for e in engines[1:]:
        for x, y in zip(ref, e.state_tensors()):
            assert torch.equal(x, y)


@pytest.mark.parametrize("shape,adjoint", [((203, 187, 161), False), ((256, 257, 140), False), ((203, 187, 161), True)])
def test_real_engines(gpu, shape, adjoint):
    ns = cases.product_ns()
    kw = dict(pml=(0, 1, 2), kappa=2.0, material="dense", adjoint=adjoint)
    es = [lean_engine(ns, gpu, shape, **kw), lean_engine(ns, gpu, shape, tiling=(2, 4, 64, 5), **kw)]
    if not adjoint:
        inv = 1 / np.random.default_rng(4).uniform(1, 6, size=(3,) + shape)
        e = cases.make(ns, gpu, shape=shape, dx=2.0, dt=0.9 * 2.0 / np.sqrt(3), inv_eps=inv, material="dense", fused=True,
                       pml=ns.PMLSpec(cells=((2, 3),) * 3, kappa_max=2.0, alpha_max=0.01))
        cases.random_fields(e, 5)
        assert e._two_sets
        es.append(e)
    _same(es)


def test_periodic_engines(gpu):
    ns = cases.product_ns()
    _same([flat_engine(ns, gpu, (131, 121, 280), (True, True, False), True, True, tiling=t) for t in (None, (2, 4, 64, 5))])
