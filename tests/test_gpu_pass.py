"""The single-pass step against the H and E row kernels, bit for bit: row widths and planes around the 62 cells a wavefront
owns (rows shorter than one, a plane of one wavefront, several rows per wavefront), z extents around the planes of a
tile, CPML on every axis, on one or on none, with and without kappa, D-form nodes of one to four poles (dense enough
for several rounds a plane), dense and indexed material, odd step counts.
"""

import numpy as np
import pytest
import torch

from tests import cases

pytestmark = pytest.mark.gpu

SHAPES = [(5, 5, 6), (6, 10, 5), (7, 9, 31), (31, 3, 9), (62, 6, 17), (63, 7, 8), (124, 11, 9), (125, 130, 13),
          (40, 66, 122)]


def _engine(ns, device, shape, pml, kappa, poles, material, fused, frac=0.5, seed=4):
    rng = np.random.default_rng(seed)
    eps = rng.choice([1.0, 2.25, 4.0], size=(3,) + shape) if material == "indexed" else \
        rng.uniform(1, 6, size=(3,) + shape)
    inv = 1 / eps
    groups = []
    if poles:  # the components of the E-stepped box, each its own draw
        pick = rng.random((3,) + shape) < frac
        for c in range(3):
            for ax in range(3):
                edge = np.arange(shape[ax])
                keep = (edge >= (0 if ax == c else 1)) & (edge < shape[ax] - 1)
                pick[c] &= keep.reshape([-1 if a == ax else 1 for a in range(3)])
        which = rng.integers(0, 2, size=pick.shape)
        for q in range(2):  # two media
            c, i, j, k = np.nonzero(pick & (which == q))
            idx = np.sort(ns.flat_index(c, i, j, k, shape))
            if len(idx):
                med = cases.medium(ns, 1.5 + q, cases.lorentz3(np.random.default_rng(seed + q), poles))
                groups.append(ns.DispersiveGroup(idx=idx, media=[med], frac=np.ones((1, len(idx))), w=None))
                inv.reshape(-1)[idx] = 1 / (1.5 + q)
    cells = tuple((0, 0) if n < 6 or ax not in pml else (2, 3 if n > 6 else 2) for ax, n in enumerate(shape))
    kw = dict(shape=shape, dx=2.0, dt=0.9 * 2.0 / np.sqrt(3), inv_eps=inv, groups=groups,
              pml=ns.PMLSpec(cells=cells, kappa_max=kappa, alpha_max=0.01), material=material, fused=fused)
    e = cases.make(ns, device, **kw)
    cases.random_fields(e, seed + 1)
    return e


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("pml,kappa", [((), 1.0), ((0,), 1.0), ((1,), 2.0), ((2,), 1.0), ((0, 1, 2), 1.0), ((0, 1, 2), 3.0)])
def test_pass_equals_the_two_kernels(gpu, shape, pml, kappa):
    ns = cases.product_ns()
    for poles in (0, 1, 2, 3, 4):
        for material in ("dense", "indexed"):
            a, b = (_engine(ns, gpu, shape, pml, kappa, poles, material, f) for f in (True, False))
            assert a._two_sets and not b._two_sets
            for n in (1, 4, 7):
                a.steps(n)
                b.steps(n)
            for q, (x, y) in enumerate(zip(a.state_tensors(), b.state_tensors())):
                assert torch.equal(x, y), (shape, pml, kappa, poles, material, q)
            assert torch.isfinite(a.E_flat).all()


def test_the_pass_is_taken_by_working_set(gpu):
    """Small boxes step by passes unless told not to; complex or periodic engines, other tile shapes and engines with
    work between the H and the E update never do."""
    ns = cases.product_ns()
    small = cases.dispersive_box(ns, gpu, shape=(30, 28, 26))
    assert not small._two_sets  # not before it steps by itself
    small.step()
    assert small._two_sets
    for e in (cases.dispersive_box(ns, gpu, shape=(30, 28, 26), fused=False), cases.tfsf_box(ns, gpu)):
        e.step()
        assert not e._two_sets
    old = ns.Engine.tiling
    ns.Engine.tiling = (2, 4, 64, 8)
    try:
        assert not cases.dispersive_box(ns, gpu, shape=(30, 28, 26), fused=True)._two_sets
    finally:
        ns.Engine.tiling = old
