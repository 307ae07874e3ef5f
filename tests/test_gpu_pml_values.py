"""CPML values at their limits, every bulk kernel against the row kernels of another tile shape: an infinite or undefined psi
reaches the cells that the update carries it to and no others; a profile's b, c and 1/kappa count only inside its slab,
and 1/kappa only where the axis was given with has_kappa. Single pass, lean, flat (real and complex) and adjoint kernels.
"""

import numpy as np
import pytest
import torch

from tests import cases

pytestmark = pytest.mark.gpu

SHAPE = (21, 18, 17)
FORMS = {"pass": dict(fused=True), "lean": dict(fused=False), "flat": dict(periodic=(False, True, False)),
         "flat complex": dict(periodic=(False, True, False), bloch=True), "adjoint": dict(fused=False, adjoint=True)}


def _engine(gpu, form, rows=False):
    """An engine of the form, or its twin on the row kernels."""
    ns, kw = cases.product_ns(), dict(FORMS[form])
    adjoint, bloch, per = kw.pop("adjoint", False), kw.pop("bloch", False), kw.pop("periodic", (False,) * 3)
    old = ns.Engine.tiling
    ns.Engine.tiling = (2, 4, 64, 5) if rows else old
    try:
        e = cases.make(ns, gpu, shape=SHAPE, dx=2.0, dt=0.9 * 2.0 / np.sqrt(3), periodic=per,
                       bloch=tuple(0.03 if bloch and p else 0.0 for p in per),
                       inv_eps=1 / np.random.default_rng(1).uniform(1, 4, (3,) + SHAPE),
                       pml=ns.PMLSpec(cells=tuple((0, 0) if p else (3, 4) for p in per), kappa_max=2.0, alpha_max=0.01),
                       **({} if rows else kw))
    finally:
        ns.Engine.tiling = old
    g = torch.Generator().manual_seed(3)
    for F, R in ((e.E, e.RE), (e.H, e.RH)):
        for c in range(3):
            F[c][tuple(R[c])] = torch.randn(F[c][tuple(R[c])].shape, generator=g, dtype=F.dtype).to(F.device)
    if adjoint:
        from lightsmith_amd import _lib
        _lib.check(e.lib.lsf_set_adjoint(e._h, 1), "lsf_set_adjoint")
    return e


def _same(a, b, what):
    torch.cuda.synchronize()
    for q, (x, y) in enumerate(zip(a.state_tensors(), b.state_tensors())):
        x, y = (torch.view_as_real(v) if v.is_complex() else v for v in (x, y))
        assert torch.equal(torch.isnan(x), torch.isnan(y)), (what, q)
        assert torch.equal(torch.nan_to_num(x, nan=0.0), torch.nan_to_num(y, nan=0.0)), (what, q)


@pytest.mark.parametrize("value", [np.inf, np.nan])
@pytest.mark.parametrize("form", FORMS)
def test_a_non_finite_psi_stays_with_its_cell(gpu, form, value):
    n_psi = len(_engine(gpu, form)._state)
    for block in range(n_psi):
        a, b = _engine(gpu, form), _engine(gpu, form, rows=True)
        assert a._two_sets == (form == "pass")
        for e in (a, b):
            psi = e._state[block]
            psi.view(2, -1)[:, 0] = value  # the first cell of either component's slab
            psi[psi.numel() // 3] = value
            e.steps(3)
        _same(a, b, (form, block))
        assert torch.isfinite(a.E_flat.abs()).float().mean() > 0.9


def _axes(e):
    """(field, axis, profile, slab cells, psi) of the engine's CPML, as it gave them to the library."""
    from lightsmith_amd.fdtd.engine import pml_axis_profile
    spec = cases.product_ns().PMLSpec(cells=e.pml_cells, kappa_max=2.0, alpha_max=0.01)
    state = iter(e._state)
    for d in range(3):
        if any(e.pml_cells[d]):
            for f in range(2):
                prof, ns, has_k = pml_axis_profile(spec, e.shape, e.dt, e.spacing, d, f)
                yield f, d, prof, ns, has_k, next(state).view(2, -1)


def _set(e, f, d, prof, ns, has_k, psi):
    from lightsmith_amd import _lib
    p = [_lib.ptr(psi[0 if c == min(q for q in range(3) if q != d) else 1]) if c != d else None for c in range(3)]
    _lib.check(e.lib.lsf_set_pml(e._h, f, d, _lib.ptr(e.to_device(prof.astype(np.float32))), ns, *p, int(has_k)), "lsf_set_pml")


@pytest.mark.parametrize("form", FORMS)
def test_a_profile_counts_inside_its_slab_only(gpu, form):
    a, b, ref = _engine(gpu, form), _engine(gpu, form, rows=True), _engine(gpu, form, rows=True)
    for e in (a, b):
        for f, d, prof, ns, has_k, psi in _axes(e):
            prof[prof[:, 3] < 0, :3] = 1.0, 0.5, 0.25
            _set(e, f, d, prof, ns, has_k, psi)
    for e in (a, b, ref):
        e.steps(5)
    _same(b, ref, form)
    _same(a, ref, form)


@pytest.mark.parametrize("plain", [0, 1, 2])
@pytest.mark.parametrize("form", FORMS)
def test_kappa_is_skipped_on_an_axis_given_without(gpu, form, plain):
    a, b = _engine(gpu, form), _engine(gpu, form, rows=True)
    for e in (a, b):
        for f, d, prof, ns, has_k, psi in _axes(e):
            assert has_k
            if d == plain:
                _set(e, f, d, prof, ns, False, psi)
        e.steps(5)
    _same(a, b, (form, plain))
