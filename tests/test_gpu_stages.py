"""Per-step operations that share a launch against one launch each (lsf_step against lsf_step_noalloc, which launches every
operation by itself), bit for bit: the adjoint's source, gradient and D-form restore, also where the gradient's nodes are
D-form nodes (then it has to wait for the restore), and the 1D lines of several TFSF sources of odd lengths; and engines
of one batch, whose operations share launches across members, against the same engines alone.
"""

import ctypes

import numpy as np
import pytest
import torch

from tests import cases

pytestmark = pytest.mark.gpu


def _twins(lib, a, b, n):
    from lightsmith_amd import _lib
    from tests.test_zz_no_alloc import _bind
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    _lib.check(lib.lsf_step(a._h, n, stream), "lsf_step")
    _lib.check(_bind(lib)(b._h, n, stream), "lsf_step_noalloc")


def _adjoint(gpu, case, overlap=False, seed=5):
    p = cases.adjoint_problem(case, gpu)
    rng = np.random.default_rng(seed)
    p.forward(torch.as_tensor(case["rho"]))
    p.release_graphs()
    if overlap:  # a second gradient, over the D-form nodes themselves
        from lightsmith_amd import _lib
        f = p.fwd
        p._g2 = torch.zeros(f.n_ade, dtype=torch.float64, device=p._dev)
        p._tape2 = torch.rand(f.n_ade * 4, generator=torch.Generator().manual_seed(1)).to(p._dev)
        p._base2 = torch.full((1,), p.n_steps - 4, dtype=torch.int64, device=p._dev)
        p._cb2 = torch.ones(f.n_ade, dtype=torch.float32, device=p._dev)
        _lib.check(f.lib.lsf_add_adjoint_gradient(p.adj._h, f.n_ade, _lib.ptr(p._ade_nodes), _lib.ptr(p._cb2),
                                                  _lib.ptr(p._tape2), 4, _lib.ptr(p._base2), p.n_steps,
                                                  _lib.ptr(p._g2)), "lsf_add_adjoint_gradient")
    g = lambda t: torch.complex(torch.as_tensor(rng.standard_normal(t.shape)),  # noqa: E731
                                torch.as_tensor(rng.standard_normal(t.shape))).to(t)
    p.begin_backward(g(p.monitor.acc_e), g(p.monitor.acc_h) if p.monitor.acc_h is not None else None)
    p.base.fill_(0)
    return p


@pytest.mark.parametrize("ade,overlap", [(False, False), (True, False), (True, True)])
def test_adjoint_operations_sharing_launches(gpu, ade, overlap):
    case = cases.adjoint_case(steps=40, stride=8, **({"ade": True} if ade else {}))
    a, b = (_adjoint(gpu, case, overlap) for _ in range(2))
    for n in (1, 9, 23):
        _twins(a.fwd.lib, a.adj, b.adj, n)
    torch.cuda.synchronize()
    outs = [p.adj.state_tensors() + [p.g] + ([p._g2] if overlap else []) for p in (a, b)]
    for q, (x, y) in enumerate(zip(*outs)):
        assert torch.equal(x, y), q
    assert a.g.abs().max() > 0 and (not overlap or a._g2.abs().max() > 0)


def _lines(gpu, khats):
    ns = cases.product_ns()
    shape = (30, 28, 34)
    src = [ns.TFSFPlaneWave(shape=shape, origin=np.zeros(3), dx=1.0, dt=0.95 / np.sqrt(3), r0=np.array([15.0, 14, 17]),
                            lo=np.array([9, 8, 10]) + q, hi=np.array([21, 20, 24]) - q, khat=k, ehat=e, eps_b=1.77,
                            omega_c=0.6, omega_half=0.2, max_steps=100) for q, (k, e) in enumerate(khats)]
    return cases.make(ns, gpu, shape=shape, dx=1.0, dt=0.95 / np.sqrt(3), inv_eps=np.full((3,) + shape, 1 / 1.77),
                      pml=ns.PMLSpec(cells=((5, 5),) * 3, eps_ref=1.77), sources=src)


KHATS = [((0, 0, 1.0), (1.0, 0, 0)), ((1.0, 0, 0), (0, 1.0, 0)), ((0, -1.0, 0), (0, 0, 1.0))]


def test_lines_sharing_launches(gpu):
    a, b = (_lines(gpu, KHATS) for _ in range(2))
    for n in (1, 30, 29):
        _twins(a.lib, a, b, n)
    torch.cuda.synchronize()
    for x, y in zip(a.state_tensors(), b.state_tensors()):
        assert torch.equal(x, y)
    assert a.E_flat.abs().max() > 0


def test_batch_operations_sharing_launches(gpu):
    from lightsmith_amd.fdtd.batch import Batch
    plain, ade = (cases.adjoint_case(steps=40, stride=8, **kw) for kw in ({}, {"ade": True}))
    make = lambda: [_adjoint(gpu, plain), _adjoint(gpu, ade), _adjoint(gpu, ade, True, seed=6)]  # noqa: E731
    alone, mem = make(), make()
    lines = [[_lines(gpu, KHATS[:q]) for q in (1, 3)] for _ in range(2)]
    batch = Batch([p.adj for p in mem], schedule=(1, 4, 64, 8, 0))
    batch.steps(33)
    b2 = Batch(lines[0], schedule=(1, 4, 64, 8, 0))
    b2.steps(60)
    for p in alone:
        p.adj.set_tiling(1, 4, 64, 8)
        p.adj.steps(33)
    for e in lines[1]:
        e.steps(60)
    torch.cuda.synchronize()
    for p, m in zip(alone, mem):
        for x, y in zip(p.adj.state_tensors() + [p.g], m.adj.state_tensors() + [m.g]):
            assert torch.equal(x, y)
    for e, m in zip(lines[1], lines[0]):
        for x, y in zip(e.state_tensors(), m.state_tensors()):
            assert torch.equal(x, y)
    batch.close()
    b2.close()


def test_members_of_a_batch_that_share_a_gradient(gpu):
    """Adjoint engines whose gradients are added to one array, as for an objective over several runs of a design: the members'
    terms in their order, step by step, as one engine after another adds them."""
    from lightsmith_amd import _lib
    from lightsmith_amd.fdtd.batch import Batch
    case = cases.adjoint_case(steps=40, stride=8)
    make = lambda: [_adjoint(gpu, case, seed=s) for s in (5, 6, 7)]  # noqa: E731
    alone, mem = make(), make()
    shared = []
    for probs in (alone, mem):
        n = alone[0].n_nodes
        both = torch.zeros(2 * n, dtype=torch.float64, device=gpu)  # the third's gradient overlaps half of the others'
        for p, at in zip(probs, (0, 0, n // 2)):
            _lib.check(p.fwd.lib.lsf_add_adjoint_gradient(p.adj._h, n, _lib.ptr(p._nodes), _lib.ptr(p.cb_design), _lib.ptr(p.tape),
                                                          p.n_slots, _lib.ptr(p.base), p.n_steps, _lib.ptr(both[at:])),
                       "lsf_add_adjoint_gradient")
            p.adj.set_tiling(1, 4, 64, 8)
        shared.append(both)
    batch = Batch([p.adj for p in mem], schedule=(1, 4, 64, 8, 0))
    for _ in range(33):
        batch.steps(1)
        for p in alone:
            p.adj.steps(1)
    torch.cuda.synchronize()
    assert torch.equal(*shared) and shared[0].abs().max() > 0
    for p, m in zip(alone, mem):
        assert torch.equal(p.g, m.g)
    batch.close()
