"""Configuration calls while a chunk graph is captured: replays after the next step follow the new configuration, against an
engine that steps eagerly, bit for bit. Engines whose graphs name library memory that such a call makes anew: joined
sub-engines, operations that share a launch, corrections made in the bulk kernels, single passes.
"""

import ctypes

import numpy as np
import pytest
import torch

from tests import cases
from tests.test_gpu_corr import LISTS
from tests.test_gpu_corr import _engine as _corrected
from tests.test_gpu_joined import _engine as _joined
from tests.test_gpu_stages import KHATS, _lines

pytestmark = pytest.mark.gpu

MAKE = {"joined": lambda gpu: _joined(gpu, (), True, (1, 4, 64, 4)),
        "lines": lambda gpu: _lines(gpu, KHATS),
        "corrections": lambda gpu: _corrected(cases.product_ns(), gpu, (17, 12, 15), LISTS[1], fused=False),
        "pass": lambda gpu: _corrected(cases.product_ns(), gpu, (17, 12, 15), LISTS[3], poles=2),
        "periodic": lambda gpu: _corrected(cases.product_ns(), gpu, (17, 12, 15), LISTS[1], periodic=(True, True, False), bloch=True)}


def _material(e, on, seed):
    """A new material for the engine `on` (D-form nodes keep theirs), kept by e."""
    from lightsmith_amd import _lib
    cb = on.cdx / torch.rand(3 * on.N, generator=torch.Generator().manual_seed(seed)).add(1.0)
    if on.n_ade:
        cb[torch.as_tensor(on.ade_nodes)] = -(torch.as_tensor(on.ade_medium).to(cb.dtype) + 1)
    e._keep.append(cb.to(on.E_flat.device))
    _lib.check(on.lib.lsf_set_material_dense(on._h, _lib.ptr(e._keep[-1])), "lsf_set_material_dense")


@pytest.mark.parametrize("which", MAKE)
def test_replays_follow_the_configuration(gpu, which):
    from lightsmith_amd import _lib
    a, b = (MAKE[which](gpu) for _ in range(2))
    a.steps(1)
    b.steps(1)
    lib, side = a.lib, torch.cuda.Stream(device=gpu)
    torch.cuda.synchronize()
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    _lib.check(lib.lsf_graph_capture(a._h, 5, ctypes.c_void_p(side.cuda_stream)), "lsf_graph_capture")
    for change in range(3):
        _lib.check(lib.lsf_graph_replay(a._h, 2, stream), "lsf_graph_replay")
        b.steps(10)
        for e in (a, b):
            for on in [e] + (e._subs if change == 1 else []):
                _material(e, on, change)
            e.steps(3)
        # memory that the change gave back is someone else's now
        junk = [torch.full((n,), 0x7f, dtype=torch.uint8, device=gpu) for n in (1 << 12, 1 << 16, 1 << 20)]
        _lib.check(lib.lsf_graph_replay(a._h, 2, stream), "lsf_graph_replay")
        b.steps(10)
        torch.cuda.synchronize()
        del junk
        for q, (x, y) in enumerate(zip(a.state_tensors(), b.state_tensors())):
            assert torch.equal(x, y), (change, q)
    assert a.E_flat.abs().max() > 0 and torch.isfinite(a.E_flat.abs()).all()
    _lib.check(lib.lsf_graph_reset(a._h), "lsf_graph_reset")


def test_a_sub_engine_stepped_or_planned_by_itself(gpu):
    """A sub-engine that is configured and then stepped directly, or whose engine joins a batch, before its engine goes on."""
    from lightsmith_amd import _lib
    from lightsmith_amd.fdtd.batch import Batch
    a, b = (_joined(gpu, (), True, t) for t in ((1, 4, 64, 4), (2, 4, 64, 4)))
    side = torch.cuda.Stream(device=gpu)
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    for e in (a, b):
        for sub in e._subs:
            sub.add_modal(3, "E", sub.native_index([cases.product_ns().flat_index(0, 1, 1, 9, sub.shape)]), [[0.3]], np.ones((99, 1)))
        e.steps(2)
    torch.cuda.synchronize()
    _lib.check(a.lib.lsf_graph_capture(a._h, 3, ctypes.c_void_p(side.cuda_stream)), "lsf_graph_capture")
    for n in range(2):
        for e in (a, b):
            _material(e, e._subs[n], n)
            if n == 0:
                e._subs[0].steps(1)
            else:
                Batch([e], schedule=(1, 4, 64, 4, 0)).close()
            if n == 0 or e is b:
                e.steps(3)
        if n == 1:
            _lib.check(a.lib.lsf_graph_replay(a._h, 1, stream), "lsf_graph_replay")
        _lib.check(a.lib.lsf_graph_replay(a._h, 2, stream), "lsf_graph_replay")
        b.steps(6)
        torch.cuda.synchronize()
        for q, (x, y) in enumerate(zip(a.state_tensors(), b.state_tensors())):
            assert torch.equal(x, y), (n, q)
    assert a._subs[0].E_flat.abs().max() > 0 and torch.isfinite(a.E_flat.abs()).all()
    _lib.check(a.lib.lsf_graph_reset(a._h), "lsf_graph_reset")
