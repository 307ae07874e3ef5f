"""The second buffer set of single-pass stepping: who is given one, what is refused with it, and a GPU without room for it."""

import ctypes
import gc

import numpy as np
import pytest
import torch

from tests import cases
from tests.test_zz_no_alloc import _bind

pytestmark = pytest.mark.gpu


def _box(gpu, shape=(24, 20, 18), dx=2.0, tiling=None, **kw):
    ns = cases.product_ns()
    d = np.broadcast_to(dx, 3)
    old = ns.Engine.tiling
    ns.Engine.tiling = tiling or old
    try:
        e = cases.make(ns, gpu, shape=shape, dx=dx, dt=0.9 / np.sqrt(sum(1 / v ** 2 for v in d)),
                       inv_eps=np.full((3,) + shape, 1 / 2.25), pml=ns.PMLSpec(cells=((3, 3),) * 3), **kw)
    finally:
        ns.Engine.tiling = old
    cases.random_fields(e, 2)
    return e


@pytest.mark.parametrize("dx,tiling,refused", [(2.0, None, True), ((2.0, 1.5, 3.0), None, True), (2.0, (1, 8, 64, 8), True),
                                               (2.0, (2, 4, 64, 8), False), (2.0, (1, 4, 32, 8), False)])
def test_no_alloc_steps_refuse_what_was_asked_to_step_in_single_passes(gpu, dx, tiling, refused):
    """fused=True on one-row tiles of 64 cells; other tiles, and engines that were not asked, are stepped."""
    from lightsmith_amd import _lib
    lib = _lib.load()
    noalloc = _bind(lib)
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    for fused in (True, None):
        a, b = (_box(gpu, dx=dx, tiling=tiling, fused=f) for f in (fused, False))
        rc = noalloc(a._h, 3, stream)
        if fused and refused:
            assert rc == _lib.LSF_EINVAL and b"single-pass" in lib.lsf_last_error()
            a.steps(3)
        else:
            assert rc == 0
        b.steps(3)
        torch.cuda.synchronize()
        for x, y in zip(a.state_tensors(), b.state_tensors()):
            assert torch.equal(x, y)


def test_chunk_offsets_past_four_gigabytes_do_not_step_in_single_passes(gpu):
    """D-form nodes on a grid a few cells wide: 24 bytes a chunk of 32 cells and row pass 2^32 before a component does. (Only asked:
    the handle's arrays are never used.)"""
    from lightsmith_amd import _lib
    lib = _lib.load()
    word = torch.zeros(64, dtype=torch.float32, device=gpu)
    media = torch.tensor([1.0, 1.0, 0.5, 0.1, 0.2], device=gpu)
    for shape, ok in (((3, 15000, 13000), 0), ((3, 9000, 13000), 2), ((40, 4000, 4000), 2)):
        g = _lib.LsfGrid()
        g.shape[:], g.spacing[:], g.dt, g.tick = shape, (2.0,) * 3, 1.0, 1
        g.dev_E = g.dev_H = g.dev_counter = word.data_ptr()
        h = ctypes.c_void_p()
        _lib.check(lib.lsf_create(ctypes.byref(g), ctypes.byref(h)), "lsf_create")
        _lib.check(lib.lsf_set_material_dense(h, _lib.ptr(word)), "lsf_set_material_dense")
        _lib.check(lib.lsf_set_tiling(h, 1, 4, 64, 8), "lsf_set_tiling")
        assert lib.lsf_can_pair(h) == 2
        _lib.check(lib.lsf_set_ade(h, _lib.ptr(word), _lib.ptr(word), 10, 1, _lib.ptr(media), 1), "lsf_set_ade")
        assert lib.lsf_can_pair(h) == ok, shape
        lib.lsf_destroy(h)


def test_without_room_the_second_set_leaves_nothing_behind(gpu):
    """Where not all of it fits, the engine steps with two kernels and holds no part of it, and one that asked for it raises."""
    a, b = _box(gpu, shape=(260, 256, 256)), _box(gpu, shape=(260, 256, 256), fused=False)
    torch.cuda.synchronize()
    gc.collect()
    torch.cuda.empty_cache()
    held = torch.cuda.memory_reserved(gpu)
    total = torch.cuda.get_device_properties(gpu).total_memory
    torch.cuda.set_per_process_memory_fraction(held / total, gpu)
    kept = []  # reserved memory that would do
    try:
        while True:
            kept.append(torch.empty(2 * a.E_flat.numel(), device=gpu))
    except torch.cuda.OutOfMemoryError:
        held = torch.cuda.memory_reserved(gpu)
    torch.cuda.set_per_process_memory_fraction((held + 1.5 * 4 * a.E_flat.numel()) / total, gpu)  # room for one field of two
    try:
        a.steps(2)
        b.steps(2)
        assert not a._two_sets and torch.cuda.memory_reserved(gpu) == held
        with pytest.raises(torch.cuda.OutOfMemoryError):
            _box(gpu, shape=(260, 256, 256), fused=True)
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0, gpu)
    torch.cuda.synchronize()
    for x, y in zip(a.state_tensors(), b.state_tensors()):
        assert torch.equal(x, y)
