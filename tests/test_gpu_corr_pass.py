"""Source corrections in single passes against the same corrections as launches of their own, bit for bit: engines that do step by
single passes (asserted), every list of E-side corrections, D-form nodes among their targets, one and two passes of a pair
past the end of a source's table.
"""

import ctypes

import pytest
import torch

from tests import cases
from tests.test_gpu_corr import LISTS, E, _engine
from tests.test_zz_no_alloc import _bind

pytestmark = pytest.mark.gpu

E_LISTS = [q for q, ops in enumerate(LISTS) if all(phase == E for _, phase, _ in ops)]


@pytest.mark.parametrize("poles", [0, 1, 3])
@pytest.mark.parametrize("ops", E_LISTS)
def test_corrections_in_single_passes(gpu, ops, poles):
    from lightsmith_amd import _lib
    lib, ns = _lib.load(), cases.product_ns()
    noalloc = _bind(lib)
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    for shape in ((17, 12, 15), (66, 9, 11)):
        for calls in ((1, 4, 9), (2, 4, 9)):  # the tables hold 11 steps
            a, b = (_engine(ns, gpu, shape, LISTS[ops], poles=poles) for _ in range(2))
            for n in calls:
                a.steps(n)
                _lib.check(noalloc(b._h, n, stream), "lsf_step_noalloc")
            assert a._two_sets
            torch.cuda.synchronize()
            for q, (x, y) in enumerate(zip(a.state_tensors(), b.state_tensors())):
                assert torch.equal(x, y), (shape, calls, q)
            assert a.E_flat.abs().max() > 0


def test_the_lists_cover_the_kernel():
    """Several corrections of one node and more than a kernel makes are among the lists above."""
    assert {0, 3, 5} <= set(E_LISTS) and max(len(LISTS[q]) for q in E_LISTS) > 3
