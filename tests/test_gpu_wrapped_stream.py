"""Replays on a stream that torch only wraps, which is gone before the next replay on another one, against eager chunks, bit for
bit; and which streams count as such."""

import ctypes
import re

import pytest
import torch

from tests import cases

pytestmark = pytest.mark.gpu


def _hip():
    with open("/proc/self/maps") as f:
        return ctypes.CDLL(re.search(r"\S*libamdhip64\.so\S*", f.read())[0])


@pytest.mark.parametrize("batched", [False, True])
def test_replays_from_streams_that_are_gone(gpu, batched):
    from lightsmith_amd.fdtd.batch import Batch
    hip, ns = _hip(), cases.product_ns()
    make = lambda: cases.dispersive_box(ns, gpu, shape=(40, 36, 32), n_steps_hint=200)  # noqa: E731
    a, b = make(), make()
    owner = Batch([a]) if batched else a
    run, used = owner.make_runner(True)
    assert used
    run()  # the eager chunk, then capture
    torch.cuda.synchronize()
    for q in range(6):
        if q % 3 == 2:
            run()
            continue
        s = ctypes.c_void_p()
        assert hip.hipStreamCreate(ctypes.byref(s)) == 0
        with torch.cuda.stream(torch.cuda.ExternalStream(s.value, device=gpu)):
            run()
        assert hip.hipStreamDestroy(s) == 0
    torch.cuda.synchronize()
    for _ in range(7):
        b.chunk()
    torch.cuda.synchronize()
    for x, y in zip(a.state_tensors(), b.state_tensors()):
        assert torch.equal(x, y)
    owner.release()
    if batched:
        owner.close()


def test_only_wrapped_streams_keep_an_event(gpu):
    from lightsmith_amd.fdtd.engine import CallerStream
    hip = _hip()
    s = ctypes.c_void_p()
    assert hip.hipStreamCreate(ctypes.byref(s)) == 0
    caller = CallerStream(torch.device(gpu))
    for stream, kept in ((torch.cuda.default_stream(gpu), False), (torch.cuda.Stream(device=gpu), False),
                         (torch.cuda.ExternalStream(s.value, device=gpu), True), (torch.cuda.default_stream(gpu), False)):
        with torch.cuda.stream(stream):
            assert caller.begin().value in (stream.cuda_stream, None)
            caller.end()
        assert (caller._event is not None) == kept
    torch.cuda.synchronize()
    assert hip.hipStreamDestroy(s) == 0
