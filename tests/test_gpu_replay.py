"""Chunk graphs replay on the caller's stream: runs that move between streams (no other synchronisation) against eager chunks,
bit for bit, alone and in a batch."""

import pytest
import torch

from tests import cases

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("batched", [False, True])
def test_replays_from_several_streams(gpu, batched):
    from lightsmith_amd.fdtd.batch import Batch
    ns = cases.product_ns()
    make = lambda: cases.dispersive_box(ns, gpu, shape=(40, 36, 32), n_steps_hint=200)  # noqa: E731
    a, b = make(), make()
    owner = Batch([a]) if batched else a
    run, used = owner.make_runner(True)
    assert used
    streams = [torch.cuda.Stream(device=gpu) for _ in range(2)] + [torch.cuda.current_stream()]
    run()  # the eager chunk, then capture
    torch.cuda.synchronize()
    for q in range(9):
        with torch.cuda.stream(streams[q % 3]):
            run()
    torch.cuda.synchronize()
    for _ in range(10):
        b.chunk()
    torch.cuda.synchronize()
    for x, y in zip(a.state_tensors(), b.state_tensors()):
        assert torch.equal(x, y)
    owner.release()
    if batched:
        owner.close()
