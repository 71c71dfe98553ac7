"""The ring and threads for large results are set up by the transfer that pays for
them: not for a context's one result of a few MB, and once 32 MB have gone.
The data come back byte for byte on both sides of that."""
import os

import numpy as np
import pytest

from mechafm_amd import abi

pytestmark = pytest.mark.gpu

MB = 32768            # points of 32 bytes in a MiB


def _threads():
    return len(os.listdir("/proc/self/task"))


def _download(ctx, mib):
    fe = np.random.default_rng(mib).normal(size=(mib * MB, 1, 1, 4))
    h = ctx.grid_upload((mib * MB, 1, 1), np.eye(3), np.zeros(3), fe, False)
    before = _threads()
    got = ctx.grid_download(h, (mib * MB, 1, 1))
    started = _threads() - before
    assert got.tobytes() == fe.tobytes()
    ctx.grid_free(h)
    return started


@pytest.mark.parametrize("sizes,started", [([8, 8, 8, 8], [0, 0, 0, 5]), ([31, 1, 3, 31], [0, 0, 0, 5]), ([33, 8], [5, 0])])
def test_ring_is_set_up_when_it_pays(gpu_ctx, sizes, started):
    ctx = abi.Context(0)
    _download(ctx, 1)
    before = _threads()
    assert [_download(ctx, m) for m in sizes] == started
    ctx.close()
    assert _threads() <= before
