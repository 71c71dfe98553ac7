"""Large results into pageable arrays: what a grid was loaded with comes back
byte for byte, below and at the size where the pinned ring takes over, at whole
and odd numbers of ring slots and of turns round the ring, into pinned memory,
from several threads at once, and in a grid that takes a freed grid's memory."""
import threading

import numpy as np
import pytest
import torch

from mechafm_amd import abi

pytestmark = pytest.mark.gpu

SLOT = 65536          # points of 32 bytes in a slot of 2 MiB


def _round_trip(ctx, points, seed, out=None):
    fe = np.random.default_rng(seed).normal(size=(points, 1, 1, 4))
    h = ctx.grid_upload((points, 1, 1), np.eye(3), np.zeros(3), fe, False)
    try:
        got = ctx.grid_download(h, (points, 1, 1))
        assert got.tobytes() == fe.tobytes()
        if out is not None:
            ctx.check(abi.lib().mafm_grid_download(ctx.h, h, abi._dp(out)))
            assert out.tobytes() == fe.tobytes()
    finally:
        ctx.grid_free(h)


@pytest.mark.parametrize("points", [1, 2 * SLOT - 1, 2 * SLOT, 2 * SLOT + 1, 3 * SLOT, 8 * SLOT, 8 * SLOT + 1,
                                    9 * SLOT - 1, 20 * SLOT + 7])
def test_what_goes_up_comes_down(gpu_ctx, points):
    for seed in range(2):
        _round_trip(gpu_ctx, points, seed)


def test_pinned_memory_is_filled_directly(gpu_ctx):
    out = torch.empty(5 * SLOT + 3, 1, 1, 4, dtype=torch.float64, pin_memory=True).numpy()
    _round_trip(gpu_ctx, 5 * SLOT + 3, 5, out)


def test_contexts_on_threads(gpu_ctx):
    errors = []

    def work(seed):
        try:
            ctx = abi.Context(0)
            for k in range(3):
                _round_trip(ctx, (9 + seed) * SLOT + 11 * k, 10 * seed + k)
            ctx.close()
        except Exception as e:   # noqa: BLE001 -- reported below
            errors.append(e)

    threads = [threading.Thread(target=work, args=(s,)) for s in range(3)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors, errors
