"""Device memory a context keeps for its next call (the grid freed last, the
workspace) goes back when an allocation of the context needs it: on a device
with 800 MB free beside some 520 MB kept, a grid of 1150 MB still fits."""

import numpy as np
import pytest
import torch

from mechafm_amd import abi

pytestmark = pytest.mark.gpu

KEPT, FREE, NEW = 11_000_000, 800_000_000, 24_000_000      # points of 48 bytes; bytes; points


def _upload(ctx, points):
    return ctx.grid_upload((points, 1, 1), np.eye(3), np.zeros(3), np.zeros((points, 4)), False)


@pytest.mark.parametrize("kept", ["grid", "workspace", "none"])
def test_kept_memory_is_given_back(kept):
    ctx = abi.Context(0)
    hold = []
    try:
        if kept == "grid":
            ctx.grid_free(_upload(ctx, KEPT))
        elif kept == "workspace":
            ctx.fft3d(np.zeros((320, 320, 320), dtype=np.complex128))
        torch.cuda.empty_cache()
        for _ in range(4):         # the first block leaves more than the device had reported
            free, _ = torch.cuda.mem_get_info()
            if free > FREE + (32 << 20):
                hold.append(torch.empty(free - FREE, dtype=torch.uint8, device="cuda"))
        if kept == "none":         # what does not fit is still refused, and the context goes on
            with pytest.raises(abi.MafmError):
                _upload(ctx, NEW)
            ctx.grid_free(_upload(ctx, 1000))
        else:
            ctx.grid_free(_upload(ctx, NEW))
    finally:
        hold.clear()
        torch.cuda.empty_cache()
        ctx.close()
