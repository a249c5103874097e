"""Host buffers that go through the pinned staging slots (GPU), at its edges: just below and at
the size from which transfers are staged (4 MiB), whole slots (2 MiB) and a few bytes more,
fewer and more chunks than slots. Staging only moves bytes, so the result equals that of the
same call on device memory."""

import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# 24 bytes a pixel: 4 MiB - 16, 4 MiB + 32, 6 MiB, 12 MiB, 14 MiB + 16, 37 MiB
@pytest.mark.parametrize("w,h", [(3, 58254), (4, 43691), (512, 512), (1024, 512), (30, 20389), (1271, 1273)])
@pytest.mark.parametrize("pinned", [False, True])
def test_staged_copies_move_every_byte(ctx, w, h, pinned):
    import torch
    from luz_amd import renderer
    rng = np.random.default_rng(w)
    host = torch.from_numpy(rng.random((h, w, 3)))
    out = torch.empty_like(host)
    if pinned:
        host, out = host.pin_memory(), torch.empty(host.shape, dtype=host.dtype, pin_memory=True)
    ps = renderer._post_settings({"exposure": 0.5, "contrast": 1.0, "bloom": False, "view_transform": "agx"})
    dev = host.to("cuda:0")
    ref = torch.empty_like(dev)
    torch.cuda.synchronize()
    run = lambda a, b, device: renderer._lib.check(
        ctx._lib.luzgpu_postprocess(ctx.handle, ctypes.byref(ps), w, h, a.data_ptr(), b.data_ptr(), device))
    run(dev, ref, 1)
    for _ in range(2):  # the slots are used again
        out.fill_(-1.0)
        run(host, out, 0)
        assert torch.equal(out, ref.cpu())
