"""DepthImage at the edges of its vector loads: sizes around two and four
pixels a thread and around the unrolled loop, written to device buffers that
start at any pixel of a larger one (8-byte stores only where they are
aligned), against the definition (context.go:87-117) in float64: equal."""
import ctypes

import numpy as np
import pytest
import torch

from fauxgl_amd import _native as N
from fauxgl_amd import api as A


def _gray(depth):
    drawn = depth != A.MaxFloat64
    lo, hi = (depth[drawn].min(), depth[drawn].max()) if drawn.any() else (A.MaxFloat64, -A.MaxFloat64)
    with np.errstate(all="ignore"):
        t = np.where(drawn, (depth - lo) / (hi - lo), 1.0)
    v = t * 65535.0
    return np.where(np.isfinite(v), v, 0).astype(np.int64).astype(np.uint16)


@pytest.mark.gpu
@pytest.mark.parametrize("w,h", [(1, 1), (3, 1), (2, 2), (5, 1), (7, 9), (255, 3), (641, 479), (2050, 1029)])
def test_depth_image_sizes_and_offsets(w, h):
    print(f"[case] depth image {w}x{h}", flush=True)
    rng = np.random.Generator(np.random.PCG64(w * 10007 + h))
    depth = rng.uniform(-0.5, 0.9, (h, w))
    depth[rng.uniform(size=(h, w)) < 0.3] = A.MaxFloat64
    if w > 2:
        depth[0, :3] = [0.25, -0.0, 0.0]
    ctx = A.NewContext(w, h)
    ctx.SetDepthBuffer(depth)
    want = _gray(depth)
    np.testing.assert_array_equal(ctx.DepthImage(), want)
    buf = torch.zeros(w * h + 8, dtype=torch.int16, device="cuda")
    for off in range(4):
        buf.fill_(0x5a5a)
        torch.cuda.synchronize()
        N.check(N.load().fgl_depth_image_noalloc_async(ctx._ptr(), ctypes.c_void_p(buf.data_ptr() + 2 * off)), ctx._ptr())
        ctx.Sync()
        got = buf.cpu().numpy().view(np.uint16)
        np.testing.assert_array_equal(got[off:off + w * h].reshape(h, w), want)
        assert (got[:off] == 0x5a5a).all() and (got[off + w * h:] == 0x5a5a).all()
