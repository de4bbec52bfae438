"""The weight gradient's strips, bands and waves: frames whose sizes straddle
its 128-pixel strips, 32-pixel waves and 8-row bands, with a target that
equals the network's own output except on the rows and columns beside those
edges, so that a pixel lost or counted twice there changes the gradient by
far more than the tolerance.  The tolerance is the BF16 one of the gradient
test: 2e-2 relative L2 per layer against the FP32 reference that rounds
where the GPU rounds."""
import numpy as np
import pytest

import nn_ref as R
from fauxgl_amd import api as A
from fauxgl_amd import nnaa
from test_gpu_nn import _say, frame_ctx, rand_params, random_frame


@pytest.mark.gpu
@pytest.mark.parametrize("h,w", [(9, 131), (17, 257), (70, 129), (40, 1), (1, 300), (24, 96)])
def test_gradient_at_strip_and_band_edges(h, w):
    _say(f"nn dw {w}x{h}")
    color, depth = random_frame(h, w, h * 1000 + w)
    src = frame_ctx(color, depth)
    tgt = A.NewContext(w, h)
    net = nnaa.Network(src, seed=1)
    p = rand_params(h + w)
    net.SetParams(p)
    net.Infer(src, tgt)
    target = tgt.Image()
    cols = [c for c in (0, 31, 32, 63, 64, 95, 126, 127, 128, 129, 255, 256, w - 1) if c < w]
    rows = [r for r in (0, 7, 8, 15, 16, h - 1) if r < h]
    rng = np.random.Generator(np.random.PCG64(3))
    noise = rng.integers(0, 256, target.shape, dtype=np.uint8)
    on = np.zeros((h, w), bool)
    on[np.ix_(rows, cols)] = True
    target[on] = noise[on]
    tgt.SetColorBuffer(target)
    loss, g = net.Grad(src, tgt)
    rloss, rg = R.loss_and_grad(p, color, depth, target)
    assert abs(loss - rloss) <= 1e-3 * abs(rloss), (loss, rloss)
    for li, (ci, co, wo, bo) in enumerate(nnaa.layer_offsets()[0]):
        for name, a, b in (("w", wo, wo + 9 * ci * co), ("b", bo, bo + co)):
            nrm = np.linalg.norm(rg[a:b])
            rel = np.linalg.norm(g[a:b] - rg[a:b]) / nrm if nrm else np.abs(g[a:b]).max()
            print(li, name, rel)
            assert rel <= 2e-2, (li, name, rel)
