"""Textures with and without a texel of alpha 0, which decides whether a draw
may test its fragments before shading them: the host looks for it up to 262,144
texels, the device above, four or two texels a load with the rest one by one."""
import numpy as np
import pytest

from fauxgl_amd import api as A


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["NRGBA", "RGBA", "RGBA16"])
@pytest.mark.parametrize("w,h", [(1, 1), (13, 11), (512, 512), (512, 513), (523, 521), (1023, 1025)])
def test_holes(kind, w, h):
    print(f"[case] texture holes {kind} {w}x{h}", flush=True)
    ctx = A.NewContext(16, 16)
    tri = A.Prims(np.array([[[-1.0, -1, 0], [1, -1, 0], [0, 1, 0]]]), None, np.zeros((1, 3, 2)))
    n = w * h
    for hole in [None] + sorted({0, n // 2, max(n - 3, 0), max(n - 2, 0), n - 1}):
        t = np.zeros((n, 4), np.uint16 if kind == "RGBA16" else np.uint8)
        t[:, 3] = 1  # the least that is none
        if hole is not None:
            t[hole] = [9, 9, 9, 0]
        ctx.Shader = A.NewTextureShader(A.Identity(), A.NewImageTexture(t.reshape(h, w, 4), kind))
        ctx.DrawTriangles(tri)
        assert ctx.DepthFirst() == (hole is None), hole
