"""Coverage spans of triangles that cross many tiles, and groups of pairs at
their edges, bit for bit against the oracle: rows that start tiles to the
left of where they are drawn, slivers whose run ends before the tile, runs
one pixel long, 63 to 129 pairs in one tile (a group is 64), and, past 2048
groups, many small triangles with a few wide ones among them (each wave then
walks its own group).  Solid, Phong and vertex-colored shading read the spans;
nothing is within a tolerance."""
import numpy as np
import pytest

from fauxgl_amd import api as A
from fauxgl_amd import meshes as M
from helpers import compare, run_gpu, run_oracle
from test_gpu_tiny_triangles import SHADER, _say, tiny


def _wide(n, seed, W, snap):
    """Slivers: x extents up to the whole screen, heights from a fraction of
    a pixel up, edges near horizontal."""
    rng = np.random.Generator(np.random.PCG64(seed))
    x = np.sort(rng.uniform(0, W, size=(n, 3)), axis=1)
    y = rng.uniform(0, W, size=(n, 1)) + rng.uniform(-1, 1, size=(n, 3)) * rng.choice([0.4, 3.0, 40.0], size=(n, 1))
    xy = np.stack([x, np.clip(y, 0, W)], axis=2)
    if snap:
        xy = np.round(xy * 2) / 2
    pos = np.empty((n, 3, 3))
    pos[..., :2] = xy / (W / 2) - 1
    pos[..., 2] = rng.uniform(-0.9, 0.9, size=(n, 3))
    col = np.ones((n, 3, 4))
    col[..., :3] = rng.uniform(0, 1, size=(n, 3, 3))
    return A.Prims(pos, M.with_face_normals(pos), None, col)


CASES = {
    "wide": (256, lambda: _wide(400, 1, 256, False)),
    "wide, on pixel centers": (256, lambda: _wide(400, 2, 256, True)),
    "wide, odd size": (301, lambda: _wide(300, 3, 301, False)),
    "63 pairs": (32, lambda: _wide(63, 4, 32, False)),
    "64 pairs": (32, lambda: _wide(64, 5, 32, False)),
    "65 pairs": (32, lambda: _wide(65, 6, 32, False)),
    "129 pairs": (32, lambda: _wide(129, 7, 32, False)),
    "many small, some wide": (512, lambda: M.concat(tiny(170000, 8, 512, 2.0, 6.0), _wide(200, 9, 512, False))),
}


@pytest.mark.gpu
@pytest.mark.parametrize("name", list(CASES))
def test_wide_spans_match_the_oracle(name):
    _say(f"wide spans: {name}")
    W, make = CASES[name]
    prims = make()
    ops = [("clear_color", A.White), ("set", {"Cull": A.CullNone}), ("shader", SHADER), ("tris", prims)]
    got = run_gpu(W, W, ops)
    res = compare(run_oracle(W, W, ops), got, color_tol=0)
    assert res["ok"], res
    if name.startswith("many"):
        assert got[3].DrawStats()["pairs"] > 2048 * 64
