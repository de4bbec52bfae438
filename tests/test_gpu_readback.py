"""Readbacks through the page-locked chunks and buffers made from blocks that
earlier objects let go.

A readback above 768 KiB is cut into chunks of a quarter of its size, at
least 512 KiB and at most 1 MiB, in a ring of four: the sizes below lie on both
sides of one chunk, of several, and of the ring's wrap-around.  Bytes come back unchanged,
so every comparison is exact."""
import threading

import numpy as np
import pytest

from fauxgl_amd import api as A
from fauxgl_amd import meshes as M

pytestmark = pytest.mark.gpu


def _say(name):
    print(f"[case] {name}", flush=True)


def _pattern(w, h, seed):
    return np.random.default_rng(seed).integers(0, 256, (h, w, 4), dtype=np.uint8)


@pytest.mark.parametrize("w,h", [(1, 1), (131072, 1), (131073, 1), (131071, 1), (512, 384), (513, 384), (512, 512), (1023, 769),
                                 (1024, 1024), (1025, 1024), (2049, 512), (3000, 1777)])
def test_image_round_trip(w, h):
    _say(f"image {w}x{h}")
    ctx = A.NewContext(w, h)
    img = _pattern(w, h, w + h)
    ctx.SetColorBuffer(img)
    assert np.array_equal(ctx.Image(), img)
    ctx.close()


def test_readbacks_from_several_threads():
    _say("six threads, each its own context")
    bad = []

    def work(k):
        w, h = 700 + 131 * k, 500 + 67 * k
        ctx = A.NewContext(w, h)
        for it in range(4):
            img = _pattern(w, h, 10 * k + it)
            ctx.SetColorBuffer(img)
            if not np.array_equal(ctx.Image(), img):
                bad.append((k, it))
        ctx.close()

    ts = [threading.Thread(target=work, args=(k,)) for k in range(6)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not bad


def _frame(w, h, ntri, seed):
    ctx = A.NewContext(w, h)
    mesh = A.DeviceMesh(ctx, M.noise_sphere_mesh(ntri=ntri, detail=5, amplitude=0.15, seed=seed))
    mesh.SmoothNormalsThreshold(0.5)
    ctx.ClearColorBufferWith(M.BACKGROUND)
    ctx.Shader = M.phong_shader(w, h)
    ctx.DrawMesh(mesh)
    out = ctx.Image(), ctx.DepthImage(), ctx.EncodePNG()
    fresh = A.NewContext(w, h)
    blank = fresh.Image()
    fresh.close()
    mesh.close()
    ctx.close()
    return out, blank


def test_reused_blocks_give_the_same_frames():
    """The same frames before and after other work has left its data in the
    blocks; a new context's image is zero all the same."""
    sizes = [(320, 240, 6000, 1), (1000, 700, 20000, 2), (97, 33, 300, 3)]
    first = []
    for s in sizes:
        _say(f"first {s}")
        first.append(_frame(*s)[0])
    for rep in range(2):
        for s, want in zip(reversed(sizes), reversed(first)):
            _say(f"again {s}")
            got, blank = _frame(*s)
            assert not blank.any()
            assert np.array_equal(got[0], want[0])
            assert np.array_equal(got[1], want[1])
            assert got[2] == want[2]


def test_more_blocks_than_are_kept():
    """More contexts let go at once than the kept blocks' bound holds."""
    _say("40 contexts of 2560x1440")
    ctxs = [A.NewContext(2560, 1440) for _ in range(40)]
    img = _pattern(2560, 1440, 5)
    for c in ctxs:
        c.close()
    again = [A.NewContext(2560, 1440) for _ in range(3)]
    for c in again:
        assert not c.Image().any()
        c.SetColorBuffer(img)
    for c in again:
        assert np.array_equal(c.Image(), img)
        c.close()
