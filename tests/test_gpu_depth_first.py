"""Draws whose fragments are depth-tested before they are shaded, bit for bit
against the oracle (color, depth, RasterizeInfo), over what selects and ends
that path: opaque and blending colors of every shader, textures with and
without a texel of alpha 0, color, depth write and depth test off, depth
biases, marked clears before and after; few tiles (more threads a tile), many,
and more than 2304 (the device decides by the fragments per pixel: the scenes
have either side of two); every tile shape; overlap deep enough that the queue
of blended survivors fills and wraps."""
import numpy as np
import pytest

from fauxgl_amd import api as A
from fauxgl_amd import meshes as M
from helpers import compare, oracle_shader
import oracle as O
from test_gpu_tiny_triangles import _say

MATRIX = A.Identity()


def _soup(n, seed, extent):
    """n triangles across the screen, each of the given extent (NDC)."""
    rng = np.random.Generator(np.random.PCG64(seed))
    c = rng.uniform(-1, 1, size=(n, 1, 3)) * [1, 1, 0.8]
    pos = np.clip(c + rng.uniform(-extent, extent, size=(n, 3, 3)) * [1, 1, 0.1], -1, 1)
    return A.Prims(pos, M.with_face_normals(pos), rng.uniform(0, 1, size=(n, 3, 2)))


def _texture(kind, hole):
    rng = np.random.Generator(np.random.PCG64(3))
    top = 65535 if kind == "RGBA16" else 255
    t = rng.integers(1, top + 1, size=(9, 13, 4))
    if hole:
        t[2:5, 3:9] = 0
    return A.NewImageTexture(t.astype(np.uint16 if kind == "RGBA16" else np.uint8), kind)


def _phong(alpha=1.0, tex=None):
    return A.PhongShader(MATRIX, A.V(0.2, 0.4, 1).Normalize(), A.V(0, 0, 3), A.Color(0.3, 0.6, 0.4, alpha), texture=tex)


SHADERS = {
    "solid": lambda: A.NewSolidColorShader(MATRIX, A.Color(0.2, 0.4, 0.6, 1.0)),
    "solid translucent": lambda: A.NewSolidColorShader(MATRIX, A.Color(0.2, 0.4, 0.6, 0.5)),
    "solid discard": lambda: A.NewSolidColorShader(MATRIX, A.Discard),
    "texture": lambda: A.NewTextureShader(MATRIX, _texture("NRGBA", False)),
    "texture with a hole": lambda: A.NewTextureShader(MATRIX, _texture("NRGBA", True)),
    "texture 16": lambda: A.NewTextureShader(MATRIX, _texture("RGBA16", False)),
    "phong": lambda: _phong(),
    "phong translucent": lambda: _phong(0.4),
    "phong textured": lambda: _phong(tex=_texture("RGBA", False)),
}
_FIELDS = {"ReadDepth": "read_depth", "WriteDepth": "write_depth", "WriteColor": "write_color",
           "AlphaBlend": "alpha_blend", "Wireframe": "wireframe", "Cull": "cull", "DepthBias": "depth_bias"}


def _check(name, shader, W, H, draws, states, tile=None, first=None):
    """Clears, then the draws each with its state, in both; a second frame on
    the same context follows with the clears pending again.  first(state):
    whether a draw is to be tested before it is shaded."""
    _say(f"depth first: {name}")
    octx, gctx = O.Context(W, H), A.NewContext(W, H)
    if tile:
        gctx.SetTileShape(*tile)
    osh = oracle_shader(shader)
    octx.set_shader(osh)
    gctx.Shader = shader
    for bg in (A.White, A.Color(0.1, 0.2, 0.3, 0.5)):
        ri, gi = [], []
        octx.clear_color(tuple(bg))
        octx.clear_depth(A.MaxFloat64)
        gctx.ClearColorBufferWith(bg)
        gctx.ClearDepthBuffer()
        for prims, st in zip(draws, states):
            full = {"ReadDepth": True, "WriteDepth": True, "WriteColor": True, "AlphaBlend": True, "Wireframe": False,
                    "Cull": A.CullNone, "DepthBias": 0.0, **st}
            octx.set_state(O.make_state(front_face=O.FACE_CCW, line_width=2.0,
                                        **{_FIELDS[k]: v for k, v in full.items()}))
            for k, v in full.items():
                setattr(gctx, k, v)
            m = O.Mesh(tris=prims.arrays())
            ri.append(octx.draw_triangles(m, 1))
            gi.append(tuple(gctx.DrawTriangles(prims)))
            if first is not None:
                assert gctx.DepthFirst() == first(full), full
        res = compare((octx.color(), octx.depth(), ri), (gctx.Image(), gctx.DepthBuffer, gi), color_tol=0)
        assert res["ok"], res
    return gctx


STATES = {
    "as it is": [{}, {}],
    "no blending": [{"AlphaBlend": False}, {}],
    "no color, then color": [{"WriteColor": False}, {}],
    "color, then no color": [{}, {"WriteColor": False}],
    "no depth write": [{"WriteDepth": False}, {}],
    "no depth test": [{"ReadDepth": False}, {"ReadDepth": False, "WriteDepth": False}],
    "biased": [{"DepthBias": 1e-2}, {"DepthBias": -1e-2}],
    "wireframe": [{}, {"Wireframe": True, "DepthBias": -1e-3}],
}


@pytest.mark.gpu
@pytest.mark.parametrize("state", list(STATES))
@pytest.mark.parametrize("shader", list(SHADERS))
def test_states_and_shaders(shader, state):
    draws = [_soup(60, 1, 0.7), _soup(60, 2, 0.3)]

    def first(st):
        if shader in ("solid discard", "texture with a hole"):
            return False
        # without a depth test blended fragments are shaded as they come
        return st["ReadDepth"] or not (st["AlphaBlend"] and st["WriteColor"]) or shader in ("solid", "phong")
    _check(f"{shader}, {state}", SHADERS[shader](), 97, 67, draws, STATES[state], first=first)


@pytest.mark.gpu
@pytest.mark.parametrize("tile", [(32, 32), (64, 32), (32, 16), (64, 64), (128, 64)])
@pytest.mark.parametrize("shader", ["phong", "texture", "solid translucent"])
def test_tile_shapes(shader, tile):
    # 900 large triangles: hundreds of fragments a pixel, mostly behind
    _check(f"{shader}, {tile}", SHADERS[shader](), 257, 131, [_soup(900, 3, 0.9)], [{}], tile,
           first=lambda st: tile[0] * tile[1] <= 2048)


@pytest.mark.gpu
@pytest.mark.parametrize("shader", ["phong", "texture"])
@pytest.mark.parametrize("size", [(1000, 800), (1600, 1504)])
@pytest.mark.parametrize("deep", [True, False])
def test_many_tiles(shader, size, deep):
    W, H = size
    prims = _soup(60, 4, 0.9) if deep else _soup(40, 5, 0.1)
    ctx = _check(f"{shader}, {W}x{H}, deep {deep}", SHADERS[shader](), W, H, [prims], [{}])
    assert (ctx.DrawStats()["fragments"] >= 2 * W * H) == deep
    assert ctx.DepthFirst() == (deep or W * H < 2304 * 1024)


@pytest.mark.gpu
@pytest.mark.parametrize("n", [102400, 102401])
@pytest.mark.parametrize("deep", [True, False])
def test_dense_triangles(n, deep):
    # 800 tiles: at 128 triangles a tile depth first, above it the device picks
    W, H = 1000, 800
    prims = _soup(n, 6, 0.03 if deep else 0.004)
    ctx = _check(f"{n} triangles, deep {deep}", SHADERS["phong"](), W, H, [prims], [{}])
    assert (ctx.DrawStats()["fragments"] >= 2 * W * H) == deep
    assert ctx.DepthFirst() == (deep or n == 102400)


@pytest.mark.gpu
@pytest.mark.parametrize("shader", ["solid translucent", "texture", "phong", "texture with a hole"])
@pytest.mark.parametrize("size,n", [((97, 67), 60), ((1000, 800), 300), ((1600, 1504), 300)])
def test_forced_fragment_overflow(shader, size, n):
    """A draw over opaque pixels whose first pass runs out of fragments: no
    tile of that pass may draw, whichever of its workgroups sees the overflow
    set by another first; blended pixels drawn twice would differ.  800 and 2350
    tiles are more than are resident at once; the draw with a hole is shaded first."""
    W, H = size
    _say(f"depth first: forced fragment overflow, {shader}, {W}x{H}")
    below, prims = _soup(40, 8, 0.9), _soup(n, 9, 0.7)
    octx, ctx = O.Context(W, H), A.NewContext(W, H)
    ctx.Cull = A.CullNone
    octx.set_state(O.make_state(front_face=O.FACE_CCW, line_width=2.0, read_depth=True, write_depth=True,
                                write_color=True, alpha_blend=True, wireframe=False, cull=A.CullNone, depth_bias=0.0))
    ctx.Shader = SHADERS[shader]()
    ctx.DrawTriangles(prims)  # sizes the other buffers
    for bg in (A.White, A.Color(0.1, 0.2, 0.3, 0.5)):
        ri, gi = [], []
        octx.clear_color(tuple(bg))
        octx.clear_depth(A.MaxFloat64)
        ctx.ClearColorBufferWith(bg)
        ctx.ClearDepthBuffer()
        for p, name, forced in ((below, "solid", False), (prims, shader, True)):
            sh = SHADERS[name]()
            octx.set_shader(oracle_shader(sh))
            ctx.Shader = sh
            ri.append(octx.draw_triangles(O.Mesh(tris=p.arrays()), 1))
            if forced:
                ctx.ForceCapacities(fragments=1)
            gi.append(tuple(ctx.DrawTriangles(p)))
        st = ctx.DrawStats()
        assert st["overflow_mask"] == 32 and st["reruns"] == 1, st
        assert ctx.DepthFirst() == (shader != "texture with a hole")
        res = compare((octx.color(), octx.depth(), ri), (ctx.Image(), ctx.DepthBuffer, gi), color_tol=0)
        assert res["ok"], res
