"""Draws whose fragments are depth-tested before they are shaded, bit for bit
against the oracle (color, depth, RasterizeInfo), over what selects and ends
that path: opaque and blending colors of every shader, textures with and
without a texel of alpha 0, color, depth write and depth test off, depth
biases, marked clears before and after; few tiles, many, and more than 2304;
draws of more than 2048 triangles, where the device picks, on both sides of
what it picks by; every tile shape; overlap deep enough that the queue of
blended survivors fills and wraps.  Every test says which way each draw is to
have gone."""
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
    prims = _soup(60, 4, 0.9) if deep else _soup(40, 5, 0.1)  # up to 2304 tiles not asked
    ctx = _check(f"{shader}, {W}x{H}, deep {deep}", SHADERS[shader](), W, H, [prims], [{}])
    assert (ctx.DrawStats()["fragments"] >= 2 * W * H) == deep
    assert ctx.DepthFirst() == (deep or W * H < 2304 * 1024)


def _pad(prims, n):
    """The triangles and as many with no pixel as make n."""
    k = n - len(prims.position)
    far = np.broadcast_to(np.array([[3.0, 0, 0], [4, 0, 0], [3, 1, 0]]), (k, 3, 3))
    return A.Prims(np.concatenate([prims.position, far]), np.concatenate([prims.normal, M.with_face_normals(far)]),
                   np.concatenate([prims.texture, np.zeros((k, 3, 2))]))


def _quads(k):
    """k screens of two triangles, behind each other in turns: 32 to 128 spans a
    screen in a 32 x 32 tile (the box's last column wraps into the next row)."""
    z = np.random.Generator(np.random.PCG64(k)).permutation(np.linspace(-0.9, 0.9, k))
    a = np.array([[[-1, -1], [1, -1], [1, 1]], [[-1, -1], [1, 1], [-1, 1]]], dtype=float)
    pos = np.concatenate([np.broadcast_to(a, (k, 2, 3, 2)), np.broadcast_to(z[:, None, None, None], (k, 2, 3, 1))], axis=3)
    pos = np.ascontiguousarray(pos.reshape(-1, 3, 3))
    return A.Prims(pos, M.with_face_normals(pos), np.random.Generator(np.random.PCG64(1)).uniform(0, 1, (2 * k, 3, 2)))


def _crowd(n, W, H, px=32, size=8):
    """n triangles of some `size` pixels in the frame's first px x px."""
    p = _soup(n, 12, 1.0)
    c = p.position.mean(axis=1, keepdims=True)
    pos = c + (p.position - c) * [size / px, size / px, 0.1]
    pos = np.clip(pos, -1, 1) * [px / W, px / H, 1] + [px / W - 1, 1 - px / H, 0]
    return A.Prims(pos, M.with_face_normals(pos), p.texture)


# (frame, draw, shader, tested first).  A tile is 32 x 32.  Draws of more than
# 2048 filled triangles are tested first unless a tile is crowded: it holds more than
# 6000 spans and more than a 32nd of all (blended 3500 and a 64th; in
# more than 512 tiles 1750 and a 128th).
# Above 2304 tiles, and 128 triangles a tile in a large frame, they are where
# there are two fragments a pixel and no tile has 1280 spans and a 256th.
PICKS = {
    "crowd, the largest unasked": ((1920, 1080), lambda W, H: _crowd(2048, W, H, 32, 28), "phong", True),
    "crowd": ((1920, 1080), lambda W, H: _crowd(2500, W, H, 32, 28), "phong", False),
    "no crowd": ((1920, 1080), lambda W, H: _crowd(2500, W, H, 320, 8), "phong", True),
    "crowd, blended": ((1920, 1080), lambda W, H: _crowd(2200, W, H, 32, 8), "phong translucent", False),
    "the same, opaque": ((1920, 1080), lambda W, H: _crowd(2200, W, H, 32, 8), "phong", True),
    "crowd, few tiles": ((256, 256), lambda W, H: _crowd(2500, W, H, 32, 28), "phong", False),
    "crowd, one tile": ((32, 32), lambda W, H: _quads(450), "texture", False),
    "few tiles, short": ((96, 64), lambda W, H: _quads(40), "phong", True),
    "few tiles, uneven": ((256, 64), lambda W, H: _quads(350), "solid", False),
    "few tiles, even": ((1024, 128), lambda W, H: _quads(350), "solid", True),
    "few tiles, blended, uneven": ((512, 64), lambda W, H: _quads(180), "solid translucent", False),
    "few tiles, blended, even": ((1024, 256), lambda W, H: _quads(180), "solid translucent", True),
    "many tiles, blended, crowd": ((864, 640), lambda W, H: _crowd(1000, W, H, 32, 8), "texture", False),
    "the same, opaque, many tiles": ((864, 640), lambda W, H: _crowd(1000, W, H, 32, 8), "phong", True),
    "the same, few tiles": ((512, 512), lambda W, H: _crowd(1000, W, H, 32, 8), "texture", True),
    "the same, not asked": ((864, 640), lambda W, H: _pad(_crowd(1000, W, H, 32, 8), 2048), "texture", True),
    "dense, shallow": ((1000, 800), lambda W, H: _soup(102401, 6, 0.004), "phong", False),
    "not so dense": ((1000, 800), lambda W, H: _soup(102400, 6, 0.004), "phong", True),
    "dense, deep": ((1000, 800), lambda W, H: _soup(102401, 6, 0.03), "phong", True),
    "dense, deep, crowded": ((1000, 800), lambda W, H: _pad(_crowd(4000, W, H, 200, 190), 102401), "phong", False),
    "many tiles, deep": ((1600, 1504), lambda W, H: _quads(6), "phong", True),
    "many tiles, shallow": ((1600, 1504), lambda W, H: _quads(1), "phong", False),
    "many tiles, deep, no color": ((1600, 1504), lambda W, H: _quads(6), "solid", True),
    "many tiles, deep, crowded": ((1600, 1504), lambda W, H: _crowd(6000, W, H, 200, 190), "phong", False),
}


@pytest.mark.gpu
@pytest.mark.parametrize("name", list(PICKS))
def test_picks(name):
    (W, H), draw, shader, want = PICKS[name]
    prims = draw(W, H)
    if len(prims.position) < 2048:
        prims = _pad(prims, 2049)
    state = {"WriteColor": False} if name.endswith("no color") else {}
    ctx = _check(name, SHADERS[shader](), W, H, [prims], [state], first=lambda st: want)
    deep = ctx.DrawStats()["fragments"] >= 2 * W * H
    assert deep or ", deep" not in name
    assert ctx.DrawStats()["reruns"] == 0


# lines and wireframe triangles in one tile, more than a crowd of filled
# triangles: asked only where a tile gets 256 threads (blended, more than 512 tiles)
SMALL, MANY = (640, 480), (864, 640)


@pytest.mark.gpu
@pytest.mark.parametrize("size,shader,n,want", [(SMALL, "solid", 341, True), (SMALL, "solid", 500, True),
                                                (SMALL, "solid translucent", 500, True), (MANY, "solid", 500, True),
                                                (MANY, "solid translucent", 500, False),
                                                (MANY, "solid translucent", 341, True)])
def test_picks_wireframe(size, shader, n, want):
    """A wireframe triangle is six to the rule."""
    prims = _crowd(n, *size, 32, 28)
    _check(f"{n} wireframe triangles, {shader}, {size}", SHADERS[shader](), *size, [prims], [{"Wireframe": True}],
           first=lambda st: want)


@pytest.mark.gpu
@pytest.mark.parametrize("size,shader,n,want", [(SMALL, "solid", 1024, True), (SMALL, "solid", 1300, True),
                                                (SMALL, "solid translucent", 1300, True), (MANY, "solid", 1300, True),
                                                (MANY, "solid translucent", 1300, False),
                                                (MANY, "solid translucent", 1024, True)])
def test_picks_lines(size, shader, n, want):
    """A line is two triangles to the rule."""
    W, H = size
    _say(f"depth first: {n} lines, {shader}, {W}x{H}")
    p = _crowd(n, W, H, 32, 30).position[:, :2].copy()
    lines = A.Prims(p, None, None, None, nv=2)
    sh = SHADERS[shader]()
    octx, ctx = O.Context(W, H), A.NewContext(W, H)
    octx.clear_color(tuple(A.White))
    octx.clear_depth(A.MaxFloat64)
    ctx.ClearColorBufferWith(A.White)
    octx.set_shader(oracle_shader(sh))
    octx.set_state(O.make_state(front_face=O.FACE_CCW, line_width=2.0, read_depth=True, write_depth=True,
                                write_color=True, alpha_blend=True, wireframe=False, cull=O.CULL_BACK, depth_bias=0.0))
    ctx.Shader = sh
    ri = octx.draw_lines(O.Mesh(lines=lines.arrays()), 1)
    gi = tuple(ctx.DrawLines(lines))
    assert ctx.DepthFirst() == want
    res = compare((octx.color(), octx.depth(), [ri]), (ctx.Image(), ctx.DepthBuffer, [gi]), color_tol=0)
    assert res["ok"], res


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


@pytest.mark.gpu
@pytest.mark.parametrize("caps", [{"fragments": 1}, {"spans": 1}, {"pairs": 1}, {"spans": 1, "fragments": 1}])
def test_forced_overflow_of_a_crowd(caps):
    """A draw that a crowded tile sends the other way, and that runs out on it."""
    W, H = 256, 256
    _say(f"depth first: crowd, forced {caps}")
    prims, sh = _crowd(2500, W, H, 32, 28), SHADERS["phong translucent"]()
    octx, ctx = O.Context(W, H), A.NewContext(W, H)
    ctx.Cull, ctx.Shader = A.CullNone, sh
    octx.clear_color(tuple(A.White))
    octx.clear_depth(A.MaxFloat64)
    octx.set_shader(oracle_shader(sh))
    octx.set_state(O.make_state(front_face=O.FACE_CCW, line_width=2.0, read_depth=True, write_depth=True,
                                write_color=True, alpha_blend=True, wireframe=False, cull=A.CullNone, depth_bias=0.0))
    ctx.DrawTriangles(prims)  # sizes the buffers
    ctx.ClearColorBufferWith(A.White)
    ctx.ClearDepthBuffer()
    ri = octx.draw_triangles(O.Mesh(tris=prims.arrays()), 1)
    ctx.ForceCapacities(**caps)
    gi = tuple(ctx.DrawTriangles(prims))
    assert ctx.DrawStats()["reruns"] == 1 and not ctx.DepthFirst()
    res = compare((octx.color(), octx.depth(), [ri]), (ctx.Image(), ctx.DepthBuffer, [gi]), color_tol=0)
    assert res["ok"], res
