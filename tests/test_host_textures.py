"""An image texture used by one context after another.  CPU only."""
import pytest

import host_only


@pytest.mark.parametrize("end", ["c.close()", "del c"])
def test_a_texture_outlives_contexts(end):
    """A later context may get the address of one that is gone: the texture
    is still uploaded to it, and is not another one of its textures."""
    host_only.run(f"""
one = A.NewImageTexture(np.full((4, 4, 4), 255, dtype=np.uint8), "NRGBA")
two = A.NewImageTexture(np.full((8, 8, 4), 255, dtype=np.uint8), "NRGBA")
tri = A.Prims(np.random.default_rng(0).uniform(-1, 1, (3, 3, 3)))
seen, again = set(), 0
for k in range(20):
    c = A.NewContext(16, 16)
    again += c._ptr().value in seen
    seen.add(c._ptr().value)
    for tex in (one, two) if k % 2 else (two, one):
        c.Shader = A.NewTextureShader(A.Identity(), tex)
        c.DrawTriangles(tri)
    assert one.handle(c) != two.handle(c)
    assert (one.handle(c) < two.handle(c)) == bool(k % 2)  # each uploaded to this context, in this order
    {end}
assert again
""")
