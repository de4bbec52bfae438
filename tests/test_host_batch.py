"""Recording a batch allocates, frees and waits for nothing (a stream capture
refuses it), whatever kinds of draws share a context.  CPU only."""
import pytest

import host_only

# On one context: a draw that can be Discard, which writes its fragments out;
# a larger one whose fragments are tested first and written nowhere, and which
# raises the context's capacities; and, for the batch to be recorded into a
# graph without being asked to, a view with an empty mesh.
PROGRAM = """
def soup(n):
    r = np.random.Generator(np.random.PCG64(n))
    return A.Prims(r.uniform(-1, 1, size=(n, 3, 3)))
ctx = A.NewContext(64, 48)
small, large = ctx.Upload(A.Mesh(soup(10))), ctx.Upload(A.Mesh(soup(400)))
empty = ctx.Upload(A.Mesh(A.Prims(np.zeros((0, 3, 3)))))
hole = A.NewSolidColorShader(A.Identity(), A.Discard)
solid = A.NewSolidColorShader(A.Identity(), A.Black)
b = A.Batch()
for mesh, shader in [{views}]:
    ctx.Shader = shader
    b.Add(ctx, mesh)
b.Run()  # draws, then records
assert fake.fake_capture_calls() == 0, fake.fake_capture_calls()
n = fake.fake_mallocs()
b.Run()
b.Run()  # replays
assert fake.fake_mallocs() == n
assert fake.fake_capture_calls() == 0
"""


@pytest.mark.parametrize("views,graph", [
    ("(empty, solid), (small, hole), (large, solid)", "0"),
    ("(small, hole), (large, solid), (empty, solid)", "0"),
    ("(small, hole), (large, solid)", "1"),
    ("(small, hole), (large, solid)", "0"),
    ("(large, solid), (small, hole), (empty, hole)", "0"),
])
def test_recording_allocates_nothing(views, graph):
    host_only.run(PROGRAM.replace("{views}", views), FGL_BATCH_GRAPH=graph)
