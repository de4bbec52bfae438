"""What the host code keeps of freed device memory, and what it leaves behind
when the runtime refuses a call.  CPU only."""
import host_only

SETUP = """
def soup(n):
    r = np.random.Generator(np.random.PCG64(n))
    return A.Prims(r.uniform(-1, 1, size=(n, 3, 3)))
ctx = A.NewContext(64, 48)
"""


def test_a_refused_wait_leaves_no_error():
    """A buffer freed while the runtime refuses to wait for the device (a
    capture is open on another stream) leaves no error for the next call of
    this thread to report."""
    host_only.run(SETUP + """
dm = ctx.Upload(A.Mesh(soup(100)))
live = fake.fake_live()
fake.fake_refuse_sync(1000)
dm.SmoothNormals()  # its scratch buffers are let go at the end
assert fake.fake_last_error() == 0, fake.fake_last_error()
dm.close()
ctx.close()
assert fake.fake_last_error() == 0
assert fake.fake_live() < live  # freed all the same, and not kept
""")


def test_kept_memory_is_given_back_before_a_texture_is_refused():
    host_only.run(SETUP + """
before = fake.fake_live()
big = [A.NewContext(2000, 1500) for _ in range(4)]
for c in big:
    c.close()
kept = fake.fake_live() - before
assert kept >= 4 * 12 * 2000 * 1500, kept
# room for the texture only without what is kept
fake.fake_limit(fake.fake_live() + (1 << 20))
tex = A.NewImageTexture(np.full((2048, 1024, 4), 255, dtype=np.uint8), "NRGBA")
ctx.Shader = A.NewTextureShader(A.Identity(), tex)
ctx.DrawTriangles(soup(10))  # uploads the texture
assert fake.fake_last_error() == 0
# refused where there is no room even so, and nothing is left of the attempt
live = fake.fake_live()
fake.fake_limit(live + (1 << 20))
ctx.Shader = A.NewTextureShader(A.Identity(), A.NewImageTexture(np.full((2048, 2048, 4), 255, dtype=np.uint8), "NRGBA"))
try:
    ctx.DrawTriangles(soup(10))
    raise SystemExit("not refused")
except N.FglError:
    pass
fake.fake_limit(ctypes.c_size_t(-1).value)
ctx.DrawTriangles(soup(10))
""")


def test_trim_gives_everything_kept_back():
    host_only.run(SETUP + """
before = fake.fake_live()
c = A.NewContext(300, 200)
c.Image()
c.close()
assert fake.fake_live() > before
A.TrimMemory()
assert fake.fake_live() == before
A.TrimMemory()
""")


def test_kept_memory_is_bounded():
    host_only.run(SETUP + """
for bound, size, count in ((512 << 20, (2560, 1440), 40), (512 << 20, (64, 64), 300)):
    cs = [A.NewContext(*size) for _ in range(count)]
    for c in cs:
        c.close()
    assert fake.fake_live() <= bound + (1 << 20), fake.fake_live()
""")


def test_encoding_a_png_keeps_no_memory_in_the_context():
    """The workspace is kept as other freed blocks are, where it is one they
    take; a larger one is freed, and is no larger than the image needs (the
    fake device finds an opaque image and an empty stream)."""
    host_only.run(SETUP + """
c = A.NewContext(800, 600)
c.EncodePNG()
A.TrimMemory()
before = fake.fake_live()
c.EncodePNG()
assert before < fake.fake_live() < before + 13.2 * 800 * 600
n = fake.fake_mallocs()
c.EncodePNG()
assert fake.fake_mallocs() == n
A.TrimMemory()
assert fake.fake_live() == before
c.close()
c = A.NewContext(7680, 4320)
c.Image()
A.TrimMemory()
before = fake.fake_live()
fake.fake_peak()
c.EncodePNG()
A.TrimMemory()
assert fake.fake_live() <= before + 256, fake.fake_live() - before
assert fake.fake_peak() <= before + 6.45 * 7680 * 4320, (fake.fake_peak() - before) / (7680 * 4320)
""")


def test_encoding_a_png_leaves_recorded_batches_valid():
    """No buffer that a recorded batch uses is freed by it: the next run
    replays instead of drawing every view again (which would read counters
    back for each)."""
    host_only.run(SETUP + """
dm = ctx.Upload(A.Mesh(soup(100)))
ctx.Shader = A.NewSolidColorShader(A.Identity(), A.Black)
b = A.Batch()
b.Add(ctx, dm)
b.Run()
ctx.EncodePNG()
fake.fake_count_multi.restype = ctypes.c_long
fake.fake_count_multi()
b.Run()
assert fake.fake_count_multi() > 0  # replayed
""")
