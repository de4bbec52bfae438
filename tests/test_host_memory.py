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
