"""The PNG encoder's deflate pieces, byte for byte, against the
one-symbol-at-a-time restatement in png_ref.py: stream lengths around a
piece and around a thread's 16 bytes, runs at the match lengths' edges and
across threads, waves and pieces, pieces that take the fixed codes, and a
piece whose code-length code would pass 7 bits.  Whole numbers throughout: no
tolerance."""
import sys

import numpy as np
import pytest

import oracle as O
import png_ref
from fauxgl_amd import api as A
from test_gpu_png import chunks


def _row(data):
    """A one-row opaque image whose bytes are data."""
    data = data[:len(data) - len(data) % 3]
    img = np.full((1, len(data) // 3, 4), 255, np.uint8)
    img[0, :, :3] = np.array(data, np.uint8).reshape(-1, 3)
    return img


def _runs(lengths, n):
    out, v = [], 0
    while len(out) < n:
        for r in lengths:
            v = (v + 85) % 256
            out += [v] * r
    return out[:n]


def _geometric(seed):
    """Bytes of geometric frequencies."""
    rng = np.random.Generator(np.random.PCG64(seed))
    k = int(rng.integers(60, 257))
    w = np.exp(-rng.uniform(0.02, 0.12) * np.arange(k)) ** rng.uniform(0.5, 2)
    return rng.choice(k, size=4095, p=w / w.sum())


def _image(name):
    rng = np.random.Generator(np.random.PCG64(9))
    if name.startswith("len"):  # len<n>: a filtered stream of n bytes, n = 1 mod 3
        return _row(rng.integers(0, 4, int(name[3:]) - 1))
    if name == "random":  # every byte equally likely
        return rng.integers(0, 256, (40, 101, 4), dtype=np.uint8)
    if name == "flat":  # one run through whole pieces
        return np.full((70, 64, 4), 255, np.uint8)
    if name == "runs":  # match lengths 3, 4, 258, the remainders of 1 and 2, and their neighbours
        return _row(_runs([1, 2, 3, 4, 5, 15, 16, 17, 64, 258, 259, 260, 261, 262, 263, 517, 518, 519, 1024], 9999))
    if name == "limit":  # a code-length code that would pass 7 bits
        return _row(_geometric(LIMIT_SEED))
    assert name == "gradient"
    y, x = np.mgrid[0:96, 0:131]
    return np.stack([x * 2 % 256, y * 3 % 256, (x + y) % 256, 128 + (x * y) % 128], axis=2).astype(np.uint8)


LIMIT_SEED = 178
CASES = ["len4", "len16", "len19", "len1024", "len4093", "len4096", "len4099", "len8191", "len8194", "random", "flat",
         "runs", "limit", "gradient"]


def test_reference_pieces_inflate():
    """The restatement itself: its streams inflate to the filtered bytes, and
    the cases reach the fixed codes, the dynamic ones and the length limit."""
    import zlib
    kinds, halved = set(), False
    for name in CASES:
        _, want = O.png_filter(_image(name))
        z, how = png_ref.zlib_stream(want)
        assert zlib.decompress(z) == want.tobytes()
        kinds |= {k for k, _ in how}
        halved |= any(h for _, h in how)
    assert kinds == {"fixed", "dynamic"} and halved


@pytest.mark.gpu
@pytest.mark.parametrize("name", CASES)
def test_pieces(name):
    print(f"[case] png pieces {name}", flush=True)
    sys.stdout.flush()
    img = _image(name)
    ctx = A.NewContext(img.shape[1], img.shape[0])
    ctx.SetColorBuffer(img)
    _, want = O.png_filter(img)
    z, _ = png_ref.zlib_stream(want)
    for _ in range(2):  # the second in a kept workspace
        assert chunks(ctx.EncodePNG())[1][1] == z


@pytest.mark.gpu
@pytest.mark.parametrize("alpha", [255, 254])
@pytest.mark.parametrize("h", [2500, 2560])
def test_workspace_sizes(h, alpha):
    """Frames on both sides of the size (10.3 Mpixel) above which the workspace
    is sized by what the device has found and is not kept."""
    import zlib
    print(f"[case] png workspace 4096x{h} alpha {alpha}", flush=True)
    rng = np.random.Generator(np.random.PCG64(h))
    img = rng.integers(0, 256, (h, 4096, 4), dtype=np.uint8)
    img[:, 1000:] //= 200  # long runs
    img[..., 3] = 255
    img[h - 1, 4095, 3] = alpha
    ctx = A.NewContext(4096, h)
    ctx.SetColorBuffer(img)
    bpp, want = O.png_filter(img)
    assert bpp == (3 if alpha == 255 else 4)
    first = ctx.EncodePNG()
    assert zlib.decompress(chunks(first)[1][1]) == want.tobytes()
    assert ctx.EncodePNG() == first
    ctx.close()
