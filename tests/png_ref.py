"""numpy PNG row filters and their inverse (RFC 2083 section 6), written
from the PNG specification for the tests."""
import numpy as np


def paeth(a, b, c):
    p = a + b - c
    pa, pb, pc = np.abs(p - a), np.abs(p - b), np.abs(p - c)
    return np.where((pa <= pb) & (pa <= pc), a, np.where(pb <= pc, b, c))


def candidates(cur, prev, bpp):
    """The five filtered versions (None, Sub, Up, Average, Paeth) of a row."""
    cur = cur.astype(np.int64)
    prev = prev.astype(np.int64)
    a = np.concatenate([np.zeros(bpp, np.int64), cur[:-bpp]])
    c = np.concatenate([np.zeros(bpp, np.int64), prev[:-bpp]])
    b = prev
    return [cur % 256, (cur - a) % 256, (cur - b) % 256, (cur - (a + b) // 2) % 256, (cur - paeth(a, b, c)) % 256]


def unfilter(stream, w, h, bpp):
    """Filtered stream -> (h, w * bpp) raw rows."""
    n = w * bpp
    rows = np.zeros((h, n), np.int64)
    prev = np.zeros(n, np.int64)
    for y in range(h):
        f = int(stream[y * (n + 1)])
        d = stream[y * (n + 1) + 1:(y + 1) * (n + 1)].astype(np.int64)
        cur = np.zeros(n, np.int64)
        for i in range(n):
            a = cur[i - bpp] if i >= bpp else 0
            b = prev[i]
            c = prev[i - bpp] if i >= bpp else 0
            pred = [0, a, b, (a + b) // 2, int(paeth(np.int64(a), np.int64(b), np.int64(c)))][f]
            cur[i] = (d[i] + pred) % 256
        rows[y] = cur
        prev = cur
    return rows


# ---------------------------------------------------------------------------
# the encoder's deflate pieces, one symbol at a time (RFC 1951; code lengths
# by Moffat and Katajainen's in-place method, 1995)

CHUNK = 4096
LEN_BASE = [3, 4, 5, 6, 7, 8, 9, 10, 11, 13, 15, 17, 19, 23, 27, 31, 35, 43, 51, 59, 67, 83, 99, 115, 131, 163, 195,
            227, 258]
LEN_EXTRA = [0] * 8 + [1] * 4 + [2] * 4 + [3] * 4 + [4] * 4 + [5] * 4 + [0]
CL_ORDER = [16, 17, 18, 0, 8, 7, 9, 6, 10, 5, 11, 4, 12, 3, 13, 2, 14, 1, 15]


def tokens(p):
    """Literals (v, 0) and distance-1 matches (None, length) of a piece."""
    out, i = [], 0
    while i < len(p):
        r = 1
        while i + r < len(p) and p[i + r] == p[i]:
            r += 1
        out.append((p[i], 0))
        rest = r - 1
        while rest >= 3:
            m = min(rest, 258)
            if 0 < rest - m < 3:
                m -= 3
            out.append((None, m))
            rest -= m
        out += [(p[i], 0)] * rest
        i += r
    return out


def huffman_lengths(freq, limit):
    """(lengths, halvings it took to stay within limit)."""
    order = sorted((i for i in range(len(freq)) if freq[i]), key=lambda i: (freq[i], i))
    m = len(order)
    assert m >= 2
    shift = 0
    while True:
        w = [((freq[i] - 1) >> shift) + 1 for i in order]
        w[0] += w[1]
        root, leaf = 0, 2
        for nxt in range(1, m - 1):
            if leaf >= m or w[root] < w[leaf]:
                w[nxt], w[root] = w[root], nxt
                root += 1
            else:
                w[nxt] = w[leaf]
                leaf += 1
            if leaf >= m or (root < nxt and w[root] < w[leaf]):
                w[nxt] += w[root]
                w[root] = nxt
                root += 1
            else:
                w[nxt] += w[leaf]
                leaf += 1
        w[m - 2] = 0
        for k in range(m - 3, -1, -1):
            w[k] = w[w[k]] + 1
        avail, depth, root, nxt = 1, 0, m - 2, m - 1
        while avail > 0:
            used = 0
            while root >= 0 and w[root] == depth:
                used, root = used + 1, root - 1
            for _ in range(avail - used):
                w[nxt] = depth
                nxt -= 1
            avail, depth = 2 * used, depth + 1
        if w[0] <= limit:
            break
        shift += 1
    lens = [0] * len(freq)
    for i, s in enumerate(order):
        lens[s] = w[i]
    return lens, shift


def canonical(lens):
    code, out = 0, {}
    for b in range(1, 16):
        code <<= 1
        for s, n in enumerate(lens):
            if n == b:
                out[s] = format(code, "0%db" % b)
                code += 1
    return out


def lsb(v, n):
    return format(v, "0%db" % n)[::-1] if n else ""


def deflate_piece(p):
    """(bytes of one piece, "fixed" or "dynamic", halvings of the code-length
    code; the literal code of 4096 bytes never passes 15 bits)."""
    toks = tokens(p)
    sym = lambda m: max(k for k in range(29) if LEN_BASE[k] <= m)
    freq = [0] * 286
    freq[256] = 1
    for v, m in toks:
        freq[v if m == 0 else 257 + sym(m)] += 1
    extra = sum(LEN_EXTRA[sym(m)] for _, m in toks if m)
    nmatch = sum(1 for _, m in toks if m)
    fixed = [8] * 144 + [9] * 112 + [7] * 24 + [8] * 6
    fixed_bits = 3 + sum(f * b for f, b in zip(freq, fixed)) + extra + 5 * nmatch
    lens, none = huffman_lengths(freq, 15)
    assert none == 0
    hlit = max(257, max(i for i in range(286) if lens[i]) + 1)
    seq, rle, i = lens[:hlit] + [1], [], 0
    while i < len(seq):
        r = 1
        while i + r < len(seq) and seq[i + r] == seq[i]:
            r += 1
        left, v = r, seq[i]
        if v == 0:
            while left >= 11:
                rle.append((18, min(left, 138) - 11))
                left -= min(left, 138)
            if left >= 3:
                rle.append((17, left - 3))
                left = 0
        else:
            rle.append((v, 0))
            left -= 1
            while left >= 3:
                rle.append((16, min(left, 6) - 3))
                left -= min(left, 6)
        rle += [(v, 0)] * left
        i += r
    clfreq = [0] * 19
    for s, _ in rle:
        clfreq[s] += 1
    cl, halvings = huffman_lengths(clfreq, 7)
    hclen = 19
    while hclen > 4 and cl[CL_ORDER[hclen - 1]] == 0:
        hclen -= 1
    xb = {16: 2, 17: 3, 18: 7}
    dyn_bits = 17 + 3 * hclen + sum(cl[s] + xb.get(s, 0) for s, _ in rle) + \
        sum(f * b for f, b in zip(freq, lens)) + extra + nmatch
    dyn = dyn_bits < fixed_bits
    bits = ["0", lsb(2 if dyn else 1, 2)]
    if dyn:
        bits += [lsb(hlit - 257, 5), lsb(0, 5), lsb(hclen - 4, 4)] + [lsb(cl[s], 3) for s in CL_ORDER[:hclen]]
        cc = canonical(cl)
        bits += [cc[s] + lsb(x, xb.get(s, 0)) for s, x in rle]
    code = canonical(lens if dyn else fixed + [8, 8])
    for v, m in toks:
        if m == 0:
            bits.append(code[v])
        else:
            k = sym(m)
            bits.append(code[257 + k] + lsb(m - LEN_BASE[k], LEN_EXTRA[k]) + ("0" if dyn else "00000"))
    bits = "".join(bits) + code[256] + "000"
    bits += "0" * (-len(bits) % 8) + "0" * 16 + "1" * 16
    data = bytes(int(bits[k:k + 8][::-1], 2) for k in range(0, len(bits), 8))
    return data, "dynamic" if dyn else "fixed", halvings


def zlib_stream(stream):
    """The encoder's zlib stream for the filtered bytes, and each piece's
    (kind, halvings)."""
    import zlib
    p = bytes(stream)
    pieces = [deflate_piece(p[k:k + CHUNK]) for k in range(0, len(p), CHUNK)]
    body = b"".join(d for d, _, _ in pieces)
    return b"\x78\x9c" + body + b"\x03\x00" + zlib.adler32(p).to_bytes(4, "big"), [(k, h) for _, k, h in pieces]
