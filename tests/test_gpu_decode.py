"""The device's Huffman decoder on trees that do not resynchronize: sections of
a stream re-encoded with codes of one length (each of its phases stays possible
for the whole stream; beyond 16 bits, more of them than the decoder keeps) and
with codes of up to 64 bits must decompress to what the original does."""
import ctypes as C
import struct

import numpy as np
import pytest
import torch

import cpsz_amd as cz

pytestmark = pytest.mark.gpu


def _field(r1, r2):
    rng = np.random.default_rng(r1 * 1000 + r2)
    y, x = np.arange(r1)[:, None], np.arange(r2)[None, :]
    out = []
    for a in (0.7, 1.9):
        f = np.sin(a * y / 37 + x / 53) + 0.3 * np.cos(a * x / 11) + 1e-3 * rng.standard_normal((r1, r2))
        f[: r1 // 3] = 0.5  # a long run of one symbol
        out.append(f.astype(np.float32))
    return out


def _sections(s, r1, r2):
    """Offsets of the id, u and v Huffman sections."""
    def end(o):
        tsz = struct.unpack_from("<I", s, o + 8)[0]
        return o + 20 + tsz + struct.unpack_from("<Q", s, o + 12 + tsz)[0]

    def codes(o):
        unp = struct.unpack_from("<Q", s, o + 25)[0]
        return o + 33 + 4 * unp + ((r1 + 11) // 12 * ((r2 + 11) // 12) - 1) // 8 + 1

    u0 = end(36)
    return [36, codes(u0), codes(u0 + struct.unpack_from("<Q", s, 20)[0])], end


def _decode(s, o, n):
    nc, tsz = struct.unpack_from("<QI", s, o)
    tree = np.frombuffer(s, np.uint8, tsz, o + 12).copy()
    nb = struct.unpack_from("<Q", s, o + 12 + tsz)[0]
    bits = np.frombuffer(s, np.uint8, nb, o + 20 + tsz).copy()
    out = np.zeros(n, np.uint32)
    f = cz.lib().cpsz_huffman_decode_host
    f.argtypes = [C.c_void_p, C.c_size_t, C.c_size_t, C.c_void_p, C.c_size_t, C.c_size_t, C.c_void_p]
    assert f(tree.ctypes.data, tree.size, nc, bits.ctypes.data, bits.size, n, out.ctypes.data) == 0
    return out


def _encode(syms, kind, depth):
    """A section holding syms: codes of `depth` bits each, or a spine of codes of 1 to 64 bits."""
    present = np.unique(syms)
    if kind == "spine":
        assert depth == 64 and present.size <= depth + 1
        leaf = np.resize(present[np.argsort([-np.count_nonzero(syms == p) for p in present])], depth + 1)[::-1]
        code = {int(p): "1" * k + "0" * (k < depth) for k, p in enumerate(leaf)}  # the commonest is deepest
        N = 2 * depth + 1  # node 2k: spine, 2k + 1: its leaf
        L, R, T, S = (np.zeros(N, np.int64) for _ in range(4))
        for k in range(depth):
            L[2 * k], R[2 * k] = 2 * k + 1, 2 * k + 2
            T[2 * k + 1], S[2 * k + 1] = 1, leaf[k]
        T[2 * depth], S[2 * depth] = 1, leaf[depth]
        bits = "".join([code[int(x)] for x in syms])
        raw = np.frombuffer(bits.encode(), np.uint8) - 48
    else:
        n = 1 << depth
        leaf = np.resize(present, n)  # any leaf of a symbol will do: one at random for each use
        N = 2 * n - 1  # heap order
        i = np.arange(N)
        T = (i >= n - 1).astype(np.int64)
        L, R = np.where(T, 0, 2 * i + 1), np.where(T, 0, 2 * i + 2)
        S = np.where(T, leaf[np.maximum(i - n + 1, 0)], 0)
        rng = np.random.default_rng(depth)
        at = np.searchsorted(present, syms)
        c = at + present.size * rng.integers(0, np.maximum((n - 1 - at) // present.size + 1, 1))
        c[: c.size // 2] = at[: c.size // 2]  # and a fixed one in the first half
        assert np.array_equal(leaf[c], syms)
        raw = ((c[:, None] >> np.arange(depth - 1, -1, -1)) & 1).astype(np.uint8).ravel()
    w = np.uint8 if N <= 256 else np.uint16 if N <= 65536 else np.uint32
    tree = b"\0" + L.astype(w).tobytes() + R.astype(w).tobytes() + S.astype(np.uint32).tobytes() + T.astype(np.uint8).tobytes()
    bits = np.packbits(raw).tobytes()
    return struct.pack("<QI", N, len(tree)) + tree + struct.pack("<Q", len(bits)) + bits


# (section, kind, bits): 11 is the width of the first decode table, 16 the starts kept per segment
CASES = [(0, "fixed", 6), (0, "fixed", 17), (0, "spine", 64), (1, "fixed", 11), (1, "fixed", 12), (2, "fixed", 16), (2, "fixed", 17)]


@pytest.mark.parametrize("shape", [(5, 7), (70, 300)], ids=lambda s: f"{s[0]}x{s[1]}")
@pytest.mark.parametrize("sec,kind,depth", CASES)
def test_slow_resynchronization(shape, sec, kind, depth):
    r1, r2 = shape
    print(f"[decode] section {sec} {kind} {depth} {r1}x{r2}", flush=True)
    U, V = _field(r1, r2)
    s = cz.sz_compress_cp_preserve_2d_offline(U, V, 0.01).tobytes()
    want = cz.sz_decompress_cp_preserve_2d_offline(np.frombuffer(s, np.uint8), r1, r2)
    off, end = _sections(s, r1, r2)
    o = off[sec]
    h = _encode(_decode(s, o, 2 * r1 * r2 if sec == 0 else r1 * r2), kind, depth)
    t = bytearray(s[:o] + h + s[end(o):])
    if sec == 1:  # the u component's size
        struct.pack_into("<Q", t, 20, struct.unpack_from("<Q", s, 20)[0] + len(h) - (end(o) - o))
    t = np.frombuffer(bytes(t), np.uint8)
    outs = [(torch.empty(r1, r2, device="cuda"), torch.empty(r1, r2, device="cuda")) for _ in range(2)]
    d = [torch.from_numpy(x.copy()).cuda() for x in (t, np.frombuffer(s, np.uint8))]
    torch.cuda.synchronize()
    cz.decompress_2d_batch_dev([(x.data_ptr(), x.numel()) for x in d], [(r1, r2)] * 2,
                               [(u.data_ptr(), v.data_ptr()) for u, v in outs])
    batch = [tuple(x.cpu().numpy() for x in o) for o in outs]
    for got in [cz.sz_decompress_cp_preserve_2d_offline(t, r1, r2)] + batch:
        for g, e in zip(got, want):
            assert np.array_equal(g.view(np.uint32), e.view(np.uint32))


def test_batch_unpredictable_values():
    """Blocks with no, few and only unpredictable codes (land is stored as it is) in one batch, against the
    single-field decoder."""
    shapes = [(70, 300), (25, 13), (200, 97), (1, 40), (37, 1), (12, 12)]
    dev, streams, want = [], [], []
    for k, (r1, r2) in enumerate(shapes):
        print(f"[unpredictable] {r1}x{r2}", flush=True)
        U, V = _field(r1, r2)
        rng = np.random.default_rng(k)
        for F in (U, V):
            F[rng.random(F.shape) < 0.03] = 0
            F[r1 // 2:, : (2 * r2) // 3] = 0
        s = cz.sz_compress_cp_preserve_2d_offline(U, V, 0.05)
        want.append(cz.sz_decompress_cp_preserve_2d_offline(s, r1, r2))
        streams.append(torch.from_numpy(np.array(s)).cuda())
    outs = [(torch.empty(*s, device="cuda"), torch.empty(*s, device="cuda")) for s in shapes]
    torch.cuda.synchronize()
    cz.decompress_2d_batch_dev([(x.data_ptr(), x.numel()) for x in streams], shapes,
                               [(u.data_ptr(), v.data_ptr()) for u, v in outs])
    for o, w in zip(outs, want):
        for g, e in zip(o, w):
            assert np.array_equal(g.cpu().numpy().view(np.uint32), np.asarray(e).reshape(g.shape).view(np.uint32))
