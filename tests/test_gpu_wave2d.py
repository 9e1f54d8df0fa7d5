"""The 2D wavefronts against the oracle at the edges of their tiling: strips of
64 rows, groups of four strips (two for double fields) that hand a row to each
other through memory, chunks of 16 steps, single rows and columns, eb ids above
81 (the double-precision step), and a strip of 4 GiB (64-bit offsets)."""
import numpy as np
import pytest

import cpsz_amd as cz
from _libs import load_oracle, mask_2d_log_padding, mask_2d_padding

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def orc():
    return load_oracle()


def _field(r1, r2, seed, scale=(1.0, 1.0)):
    rng = np.random.default_rng(seed)
    y, x = np.arange(r1)[:, None], np.arange(r2)[None, :]
    out = []
    for k in range(2):
        a, b, c = rng.uniform(0.5, 3, 3)
        f = np.sin(a * y / 37 + b * x / 53) + 0.3 * np.cos(c * x / 11) + 1e-3 * rng.standard_normal((r1, r2))
        f[rng.random((r1, r2)) < 0.01] = 0
        out.append((f * scale[k]).astype(np.float32))
    return out


def _same(a, b):
    k = np.uint64 if a.dtype == np.float64 else np.uint32
    return np.array_equal(a.view(k), b.view(k))


SHAPES = [(1, 1), (1, 2), (2, 1), (1, 17), (300, 1), (3, 15), (63, 16), (64, 17), (65, 2), (127, 64), (128, 65), (129, 33),
          (255, 79), (256, 80), (257, 81), (513, 31), (320, 200)]
# fewer columns than 64 and than rows: taken with rows and columns exchanged
SHAPES += [(2, 2), (3, 2), (40, 25), (64, 63), (130, 63), (200, 12), (97, 13), (1000, 3), (301, 48), (75, 24)]


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: f"{s[0]}x{s[1]}")
@pytest.mark.parametrize("codec", ["f32", "wide", "f64", "log"])
def test_tiling_edges(orc, shape, codec):
    r1, r2 = shape
    print(f"[wave2d] {codec} {r1}x{r2}", flush=True)
    U, V = _field(r1, r2, r1 * 1000 + r2, (1e35, 1e-5) if codec == "wide" else (1.0, 1.0))
    if codec == "wide":
        # bounds up to 1e34 give ids beyond 81; v > 0, since the squares of a critical point's terms would overflow
        V = np.abs(V) + np.float32(1e-6)
    if codec == "f64":
        rng = np.random.default_rng(7)
        U, V = (a.astype(np.float64) * (1 + 1e-9 * rng.standard_normal(a.shape)) for a in (U, V))
    if codec == "log":
        s, ref = cz.sz_compress_cp_preserve_2d_offline_log(U, V, 0.1), orc.compress_2d_log(U, V, 0.1)
        assert np.array_equal(mask_2d_log_padding(s, r1, r2), mask_2d_log_padding(ref, r1, r2))
        got, want = cz.sz_decompress_cp_preserve_2d_offline_log(ref, r1, r2), orc.decompress_2d_log(ref, r1, r2)
    else:
        s, ref = cz.sz_compress_cp_preserve_2d_offline(U, V, 0.1), orc.compress_2d(U, V, 0.1)
        vb = U.dtype.itemsize
        assert np.array_equal(mask_2d_padding(s, r1, r2, vb), mask_2d_padding(ref, r1, r2, vb))
        got, want = cz.sz_decompress_cp_preserve_2d_offline(ref, r1, r2, U.dtype), orc.decompress_2d(ref, r1, r2, U.dtype)
    assert _same(got[0], want[0]) and _same(got[1], want[1])


def test_strip_of_four_gib(orc):
    r1, r2 = 2, 1 << 24
    print(f"[wave2d] {r1}x{r2}", flush=True)
    x = np.arange(r2, dtype=np.float32)
    U = np.stack([np.sin(x / 531), np.cos(x / 917)]).astype(np.float32) + np.float32(1e-3)
    V = np.stack([np.cos(x / 713), np.sin(x / 389)]).astype(np.float32)
    s, ref = cz.sz_compress_cp_preserve_2d_offline(U, V, 0.1), orc.compress_2d(U, V, 0.1)
    assert np.array_equal(mask_2d_padding(s, r1, r2), mask_2d_padding(ref, r1, r2))
    got, want = cz.sz_decompress_cp_preserve_2d_offline(ref, r1, r2), orc.decompress_2d(ref, r1, r2)
    assert _same(got[0], want[0]) and _same(got[1], want[1])


def test_flipped_strip_of_four_gib(orc):
    """Two columns, taken as two rows of 2^24."""
    r1, r2 = 1 << 24, 2
    print(f"[wave2d] {r1}x{r2}", flush=True)
    x = np.arange(r1, dtype=np.float32)
    U = np.stack([np.sin(x / 531), np.cos(x / 917)], axis=1).astype(np.float32) + np.float32(1e-3)
    V = np.stack([np.cos(x / 713), np.sin(x / 389)], axis=1).astype(np.float32)
    U[::97] = 0
    s, ref = cz.sz_compress_cp_preserve_2d_offline(U, V, 0.1), orc.compress_2d(U, V, 0.1)
    assert np.array_equal(mask_2d_padding(s, r1, r2), mask_2d_padding(ref, r1, r2))
    got, want = cz.sz_decompress_cp_preserve_2d_offline(ref, r1, r2), orc.decompress_2d(ref, r1, r2)
    assert _same(got[0], want[0]) and _same(got[1], want[1])


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_tiles_of_four_gib(orc, dtype):
    """Rows a little under 4 GiB a strip, whose tiles are a little over: the last value of the third row lies past 4 GiB.
    Zeros in every other column have it stored as it is."""
    r1, r2 = 3, (1 << 32) // 64 // np.dtype(dtype).itemsize - 1
    print(f"[wave2d] {np.dtype(dtype).name} {r1}x{r2}", flush=True)
    rng = np.random.default_rng(1)
    x = np.arange(r2, dtype=np.float32)
    fields = []
    for a, b in ((531, 713), (917, 389)):
        f = np.stack([np.sin(x / a), np.cos(x / b), np.sin(x / b)]).astype(dtype) + dtype(1.5)
        f[:, -60:] = rng.standard_normal((r1, 60))
        f[:, -60::2] = 0
        fields.append(f)
    s = cz.sz_compress_cp_preserve_2d_offline(*fields, 0.1)
    want = orc.decompress_2d(s, r1, r2, dtype)
    assert all(w[2, -1] == f[2, -1] and w[2, -1] != 0 for w, f in zip(want, fields))
    got = cz.sz_decompress_cp_preserve_2d_offline(s, r1, r2, dtype)
    assert _same(got[0], want[0]) and _same(got[1], want[1])
