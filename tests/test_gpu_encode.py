"""The 2D encoder's chunks at their edges, against the oracle's streams: 8
blocks of 12x12 codes (whole, ragged, and across a strip of 64 rows), 1024 ids,
one row, one column, and codes so long that a chunk's bits leave its LDS words
(16 bits a code and more)."""
import numpy as np
import pytest

import cpsz_amd as cz
from _libs import load_oracle, mask_2d_padding

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def orc():
    return load_oracle()


def _field(r1, r2):
    rng = np.random.default_rng(r1 * 5000 + r2)
    y, x = np.arange(r1)[:, None], np.arange(r2)[None, :]
    out = []
    for a in (0.9, 2.3):
        f = np.sin(a * y / 31 + x / 47) + 0.3 * np.cos(a * x / 13) + 1e-3 * rng.standard_normal((r1, r2))
        f[rng.random((r1, r2)) < 0.05] = 0  # unpredictable values in most chunks
        out.append(f.astype(np.float32))
    return out


def _rare(r1, r2):
    """A flat field with a patch of noise: its codes are rare, so they are long."""
    rng = np.random.default_rng(3)
    out = []
    for _ in range(2):
        f = np.ones((r1, r2))
        f[300:396, 96:288] += rng.uniform(-0.4, 0.4, (96, 192))
        out.append(f.astype(np.float32))
    return out


SHAPES = [(12, 95), (13, 96), (24, 97), (61, 192), (70, 289), (31, 33), (64, 16), (1, 1024), (1025, 1), (1, 97)]


@pytest.mark.parametrize("shape", SHAPES + ["rare"], ids=str)
@pytest.mark.parametrize("dtype", [np.float32, np.float64], ids=["f32", "f64"])
def test_chunk_edges(orc, shape, dtype):
    print(f"[encode] {shape} {dtype.__name__}", flush=True)
    r1, r2 = (1200, 1200) if shape == "rare" else shape
    U, V = _rare(r1, r2) if shape == "rare" else _field(r1, r2)
    U, V = U.astype(dtype), V.astype(dtype)
    eb = 1e-4 if shape == "rare" else 0.05
    s, ref = cz.sz_compress_cp_preserve_2d_offline(U, V, eb), orc.compress_2d(U, V, eb)
    vb = U.dtype.itemsize
    assert np.array_equal(mask_2d_padding(s, r1, r2, vb), mask_2d_padding(ref, r1, r2, vb))
