"""Host checks (no GPU) of the 2D wavefront's addressing and of the words that its strips hand to each other."""
import numpy as np
import pytest

import cpsz_amd as cz


@pytest.mark.parametrize("value_bytes", [4, 8])
@pytest.mark.parametrize("rows", [1, 2, 3, 33, 64, 1000])
def test_offsets_within_a_strip_fit(rows, value_bytes):
    """32-bit byte offsets only where a strip's last value has one, in the row-major arrays and in the tiles."""
    edge = (1 << 32) // (64 * value_bytes)  # columns of a row-major strip of 4 GiB
    for r2 in [2, 63, 4096, edge // 2] + list(range(edge - 100, edge + 3)):
        far, span = cz.wave2d_span(rows, r2, value_bytes)
        assert far or span <= (1 << 32) - 16, (rows, r2, span)  # (offsets from 2^32 - 16 on mean: no access)
        if r2 <= edge // 2:
            assert not far


@pytest.mark.parametrize("value_bytes", [4, 8])
@pytest.mark.parametrize("cols", [1, 2, 33, 63])
def test_offsets_of_a_few_columns(cols, value_bytes):
    edge = (1 << 32) // (64 * value_bytes)
    for r1 in [64, 1000, edge // 2] + list(range(edge - 100, edge + 3)):
        far, span = cz.wave2d_span(r1, cols, value_bytes)
        assert far or span <= (1 << 32) - 16, (r1, cols, span)


@pytest.mark.parametrize("bits,value", [(np.uint32, np.float32), (np.uint64, np.float64)])
def test_every_value_can_be_published(bits, value):
    """Any pattern, as a corrupt stream can hold it, reads as published: numbers as they are, a NaN as a NaN."""
    n = np.dtype(bits).itemsize * 8
    rng = np.random.default_rng(3)
    b = np.concatenate([rng.integers(0, (1 << n) - 1, 100000, dtype=bits, endpoint=True),
                        np.array([0, 1 << (n - 1), (1 << n) - 1], bits)])
    if n == 64:  # the NaNs around the pattern that stands for an empty word
        empty = 0x7FF4DEADBEEF0000
        b = np.concatenate([b, np.arange(empty - 3, empty + 4, dtype=np.uint64)])
    x = b.view(value)
    words, ready, read = cz.wave2d_boundary(x)
    assert ready.all(), [hex(int(w)) for w in words[~ready]]
    nan = np.isnan(x)
    assert np.array_equal(read[~nan].view(bits), b[~nan]) and np.isnan(read[nan]).all()


@pytest.mark.parametrize("shape", [(1, 1 << 32), ((1 << 32) + 7, 1), (3, 1 << 31), (1 << 21, 1 << 21), ((1 << 31) - 1, 2)])
def test_decompression_refuses_sides_beyond_its_range(shape):
    """(Scratch sized from a side cut to 32 bits would be written past its end.)"""
    for value_bytes in (4, 8):
        with pytest.raises(cz.CpszError):
            cz.scratch_bytes_2d(*shape, value_bytes)


@pytest.mark.parametrize("r1", [1, 2, 5, 16, 33, 63, 64, 65, 128, 130, 300])
def test_every_element_has_a_place_of_its_own(r1):
    for r2 in [1, 2, 3, 7, 8, 9, 15, 16, 17, 31, 40, 55, 56, 57, 63, 64, 65, 100, 128, 301]:
        at, n = cz.tile_index_2d(r1, r2)
        assert np.unique(at).size == r1 * r2 and at.max() < n, r2


# (r1, r2, slots per value): a compression keeps two components' eb codes by value and, by slot, these and the
# quantization codes again, a decompression ids, codes and unpredictable values by slot; either has the groups'
# boundary rows, at most 0.25 bytes a value
THIN = [(1, 1 << 20, 1), (1 << 20, 1, 1), (3, 1 << 20, 4 / 3), (33, 1 << 16, 64 / 33), (65, 1 << 16, 128 / 65), (1 << 18, 2, 1),
        (1 << 18, 3, 4 / 3), (1 << 18, 16, 1), (1 << 18, 17, 32 / 17), (1 << 18, 63, 64 / 63), (1 << 16, 64, 2),
        (1 << 16, 256, 1.25), (4096, 4096, 1.02)]


@pytest.mark.parametrize("r1,r2,slots", THIN)
def test_scratch_of_thin_fields(r1, r2, slots):
    comp, dec = (x / (r1 * r2) for x in cz.scratch_bytes_2d(r1, r2))
    assert comp <= (4 + 8 * slots + 0.25) * 1.01 + 1.2 and dec <= (16 * slots + 0.25) * 1.01
    # a row of 2^28 values is decompressed in a few gigabytes
    assert cz.scratch_bytes_2d(1, 1 << 28)[1] < 5 << 30
