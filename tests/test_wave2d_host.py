"""Host checks (no GPU) of the 2D wavefront's addressing."""
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
def test_offsets_of_a_column(value_bytes):
    edge = (1 << 32) // (64 * value_bytes)
    for r1 in [1, 1000, edge // 2, edge - 63, edge - 1, edge]:
        far, span = cz.wave2d_span(r1, 1, value_bytes)
        assert far or span <= (1 << 32) - 16
