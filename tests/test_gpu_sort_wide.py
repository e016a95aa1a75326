"""Sorts of states with a table of more than 2^20 cells: up to 12 tiles of 2,048
keys the scatter adds up the tiles' counts itself, of up to 2,048 digits each
(sort_keys, csrc/sort.hip)."""
import pytest

from test_gpu_sort_paths import TILE, check, cloud, ctx  # noqa: F401

pytestmark = pytest.mark.gpu


# side and cells' bits: digits of 4 and of 11 bits
@pytest.mark.parametrize("side,bits", [(0.04, 9), (9.5, 21)])
@pytest.mark.parametrize("n", [TILE + 1, 7 * TILE - 3, 12 * TILE, 12 * TILE + 1])
def test_counts_of_a_wide_table(ctx, n, side, bits):  # noqa: F811
    cells = check(ctx, cloud(n, side), steps=1, table_cap=1 << 22)
    assert cells.bit_length() == bits
