"""What a Q4_0 product asks of its stream's scratch (mi355x_q4_0_scratch_bytes), which cannot grow while the stream is captured. Runs without a GPU."""
import pytest

from mimir_amd import capi


@pytest.mark.parametrize("n", [64, 1000, 4096, 14336, 32768])
@pytest.mark.parametrize("k", [64, 1024, 4096, 4160, 14336, 20480])
def test_no_call_asks_for_more_than_one_with_more_rows(n, k):
    """Run once at its largest size, a call may be captured at any smaller one."""
    lib = capi.load()
    rows = [*range(1, 2200), *range(2200, 9000, 61), 65535]
    sizes = [lib.mi355x_q4_0_scratch_bytes(m, n, k) for m in rows]
    assert sizes[-1] > 0
    drops = [(a, b, x, y) for a, b, x, y in zip(rows, rows[1:], sizes, sizes[1:]) if y < x]
    assert not drops, drops[:4]
