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


@pytest.mark.parametrize("n,k", [(64, 64), (4096, 4096), (14336, 4096), (200000, 4096), (14336, 12288), (5120, 320), (64, 20480)])
def test_rows_of_one_mib_in_fixed_point_stay_within_a_first_block(n, k):
    """A stream's block of 19 MiB, which its first call leaves, holds whatever a call below the panel's 256 rows takes whose rows fill no more than 1 MiB in
    fixed point, one by one (3 1/8 bytes an element) or as the row kernel's groups of eight (1088 bytes a block of 32). mi355x_qgemv_noalloc has as much."""
    lib = capi.load()
    rows = [m for m in range(2, 256) if m * (3 * k + k // 8) <= 1 << 20 or (m + 7) // 8 * (k // 32) * 1088 <= 1 << 20]
    assert rows and max(lib.mi355x_q4_0_scratch_bytes(m, n, k) for m in rows) <= 19 << 20


def test_what_only_the_row_kernel_takes_asks_for_no_more_than_its_rows():
    """By a small matrix W is never read where it lies, nor by one whose K is no whole pairs of blocks."""
    lib = capi.load()
    for m in (16, 64, 200, 256):
        assert lib.mi355x_q4_0_scratch_bytes(m, 512, 1024) <= (m + 7) // 8 * (1024 // 32) * 1088
        assert lib.mi355x_q4_0_scratch_bytes(m, 14336, 4096 + 32) == 0
