"""The launch of a dispatch (kazan_compute_launch, what vkCmdDispatch records):
every workgroup is in exactly one block, and no dimension has more threads than
a launch takes (2^32 - 1) where the workgroups' own shape has fewer."""
import ctypes

import pytest

U3 = ctypes.c_uint32 * 3
MOST_THREADS = 2**32 - 1


def _launch(driver, local, most, groups):
    grid, block = U3(), U3()
    per = driver.lib.kazan_compute_launch(U3(*local), ctypes.c_uint32(most), U3(*groups), grid, block)
    return per, tuple(grid), tuple(block)


@pytest.mark.parametrize("local", [(64, 1, 1), (1, 1, 1), (8, 8, 1), (4, 4, 4), (3, 5, 2), (1, 256, 1), (1, 1, 64)])
@pytest.mark.parametrize("x", [1, 7, 31, 32, 33, 2047, 2048, 65535, 2**24, 2**24 + 1, 2**26 - 1, 2**31])
def test_blocks_cover_the_groups(driver, local, x):
    n = local[0] * local[1] * local[2]
    most = max(1, 512 // n)
    if x * local[0] > MOST_THREADS:
        pytest.skip("more threads than a launch takes in the workgroups' own shape")
    per, grid, block = _launch(driver, local, most, (x, 3, 2))
    assert 1 <= per <= most
    assert grid[1:] == (3, 2)
    assert (grid[0] - 1) * per < x <= grid[0] * per
    assert block == (local if per == 1 else (n * per, 1, 1))
    assert all(g * b <= MOST_THREADS for g, b in zip(grid, block))
    # several a block wherever the rule allows it
    fits = x >= 4 * most and -(-x // most) * most * n <= MOST_THREADS
    assert per == (most if fits else 1)
