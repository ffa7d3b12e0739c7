"""Which batches are binned by gathering (kazan_gather_binning): those whose
squares, segments and density leave it ahead of the radix sort, at each tile
size."""
import pytest

GATHER = [  # triangles, width, height, tile size
    (256, 64, 64, 8), (256, 64, 64, 64), (1024, 256, 256, 8), (1024, 256, 256, 16), (11834, 1023, 575, 16),
    (65536, 1280, 720, 16), (65536, 1920, 1080, 16), (65536, 2560, 1440, 16), (8192, 3840, 2160, 16),
    (65536, 640, 480, 16), (65536, 640, 480, 8), (65536, 256, 256, 8), (16384, 128, 128, 8), (8192, 1280, 720, 8),
    (32768, 1280, 720, 32), (8192, 3840, 2160, 32), (2048, 64, 64, 32), (16384, 1920, 1080, 64),
]
RADIX = [
    (65537, 1280, 720, 16), (65536, 3440, 1440, 16), (16384, 3840, 2160, 16), (65536, 3840, 2160, 16),
    (65536, 1280, 720, 8), (8192, 1920, 1080, 8), (65536, 256, 256, 16), (65536, 128, 128, 8), (16384, 64, 64, 16),
    (65536, 1280, 720, 32), (16384, 640, 480, 32), (32768, 1920, 1080, 64), (1, 16384, 16384, 16),
]


@pytest.mark.parametrize("case", GATHER)
def test_gathered(driver, case):
    assert driver.lib.kazan_gather_binning(*case) == 1


@pytest.mark.parametrize("case", RADIX)
def test_sorted(driver, case):
    assert driver.lib.kazan_gather_binning(*case) == 0


def test_limits(driver):
    f = driver.lib.kazan_gather_binning
    assert f(100, 64, 64, 12) == -1
    for tile in (8, 16, 32, 64):
        assert f(1, 1, 1, tile) == 1
        assert f(2**32 - 1, 16384, 16384, tile) == 0
        for w, h in ((64, 64), (640, 480), (1920, 1080), (16384, 16384)):
            last = 1
            for n in range(1, 70000, 997):  # past the line it stays past it
                now = f(n, w, h, tile)
                assert now <= last, (n, w, h, tile)
                last = now
