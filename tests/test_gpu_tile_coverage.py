"""Coverage relative to the tile (KzTileCov in the raster kernel): its 32-bit
thresholds against the oracle's 64-bit edge functions, through the Vulkan C
ABI. Triangles whose edges run to the guard band (their edge values reach
2^36, so a tile's thresholds saturate), edges through pixel centres (the
top-left rule at threshold 0 and 1, on tile corners), slivers, and large and
tiny triangles in one batch (64-bit and 32-bit thresholds side by side), at
every tile size the tuner tries. The bar is the parity suite's: counts equal,
coverage and depth bit-exact, colour within 1 LSB.
"""
import numpy as np
import pytest

from kazan_amd.scenes import generators as g
from scene_kit import scene_from_pixels
from test_gpu_parity import check_parity, mctx  # noqa: F401  (the per-form device fixture)

pytestmark = pytest.mark.gpu

W, H = 256, 128  # powers of two: pixel coordinates reach the rasteriser exactly


def _edges_far_away(rng):
    """Triangles with vertices up to 8,000 px off-screen through the target."""
    p = rng.uniform(-7900, 7900, (40, 3, 2))
    p[:, 0] = np.stack([rng.uniform(0, W, 40), rng.uniform(0, H, 40)], 1)
    return np.round(p * 16) / 16


def _through_centres(rng):
    """Edges on pixel centres, pixel corners and tile corners."""
    x, y = rng.integers(0, W // 8, (60, 3)) * 8, rng.integers(0, H // 8, (60, 3)) * 8
    return np.stack([x, y], 2) + rng.choice([0.0, 0.5], (60, 1, 1))


def _slivers(rng):
    a = np.stack([rng.uniform(0, W, 60), rng.uniform(0, H, 60)], 1)
    d = rng.uniform(-200, 200, (60, 2))
    return np.round(np.stack([a, a + d, a + d * 0.5 + 0.0625], 1) * 16) / 16


def _large_and_tiny(rng):
    big = _edges_far_away(rng)
    c = np.stack([rng.uniform(0, W, 400), rng.uniform(0, H, 400)], 1)
    tiny = np.round((c[:, None, :] + rng.uniform(-2, 2, (400, 3, 2))) * 16) / 16
    both = np.concatenate([big, tiny])
    return both[rng.permutation(len(both))]


@pytest.mark.parametrize("samples", [1, 4])
@pytest.mark.parametrize("make", [_edges_far_away, _through_centres, _slivers, _large_and_tiny])
def test_tile_relative_coverage(mctx, oracle, make, samples):
    rng = np.random.default_rng(17)
    tris = make(rng)
    n = len(tris)
    s = scene_from_pixels(tris, W, H, colors=rng.random((n, 3, 4)), z=rng.random((n, 3)), samples=samples)
    s.blend = (1, g.BLEND_SRC_ALPHA, g.BLEND_ONE_MINUS_SRC_ALPHA, 0, g.BLEND_ONE, g.BLEND_ONE_MINUS_SRC_ALPHA, 0)
    s.scissor = (3, 5, W - 10, H - 6)
    # (the balanced form draws its first frames with its tile sizes: 16, 8, 32 and, where they fit, 64 px)
    for frames in (1, 2, 3, 4):
        check_parity(mctx, oracle, s, frames=frames)
