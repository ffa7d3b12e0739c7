"""Where the (triangle, tile) pairs are written from: chunks of 1,024
triangles, by their lanes when the chunk has at most two pairs a triangle,
else 1,024 pairs at a time on workgroups of their own. Triangle counts at the
edges of binning blocks and chunks, large triangles (hundreds of tiles each)
alone, among small ones and after a chunk of small ones, and a list storage
that ends within a chunk of large ones; clipped triangles, whose pieces are
entries of their own, at one and four samples and past the storage, against
the oracle through the Vulkan C ABI at every tile size the tuner tries. The
bar is the parity suite's: counts equal, coverage and depth bit-exact,
colour within 1 LSB.
"""
import numpy as np
import pytest

from kazan_amd.scenes import generators as g
from scene_kit import scene_from_pixels
from test_gpu_parity import check_parity

pytestmark = pytest.mark.gpu

W, H = 256, 128


_CTX = {}


@pytest.fixture(params=["balanced", "plain"])
def rctx(request, driver, monkeypatch):
    """A device of each pipeline form that bins by the radix sort."""
    from kazan_amd.scenes.renderer import Context
    if request.param not in _CTX:
        monkeypatch.setenv("KAZAN_PIPELINE", request.param)
        monkeypatch.setenv("KAZAN_BINNING", "radix")
        _CTX[request.param] = Context(driver)
    return _CTX[request.param]


def _scene(n, large):
    """n triangles of about a pixel, those in `large` over most of the target."""
    rng = np.random.default_rng(n)
    c = np.stack([rng.uniform(0, W, n), rng.uniform(0, H, n)], 1)
    tris = c[:, None, :] + rng.uniform(-1, 1, (n, 3, 2))
    at = np.asarray(large, int)
    tris[at] = np.stack([rng.uniform(-20, W + 20, (len(at), 3)), rng.uniform(-20, H + 20, (len(at), 3))], 2)
    s = scene_from_pixels(np.round(tris * 16) / 16, W, H, colors=rng.random((n, 3, 4)), z=rng.random((n, 3)))
    s.blend = (1, g.BLEND_SRC_ALPHA, g.BLEND_ONE_MINUS_SRC_ALPHA, 0, g.BLEND_ONE, g.BLEND_ONE_MINUS_SRC_ALPHA, 0)
    return s


@pytest.mark.parametrize("n,large", [
    (1, [0]), (65, range(65)), (255, [0, 254]), (257, range(0, 257, 3)), (1023, [1022]), (1025, [1024]),
    (2049, range(1020, 1030)), (5000, range(1024, 2048)), (5000, range(0, 5000, 40)),
])
def test_pairs_of_large_and_small(rctx, oracle, n, large):
    for frames in (1, 4):  # (the balanced form's first frames have its tile sizes, 16, 8, 32, 64 px)
        check_parity(rctx, oracle, _scene(n, large), frames=frames)


@pytest.mark.parametrize("form", ["balanced", "plain"])
def test_cut_within_large_triangles(driver, monkeypatch, oracle, form):
    from kazan_amd.scenes.renderer import Context
    monkeypatch.setenv("KAZAN_PIPELINE", form)
    monkeypatch.setenv("KAZAN_BINNING", "radix")
    monkeypatch.setenv("KAZAN_LIST_CAPACITY_LIMIT", "30000")
    st, _, _ = check_parity(Context(driver), oracle, _scene(6000, range(2000, 3500)), frames=2)
    assert st["list_overflow"] >= 1


@pytest.mark.parametrize("form", ["balanced", "plain"])
def test_clip_pieces_with_radix_binning(driver, monkeypatch, oracle, form):
    from kazan_amd.scenes.renderer import Context
    monkeypatch.setenv("KAZAN_PIPELINE", form)
    monkeypatch.setenv("KAZAN_BINNING", "radix")
    ctx = Context(driver)
    for s in (g.camera_inside(4000, 400, 256, 192), g.camera_inside(1000, 100, 128, 96, samples=4)):
        for frames in (1, 4):
            check_parity(ctx, oracle, s, frames=frames)
    monkeypatch.setenv("KAZAN_LIST_CAPACITY_LIMIT", "3000")
    st, _, _ = check_parity(Context(driver), oracle, g.camera_inside(600, 600, 256, 256), frames=2)
    assert st["list_overflow"] >= 1
