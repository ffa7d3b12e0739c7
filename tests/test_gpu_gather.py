"""Gather binning: every tile collects its list from its 128 px square's
triangles. On devices that use it wherever its tables fit (also where the rule
would sort), but for one test of the rule itself. Triangle counts at the edges of a
2,048-triangle segment, a block of tiles with more candidates than its
workgroup holds (6,144), a square with more triangles than its coarse list
takes (its segments are then tested one by one), the largest batch it takes
and one triangle more (radix binning), and a list storage that is too small
(its tiles scan every triangle), clip pieces included, against the oracle
through the Vulkan C ABI. The bar is the parity suite's: counts equal,
coverage and depth bit-exact, colour within 1 LSB.
"""
import numpy as np
import pytest

from kazan_amd.scenes import generators as g
from scene_kit import scene_from_pixels
from test_gpu_parity import check_parity

pytestmark = pytest.mark.gpu

_CTX = {}


@pytest.fixture(params=["balanced", "plain"])
def mctx(request, driver, monkeypatch):
    """A device of each pipeline form that gathers."""
    from kazan_amd.scenes.renderer import Context
    if request.param not in _CTX:
        monkeypatch.setenv("KAZAN_PIPELINE", request.param)
        monkeypatch.setenv("KAZAN_BINNING", "gather")
        _CTX[request.param] = Context(driver)
    return _CTX[request.param]


def _scene(n, w, h, box, size=1.0, large=()):
    """n triangles of about `size` px with centres in box, those in `large` over most of the target."""
    rng = np.random.default_rng(n)
    x0, y0, x1, y1 = box
    c = np.stack([rng.uniform(x0, x1, n), rng.uniform(y0, y1, n)], 1)
    tris = c[:, None, :] + rng.uniform(-size, size, (n, 3, 2))
    at = np.asarray(large, int)
    tris[at] = np.stack([rng.uniform(-20, w + 20, (len(at), 3)), rng.uniform(-20, h + 20, (len(at), 3))], 2)
    s = scene_from_pixels(np.round(tris * 16) / 16, w, h, colors=rng.random((n, 3, 4)), z=rng.random((n, 3)))
    s.blend = (1, g.BLEND_SRC_ALPHA, g.BLEND_ONE_MINUS_SRC_ALPHA, 0, g.BLEND_ONE, g.BLEND_ONE_MINUS_SRC_ALPHA, 0)
    return s


@pytest.mark.parametrize("n", [1, 2047, 2048, 2049, 4100])
def test_segment_edges(mctx, oracle, n):
    s = _scene(n, 256, 128, (0, 0, 256, 128), large=range(0, n, 97))
    for frames in (1, 2, 3, 4):  # (the balanced form's first frames have its tile sizes, 16, 8, 32, 64 px)
        check_parity(mctx, oracle, s, frames=frames)


def test_more_candidates_than_are_held(mctx, oracle):
    check_parity(mctx, oracle, _scene(30_000, 256, 256, (100, 100, 124, 124), large=range(0, 30_000, 500)), frames=2)


def test_square_past_its_coarse_list(mctx, oracle):
    # 16 x 4 squares: a square's list takes 32 * 20,000 / 64 = 10,000 triangles
    check_parity(mctx, oracle, _scene(20_000, 2048, 512, (260, 130, 380, 250)), frames=2)


@pytest.mark.parametrize("n", [65_536, 65_537])
def test_largest_batch(mctx, oracle, n):
    check_parity(mctx, oracle, _scene(n, 512, 256, (0, 0, 512, 256)), frames=2)


@pytest.mark.parametrize("form", ["balanced", "plain"])
def test_storage_too_small(driver, monkeypatch, oracle, form):
    from kazan_amd.scenes.renderer import Context
    monkeypatch.setenv("KAZAN_PIPELINE", form)
    monkeypatch.setenv("KAZAN_BINNING", "gather")
    monkeypatch.setenv("KAZAN_LIST_CAPACITY_LIMIT", "1000")
    ctx = Context(driver)
    for s in (_scene(5000, 256, 128, (0, 0, 256, 128), large=range(0, 5000, 50)), g.camera_inside(300, 300, 256, 192)):
        st, _, _ = check_parity(ctx, oracle, s, frames=2)
        assert st["list_overflow"] >= 1


def test_rule(driver, monkeypatch, oracle):
    """Either side of the rule's lines, at one tile size: the launches are those of the binning it names."""
    from kazan_amd.scenes.renderer import Context
    monkeypatch.setenv("KAZAN_AUTOTUNE", "0")
    monkeypatch.setenv("KAZAN_TILE_SHIFT", "4")
    ctxs = {}
    for binning in (None, "radix", "gather"):
        with monkeypatch.context() as m:
            if binning:
                m.setenv("KAZAN_BINNING", binning)
            ctxs[binning] = Context(driver)
    for n, w, h in ((4096, 128, 128), (4097, 128, 128), (3000, 2048, 2048), (3000, 4096, 4096)):
        s = _scene(n, w, h, (0, 0, w, h), size=4.0)
        launches = {b: check_parity(c, oracle, s)[0]["launches"] for b, c in ctxs.items()}
        named = "gather" if driver.lib.kazan_gather_binning(n, w, h, 16) else "radix"
        assert launches["gather"] != launches["radix"]
        assert launches[None] == launches[named], (n, w, h)
