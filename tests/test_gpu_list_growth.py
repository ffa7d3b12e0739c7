"""The growth of the tile lists' storage while later frames are in flight, in
every binning form: the storage follows the largest batch, not the sum of the
frames since it was last looked at, and the wait on the first frame whose lists
overflowed makes the room. A frame whose lists overflow is drawn by a scan of
every triangle: its pixels are the same either way.
"""
import ctypes

import numpy as np
import pytest

from kazan_amd import vk
from kazan_amd.scenes import generators as g

pytestmark = pytest.mark.gpu

_ref = ctypes.byref


def _fence(ctx):
    f = vk.Handle()
    ctx.d.check("vkCreateFence", ctx.device, _ref(vk.VkFenceCreateInfo(vk.ST_FENCE_CREATE_INFO, None, 0)), None, _ref(f))
    return (vk.Handle * 1)(f)


def _submit(ctx, cb, fence):
    ctx.d.check("vkResetFences", ctx.device, 1, fence)
    si = vk.VkSubmitInfo(vk.ST_SUBMIT_INFO, None, 0, None, None, 1, (vk.Handle * 1)(cb), 0, None)
    ctx.d.check("vkQueueSubmit", ctx.queue, 1, _ref(si), fence[0])


def _in_flight(ctx, cb, frames, depth=3):
    """Submits cb `frames` times, waiting for each with depth - 1 after it in flight."""
    fences = [_fence(ctx) for _ in range(depth)]
    for k in range(frames):
        if k >= depth:
            ctx.d.check("vkWaitForFences", ctx.device, 1, fences[k % depth], 1, 2**63)
        _submit(ctx, cb, fences[k % depth])
    ctx.wait_idle()
    for f in fences:
        ctx.d.vkDestroyFence(ctx.device, f[0], None)


@pytest.mark.parametrize("form", ["balanced", "plain"])
@pytest.mark.parametrize("binning", [None, "radix", "sort"])
def test_growth_with_frames_in_flight(driver, monkeypatch, oracle, form, binning):
    from kazan_amd.scenes.renderer import Context, SceneRenderer
    monkeypatch.setenv("KAZAN_PIPELINE", form)
    monkeypatch.setenv("KAZAN_AUTOTUNE", "0")
    if binning:
        monkeypatch.setenv("KAZAN_BINNING", binning)
    ctx = Context(driver)
    # about 430,000 and twice as many pairs, where 72,000 and 78,000 fit at first
    s, t = g.random_triangles(1500, 512, 512, seed=3), g.random_triangles(3000, 512, 512, seed=4)
    r = SceneRenderer(ctx, s)
    _in_flight(ctx, r.cb, 9)
    _in_flight(ctx, r.cb, 9)  # (the room is there by now)
    st = ctx.stats()
    assert st["list_overflow"] == 0 and st["list_entries"] % st["batches"] == 0
    pairs = st["list_entries"] // st["batches"]
    assert pairs > 100_000
    q = SceneRenderer(ctx, t)
    st = q.render(1)  # 5/4 of the smaller scene's pairs are fewer than this one's
    assert st["list_entries"] > 1.5 * pairs and st["list_overflow"] == 1
    st = q.render(1)
    assert st["list_overflow"] == 0
    oc, od, _, _ = oracle.render(t)
    c, d, _ = q.read_back()
    np.testing.assert_array_equal(d.view(np.uint32), od.view(np.uint32))
    assert np.abs(c.astype(np.int16) - oc.astype(np.int16)).max() <= 1


@pytest.mark.parametrize("binning", [None, "radix", "sort"])
def test_the_first_wait_makes_the_room(driver, monkeypatch, binning):
    """Twelve frames with two more in flight: the first of them overflow, not all."""
    from kazan_amd.scenes.renderer import Context, SceneRenderer
    monkeypatch.setenv("KAZAN_AUTOTUNE", "0")
    if binning:
        monkeypatch.setenv("KAZAN_BINNING", binning)
    ctx = Context(driver)
    r = SceneRenderer(ctx, g.random_triangles(1500, 512, 512, seed=3))
    fences = [_fence(ctx) for _ in range(3)]
    for k in range(12):
        if k >= 3:
            ctx.d.check("vkWaitForFences", ctx.device, 1, fences[k % 3], 1, 2**63)
        _submit(ctx, r.cb, fences[k % 3])
    # (the wait on the first frame collected the three in flight: none since)
    assert ctx.stats()["list_overflow"] == 0
