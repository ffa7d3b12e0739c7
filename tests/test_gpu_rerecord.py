"""A command buffer recorded anew for every frame, as a game does: its draw
records' memory is kept over recordings (of more draws than before, and of
fewer), each frame has the draws of its recording, and a recording that is
submitted again after all is tuned and replayed as any other. A reset that asks
for it gives the memory back. The bar is the parity suite's: counts equal, depth
bit-exact, colour within 1 LSB.
"""
import ctypes
import os

import numpy as np
import pytest

from kazan_amd import vk
from kazan_amd.scenes import generators as g

pytestmark = pytest.mark.gpu


def _check(r, oracle, st, frames):
    oc, od, _, ost = oracle.render(r.s)
    assert st["fragments"] == frames * ost["fragments"]
    c, d, _ = r.read_back()
    np.testing.assert_array_equal(d.view(np.uint32), od.view(np.uint32))
    assert np.abs(c.astype(np.int16) - oc.astype(np.int16)).max() <= 1


@pytest.mark.parametrize("form", ["balanced", "plain"])
def test_recorded_for_every_frame(driver, monkeypatch, oracle, form):
    from kazan_amd.scenes.renderer import Context, SceneRenderer
    monkeypatch.setenv("KAZAN_PIPELINE", form)
    ctx = Context(driver)
    s = g.zipf_draws(200, 20_000, 320, 180)
    draws = s.draws
    r = SceneRenderer(ctx, s)
    cb = r.cb
    for k in (2, 5, 60, 200, 3):
        s.draws = draws[:k]
        with monkeypatch.context() as m:
            m.setattr(ctx, "command_buffer", lambda: cb)
            r._record()
        _check(r, oracle, r.render(1), 1)
    _check(r, oracle, r.render(40), 40)


def test_first_submission_loads_no_other_kernels(driver, monkeypatch, tmp_path):
    """A recording's first submission, often its only one, draws with the tile
    size its pipeline was created with: a new pipeline's other sizes are
    compiled (and loaded) by the submissions after it."""
    from kazan_amd.scenes.renderer import Context, SceneRenderer
    monkeypatch.setenv("KAZAN_PIPELINE", "balanced")
    monkeypatch.setenv("KAZAN_PIPELINE_CACHE", str(tmp_path))
    ctx = Context(driver)
    s = g.zipf_draws(20, 2000, 320, 180)
    r = SceneRenderer(ctx, s)
    created = sorted(os.listdir(tmp_path))
    assert len(created) == 1
    for _ in range(3):  # command buffers allocated, submitted once and freed
        r.render(1)
        assert sorted(os.listdir(tmp_path)) == created
        r._record()
    r.render(2)
    assert len(os.listdir(tmp_path)) == 2


def _free_bytes():
    """Free device memory, by the HIP runtime the driver is linked with."""
    path = next(ln.split()[-1] for ln in open("/proc/self/maps") if "libamdhip64" in ln and "/opt/rocm" in ln)
    hip, free, total = ctypes.CDLL(path), ctypes.c_size_t(), ctypes.c_size_t()
    assert hip.hipDeviceSynchronize() == 0
    assert hip.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    return free.value


@pytest.mark.parametrize("reset", ["vkResetCommandBuffer", "vkResetCommandPool"])
def test_reset_releases(driver, oracle, reset):
    """500,000 instances are draw records of over 100 MB, kept over a plain reset."""
    from kazan_amd.scenes.renderer import Context, SceneRenderer
    ctx = Context(driver)
    s = g.random_triangles(100, 96, 64, seed=5)
    r = SceneRenderer(ctx, s)
    d, many = ctx.d, 500_000
    cb = ctx.command_buffer()

    def record():
        ctx.begin(cb)
        rbi = vk.VkRenderPassBeginInfo(vk.ST_RENDER_PASS_BEGIN_INFO, None, r.rp, r.fb,
                                       vk.VkRect2D(vk.VkOffset2D(0, 0), vk.VkExtent2D(s.width, s.height)), 2,
                                       (vk.VkClearValue * 2)())
        d.vkCmdBeginRenderPass(cb, ctypes.byref(rbi), 0)
        d.vkCmdBindPipeline(cb, 0, r.pipeline)
        d.vkCmdBindVertexBuffers(cb, 0, 1, (vk.Handle * 1)(r.vbuf[0]), (ctypes.c_uint64 * 1)(0))
        d.vkCmdDraw(cb, 3, many, 0, 0)
        d.vkCmdEndRenderPass(cb)
        d.check("vkEndCommandBuffer", cb)

    def reset_with(flags):
        d.check(reset, *((cb, flags) if reset == "vkResetCommandBuffer" else (ctx.device, ctx.pool, flags)))

    before = _free_bytes()
    record()
    assert before - _free_bytes() > 100 << 20
    reset_with(0)
    assert before - _free_bytes() > 100 << 20
    reset_with(1)
    assert before - _free_bytes() < 16 << 20
    record()  # and again, in memory of its own
    reset_with(1)
    r._record()
    _check(r, oracle, r.render(2), 2)
