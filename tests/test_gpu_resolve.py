"""Where a 4x colour attachment is resolved: in the raster of the render
pass's last batch where that batch writes every pixel of it, else by a launch
of its own. A pass without draws that resolves an earlier pass's attachment
into an image that pass sampled, several batches in a pass, and a render area
smaller than the framebuffer, against the oracle through the Vulkan C ABI. The
bar is the parity suite's: depth bit-exact, colours within 1 LSB.
"""
import ctypes

import numpy as np
import pytest

from kazan_amd import vk
from kazan_amd.scenes import generators as g
from test_gpu_parity import COLOR_TOL_LSB, mctx  # noqa: F401  (the per-form device fixture)

pytestmark = pytest.mark.gpu

_ref = ctypes.byref


def _frame():
    """A renderer whose passes the test records."""
    from kazan_amd.scenes.renderer import SceneRenderer

    class Frame(SceneRenderer):
        def _record(self):
            self.cb = self.ctx.command_buffer()

        def render_pass(self, load, resolve):
            """(render pass, framebuffer): colour and depth with load op
            `load`, the colour resolved into the view `resolve` (or not)."""
            d, dev, s = self.ctx.d, self.ctx.device, self.s
            gen = vk.IMAGE_LAYOUT_GENERAL
            atts = [vk.VkAttachmentDescription(0, f, s.samples, load, 0, 2, 1, gen, gen)
                    for f in (vk.FORMAT_R8G8B8A8_UNORM, vk.FORMAT_D32_SFLOAT)]
            atts += [vk.VkAttachmentDescription(0, vk.FORMAT_R8G8B8A8_UNORM, 1, 2, 0, 2, 1, gen, gen)] if resolve else []
            arr = (vk.VkAttachmentDescription * len(atts))(*atts)
            refs = [vk.VkAttachmentReference(i, gen) for i in range(3)]
            sub = vk.VkSubpassDescription(0, 0, 0, None, 1, ctypes.pointer(refs[0]),
                                          ctypes.pointer(refs[2]) if resolve else None, ctypes.pointer(refs[1]), 0, None)
            ci = vk.VkRenderPassCreateInfo(vk.ST_RENDER_PASS_CREATE_INFO, None, 0, len(atts), arr, 1,
                                           ctypes.pointer(sub), 0, None)
            rp, fb = vk.Handle(), vk.Handle()
            d.check("vkCreateRenderPass", dev, _ref(ci), None, _ref(rp))
            vs = [self.color[2], self.depth[2]] + ([resolve] if resolve else [])
            fci = vk.VkFramebufferCreateInfo(vk.ST_FRAMEBUFFER_CREATE_INFO, None, 0, rp, len(vs),
                                             (vk.Handle * len(vs))(*vs), s.width, s.height, 1)
            d.check("vkCreateFramebuffer", dev, _ref(fci), None, _ref(fb))
            return rp, fb

        def record_pass(self, rp, fb, draws, rebind=False):
            d, s, cb = self.ctx.d, self.s, self.cb
            clears = (vk.VkClearValue * 2)()
            for k in range(4):
                clears[0].color.float32[k] = s.clear_color[k]
            clears[1].depthStencil.depth = s.clear_depth
            a = s.render_area or (0, 0, s.width, s.height)
            rbi = vk.VkRenderPassBeginInfo(vk.ST_RENDER_PASS_BEGIN_INFO, None, rp, fb,
                                           vk.VkRect2D(vk.VkOffset2D(a[0], a[1]), vk.VkExtent2D(a[2], a[3])), 2, clears)
            d.vkCmdBeginRenderPass(cb, _ref(rbi), 0)
            for i, dr in enumerate(draws):
                if i == 0 or rebind:
                    d.vkCmdBindPipeline(cb, 0, self.pipeline)
                if i == 0:
                    d.vkCmdBindVertexBuffers(cb, 0, 1, (vk.Handle * 1)(self.vbuf[0]), (ctypes.c_uint64 * 1)(0))
                    if self.desc_set is not None:
                        d.vkCmdBindDescriptorSets(cb, 0, self.layout, 0, 1, (vk.Handle * 1)(self.desc_set), 0, None)
                    if self.ibuf is not None:
                        d.vkCmdBindIndexBuffer(cb, self.ibuf[0], 0, vk.INDEX_TYPE_UINT32)
                if dr.get("mvp") is not None:
                    m = np.ascontiguousarray(dr["mvp"], np.float32)
                    d.vkCmdPushConstants(cb, self.layout, vk.SHADER_STAGE_VERTEX, 0, 64, m.ctypes.data)
                if self.ibuf is not None:
                    d.vkCmdDrawIndexed(cb, dr["count"], 1, dr["first"], dr["vertex_offset"], 0)
                else:
                    d.vkCmdDraw(cb, dr["count"], 1, dr["first"], 0)
            d.vkCmdEndRenderPass(cb)

    return Frame


def _check(r, oracle, area=None):
    c, d, res = r.read_back()
    oc, od, ores, ost = oracle.render(r.s)
    x, y, w, h = area or (0, 0, r.s.width, r.s.height)
    at = np.s_[y:y + h, x:x + w]
    np.testing.assert_array_equal(d[at].view(np.uint32), od[at].view(np.uint32))
    assert np.abs(c[at].astype(np.int16) - oc[at].astype(np.int16)).max() <= COLOR_TOL_LSB
    assert np.abs(res[at].astype(np.int16) - ores[at].astype(np.int16)).max() <= COLOR_TOL_LSB
    return ost


def test_pass_without_draws_resolves_into_a_sampled_image(mctx, oracle):
    """The first pass's raster must not write what its other tiles sample."""
    s = g.jittered_grid(64, 64, 256, 256, 256)  # (the texture has the framebuffer's size)
    s.samples = 4
    for resolved in (False, True):
        r = _frame()(mctx, s)
        r.resolve = r.tex
        mctx.begin(r.cb)
        r.record_pass(*r.render_pass(vk.ATTACHMENT_LOAD_OP_CLEAR, None), s.draws)
        if resolved:
            r.record_pass(*r.render_pass(vk.ATTACHMENT_LOAD_OP_LOAD, r.tex[2]), [])
        mctx.d.check("vkEndCommandBuffer", r.cb)
        st = r.render(1)
        if not resolved:
            launches = st["launches"]
    assert st["launches"] == launches + 1  # the resolve is one of its own
    ost = _check(r, oracle)
    assert st["fragments"] == ost["fragments"]


@pytest.mark.parametrize("rebind", [False, True])
def test_batches_of_a_pass(mctx, oracle, rebind):
    """Draws after the first bind (or, in the plain form, at all) are batches
    of their own: the resolve is of what the last leaves."""
    s = g.stress_4k(5, 3000, 200, 136, 4)
    r = _frame()(mctx, s)
    mctx.begin(r.cb)
    r.record_pass(*r.render_pass(vk.ATTACHMENT_LOAD_OP_CLEAR, r.resolve[2]), s.draws, rebind)
    mctx.d.check("vkEndCommandBuffer", r.cb)
    for frame in range(4):
        st = r.render(1)
        ost = _check(r, oracle)
        assert st["fragments"] == ost["fragments"], frame


def test_partial_area(mctx, oracle):
    s = g.stress_4k(4, 3000, 200, 136, 4)
    s.render_area = s.scissor = (24, 16, 120, 96)
    r = _frame()(mctx, s)
    mctx.begin(r.cb)
    r.record_pass(*r.render_pass(vk.ATTACHMENT_LOAD_OP_CLEAR, r.resolve[2]), s.draws)
    mctx.d.check("vkEndCommandBuffer", r.cb)
    st = r.render(2)
    ost = _check(r, oracle, s.render_area)
    assert st["fragments"] == 2 * ost["fragments"]
