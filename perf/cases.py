"""What this driver's users have it do, at the sizes they have it done.

A case is one frame (or one compute dispatch) of an application: a command
buffer of draws submitted through vkQueueSubmit, its attachments the result.
Applications either record a command buffer once and submit it every frame
("static": a viewer, a benchmark, a simulation's output) or record it again
for each frame (family "dynamic": a game). `prepare` is the application's
loading screen: pipelines, buffers, textures, attachments and, for a command
buffer that stays, its first frames, over which the driver picks the
configuration it keeps for it. `run` is one frame.

The frame's results are the attachments, which stay in device memory: they
are handed out as tensors over that memory.
"""
import ctypes
import math

import numpy as np
import torch

from kazan_amd import vk
from kazan_amd.scenes import compute_shaders as cs
from kazan_amd.scenes import generators as g
from kazan_amd.scenes.compute import ComputeKernel
from kazan_amd.scenes.renderer import Context, SceneRenderer

BLEND = (1, g.BLEND_SRC_ALPHA, g.BLEND_ONE_MINUS_SRC_ALPHA, 0, g.BLEND_ONE, g.BLEND_ONE_MINUS_SRC_ALPHA, 0)


def listed():
    return [
        # the smallest frame: an icon or a thumbnail; all of it is launches and latency
        {"name": "icon_64", "family": "triangles", "n": 256, "width": 64, "height": 64},
        # large overlapping triangles in a small frame (the repository's first workload)
        {"name": "triangles_256", "family": "triangles", "n": 1024, "width": 256, "height": 256},
        # a small textured terrain in a window of odd size
        {"name": "grid_window", "family": "grid", "cols": 97, "rows": 61, "width": 1023, "height": 575, "tex": 300},
        # the headline: a dense textured, blended mesh at full HD
        {"name": "grid_1080p", "family": "grid", "cols": 512, "rows": 1024, "width": 1920, "height": 1080, "tex": 1024},
        # a particle cloud or point-like scan, most of it in the middle of the screen
        {"name": "cluster_4m_1080p", "family": "cluster", "n": 4_194_304, "width": 1920, "height": 1080},
        # near and far detail side by side: many tiny triangles, some larger
        {"name": "mixed_1080p", "family": "mixed", "n": 3_000_000, "coarse": 30_000, "width": 1920, "height": 1080},
        # a CAD or level scene: thousands of objects, a draw and a matrix each
        {"name": "zipf_4096_1440p", "family": "zipf", "draws": 4096, "n": 4_194_304, "width": 2560, "height": 1440},
        # the heaviest: 4K, four samples, eight lights per fragment
        {"name": "stress_4k_msaa4", "family": "phong", "draws": 2048, "n": 8_388_608, "width": 3840, "height": 2160},
        # the same shading at an ordinary size
        {"name": "phong_720p_msaa4", "family": "phong", "draws": 64, "n": 131_072, "width": 1280, "height": 720},
        # a camera inside the geometry: clipping, large and small triangles, an odd size
        {"name": "camera_inside", "family": "camera", "n": 40_000, "big": 400, "width": 1279, "height": 719},
        # a game's frame: its command buffer is recorded for every frame
        {"name": "dynamic_720p", "family": "dynamic", "draws": 64, "n": 65_536, "width": 1280, "height": 720},
        # a compute dispatch over a ragged number of elements
        {"name": "saxpy_16m", "family": "saxpy", "n": 16_777_229},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


_SIZES = ((640, 480), (1280, 720), (1366, 768), (1920, 1080), (2560, 1440))


def _window(rng, most=5):
    """A common resolution, or a window of any (odd) size."""
    if rng.random() < 0.5:
        return _SIZES[rng.randrange(most)]
    w, h = _SIZES[rng.randrange(most)]
    return int(w * rng.uniform(0.6, 1.0)) | 1, int(h * rng.uniform(0.6, 1.0)) | 1


def draw(rng):
    family = rng.choice(["triangles", "grid", "cluster", "mixed", "zipf", "phong", "camera", "dynamic", "saxpy"])
    w, h = _window(rng)
    if family == "triangles":
        w, h = _log(rng, 48, 640), _log(rng, 48, 480)
        return {"family": family, "n": _log(rng, 64, 8192), "width": w, "height": h}
    if family == "grid":
        return {"family": family, "cols": _log(rng, 24, 700), "rows": _log(rng, 24, 1024), "width": w, "height": h,
                "tex": _log(rng, 64, 1024)}
    if family == "cluster":
        return {"family": family, "n": _log(rng, 50_000, 4_000_000), "width": w, "height": h}
    if family == "mixed":
        n = _log(rng, 50_000, 3_000_000)
        return {"family": family, "n": n, "coarse": max(16, n // rng.randint(30, 300)), "width": w, "height": h}
    if family == "zipf":
        return {"family": family, "draws": _log(rng, 8, 4096), "n": _log(rng, 50_000, 4_000_000), "width": w, "height": h}
    if family == "phong":
        return {"family": family, "draws": _log(rng, 8, 1024), "n": _log(rng, 50_000, 4_000_000), "width": w, "height": h}
    if family == "camera":
        n = _log(rng, 3_000, 200_000)
        return {"family": family, "n": n, "big": max(8, n // rng.randint(20, 200)), "width": w, "height": h}
    if family == "dynamic":
        w, h = _window(rng, 4)
        return {"family": family, "draws": _log(rng, 2, 256), "n": _log(rng, 10_000, 500_000), "width": w, "height": h}
    return {"family": family, "n": _log(rng, 100_000, 60_000_000)}


# --- inputs ----------------------------------------------------------------


class _Uniform:
    """Uniform floats from the seed, on the GPU where there is one."""

    def __init__(self, seed):
        self.device = "cuda" if torch.cuda.is_available() else "cpu"
        self.gen = torch.Generator(device=self.device).manual_seed(seed)

    def __call__(self, *shape):
        return torch.rand(shape, generator=self.gen, device=self.device)


def _cluster_vertices(u, n, width, height, frac, sigma, radius, centre):
    """Triangles around normally distributed centres (and a uniform rest),
    as generators.gaussian_cluster describes them: pos4 + colour4."""
    nc = int(round(n * frac))
    a = torch.sqrt(-2.0 * torch.log(u(n).clamp_min(1e-7)))
    t = 2 * math.pi * u(n)
    c = torch.stack([width * (centre[0] + sigma * a * torch.cos(t)), height * (centre[1] + sigma * a * torch.sin(t))], 1)
    c[nc:] = u(n - nc, 2) * torch.tensor([float(width), float(height)], device=u.device)
    p = c[:, None, :] + (u(n, 3, 2) * 2 - 1) * radius
    v = torch.ones(n, 3, 8, device=u.device)
    v[:, :, 0] = p[:, :, 0] * (2.0 / width) - 1.0
    v[:, :, 1] = p[:, :, 1] * (2.0 / height) - 1.0
    v[:, :, 2] = u(n, 3)
    v[:, :, 4:8] = u(n, 3, 4)
    return v.reshape(n * 3, 8)


def _object_vertices(u, n, size, normals):
    """Small triangles over the unit cube, as generators.cube_meshes
    describes them: position and colour, or position and normal."""
    pos = (u(n, 1, 3) + (u(n, 3, 3) * 2 - 1) * size).reshape(n * 3, 3)
    if not normals:
        return torch.cat([pos, u(n * 3, 4)], 1)
    d = pos - 0.5
    return torch.cat([pos, d / d.norm(dim=1, keepdim=True).clamp_min(1e-6)], 1)


def _object_draws(case, seed):
    counts = g.zipf_counts(case["draws"], case["n"], seed=seed)
    draws, first = [], 0
    for d, n in enumerate(counts):
        draws.append(dict(count=int(3 * n), first=first, vertex_offset=0,
                          mvp=g.draw_mvp(seed + 1000 + d, case["width"] / case["height"])))
        first += int(3 * n)
    return draws, int(counts.sum())


def _scene(case, seed):
    family, w, h = case["family"], case["width"], case["height"]
    seed = int(seed) % (1 << 31)
    u = _Uniform(seed)
    if family == "triangles":
        return g.random_triangles(case["n"], w, h, seed)
    if family == "grid":
        return g.jittered_grid(case["cols"], case["rows"], w, h, case["tex"], seed)
    if family == "camera":
        return g.camera_inside(case["n"], case["big"], w, h, 4, 1, seed)
    if family in ("cluster", "mixed"):
        if family == "cluster":
            v = _cluster_vertices(u, case["n"], w, h, 0.9, 0.05, 0.92, (0.5, 0.5))
        else:
            v = torch.cat([_cluster_vertices(u, case["n"], w, h, 1.0, 0.05, 0.92, (0.3, 0.5)),
                           _cluster_vertices(u, case["coarse"], w, h, 1.0, 0.04, 10.0, (0.7, 0.5))])
        s = g.Scene(family, w, h, g.VS_POS4_COLOR4, g.FS_COLOR, v.cpu().numpy())
        s.blend = BLEND
        return s
    draws, n = _object_draws(case, seed)
    if family == "phong":
        v = _object_vertices(u, n, 0.008, True).cpu().numpy()
        s = g.Scene(family, w, h, g.VS_MVP_POS3_NORMAL3, g.FS_PHONG, v, draws=draws, samples=4)
        s.ubo, s.num_lights = g.phong_lights(8, seed + 21), 8
        s.clear_color = (0.0, 0.0, 0.0, 1.0)
        return s
    v = _object_vertices(u, n, 0.012, False).cpu().numpy()
    return g.Scene(family, w, h, g.VS_MVP_POS3_COLOR4, g.FS_COLOR, v, draws=draws)


# --- the application ---------------------------------------------------------

_context = None


def _app():
    """The application's Vulkan device: one for all its frames."""
    global _context
    if _context is None:
        _context = Context()
    return _context


class _Memory:
    """A tensor's view of a VkDeviceMemory (a non-dispatchable handle is its
    object's address, and the object begins with the allocation's). Keeps the
    owner of the allocation alive as long as a tensor is."""

    def __init__(self, owner, memory, shape, dtype):
        self.owner = owner
        address = ctypes.c_uint64.from_address(memory.value).value
        self.__cuda_array_interface__ = {"shape": shape, "typestr": dtype, "data": (address, False), "version": 2}


def _view(owner, memory, shape, dtype):
    return torch.as_tensor(_Memory(owner, memory, shape, dtype), device="cuda")


class _Frame(SceneRenderer):
    """A scene's Vulkan objects, freed with it."""

    def __init__(self, ctx, scene):
        super().__init__(ctx, scene)
        self.fences = []
        self.spare = []

    def outputs(self):
        s = self.s
        shape = (s.height, s.width, s.samples)
        out = {"color": _view(self, self.color[1], shape + (4,), "|u1"), "depth": _view(self, self.depth[1], shape, "<f4")}
        if self.resolve:
            out["resolved"] = _view(self, self.resolve[1], (s.height, s.width, 4), "|u1")
        return out

    def settle(self):
        """The loading screen of a command buffer that stays: frames until
        the driver has chosen its configuration."""
        caps, launches = ctypes.c_uint32(), ctypes.c_uint32()
        d, dev = self.ctx.d, self.ctx.device
        d.vkGetGraphStatsKAZAN(dev, ctypes.byref(caps), ctypes.byref(launches))
        before = caps.value
        for _ in range(100):
            self.ctx.submit(self.cb)
            d.vkGetGraphStatsKAZAN(dev, ctypes.byref(caps), ctypes.byref(launches))
            if caps.value > before:
                break

    def frames_in_flight(self, n):
        """n command buffers and fences, taken in turn by record_frame."""
        for _ in range(n):
            fence = vk.Handle()
            fci = vk.VkFenceCreateInfo(vk.ST_FENCE_CREATE_INFO, None, 0)
            self.ctx.d.check("vkCreateFence", self.ctx.device, ctypes.byref(fci), None, ctypes.byref(fence))
            self.fences.append(fence)
            self.spare.append(self.ctx.command_buffer())
        self.used = [False] * n
        self.turn = 0

    def record_frame(self):
        """Waits for the frame that last used this turn's command buffer,
        records the scene into it and submits it."""
        ctx, d, s, k = self.ctx, self.ctx.d, self.s, self.turn
        self.turn = (k + 1) % len(self.spare)
        cb, fence = self.spare[k], (vk.Handle * 1)(self.fences[k])
        if self.used[k]:
            d.check("vkWaitForFences", ctx.device, 1, fence, 1, 2**63)
            d.check("vkResetFences", ctx.device, 1, fence)
        self.used[k] = True
        ctx.begin(cb)
        clears = (vk.VkClearValue * 2)()
        for c in range(4):
            clears[0].color.float32[c] = s.clear_color[c]
        clears[1].depthStencil.depth = s.clear_depth
        rbi = vk.VkRenderPassBeginInfo(vk.ST_RENDER_PASS_BEGIN_INFO, None, self.rp, self.fb,
                                       vk.VkRect2D(vk.VkOffset2D(0, 0), vk.VkExtent2D(s.width, s.height)), 2, clears)
        d.vkCmdBeginRenderPass(cb, ctypes.byref(rbi), 0)
        d.vkCmdBindPipeline(cb, 0, self.pipeline)
        d.vkCmdBindVertexBuffers(cb, 0, 1, (vk.Handle * 1)(self.vbuf[0]), (ctypes.c_uint64 * 1)(0))
        for dr in s.draws:
            d.vkCmdPushConstants(cb, self.layout, vk.SHADER_STAGE_VERTEX, 0, 64, dr["mvp"].ctypes.data)
            d.vkCmdDraw(cb, dr["count"], 1, dr["first"], 0)
        d.vkCmdEndRenderPass(cb)
        d.check("vkEndCommandBuffer", cb)
        cbs = (vk.Handle * 1)(cb)
        si = vk.VkSubmitInfo(vk.ST_SUBMIT_INFO, None, 0, None, None, 1, cbs, 0, None)
        d.check("vkQueueSubmit", ctx.queue, 1, ctypes.byref(si), self.fences[k])

    def __del__(self):
        if not hasattr(self, "pipeline"):
            return
        ctx, d, dev = self.ctx, self.ctx.d, self.ctx.device
        d.vkDeviceWaitIdle(dev)
        for cb in [self.cb] + self.spare:
            d.vkFreeCommandBuffers(dev, ctx.pool, 1, (vk.Handle * 1)(cb))
        for fence in self.fences:
            d.vkDestroyFence(dev, fence, None)
        d.vkDestroyPipeline(dev, self.pipeline, None)
        for buf in [self.vbuf, self.ibuf, getattr(self, "ubo", None)]:
            if buf:
                ctx.destroy_buffer(buf)
        d.vkDestroyFramebuffer(dev, self.fb, None)
        for img in [self.color, self.depth, self.resolve, getattr(self, "tex", None)]:
            if img:
                d.vkDestroyImageView(dev, img[2], None)
                d.vkDestroyImage(dev, img[0], None)
                d.vkFreeMemory(dev, img[1], None)


class _Saxpy:
    """y = a x + y over storage buffers, recorded once."""

    def __init__(self, ctx, case, seed):
        x, y = _vectors(case, seed)
        n = case["n"]
        self.ctx, self.n = ctx, n
        self.x, self.y = ctx.device_buffer_with(x.cpu().numpy()), ctx.device_buffer_with(y.cpu().numpy())
        self.kernel = ComputeKernel(ctx, cs.cs_saxpy(), 2, push_bytes=8)
        self.kernel.bind([(self.x[0], 4 * n), (self.y[0], 4 * n)])
        self.cb = ctx.command_buffer()
        ctx.begin(self.cb)
        push = np.array([np.float32(A).view(np.uint32), n], np.uint32)
        self.kernel.record(self.cb, ((n + 63) // 64,), push=push)
        ctx.d.check("vkEndCommandBuffer", self.cb)

    def outputs(self):
        return {"y": _view(self, self.y[1], (self.n,), "<f4")}

    def __del__(self):
        if not hasattr(self, "cb"):
            return
        ctx = self.ctx
        ctx.d.vkDeviceWaitIdle(ctx.device)
        ctx.d.vkFreeCommandBuffers(ctx.device, ctx.pool, 1, (vk.Handle * 1)(self.cb))
        self.kernel.destroy()
        ctx.destroy_buffer(self.x)
        ctx.destroy_buffer(self.y)


A = 1e-3


def _vectors(case, seed):
    u = _Uniform(int(seed) % (1 << 31))
    return u(case["n"]) * 2 - 1, u(case["n"]) * 2 - 1


def prepare(case, seed):
    ctx = _app()
    if case["family"] == "saxpy":
        app = _Saxpy(ctx, case, seed)
    else:
        app = _Frame(ctx, _scene(case, seed))
        if case["family"] == "dynamic":
            app.frames_in_flight(3)
        else:
            app.settle()
    return {"app": app, "dynamic": case["family"] == "dynamic", "out": app.outputs()}


def run(state):
    app = state["app"]
    if state["dynamic"]:
        app.record_frame()
    else:
        app.ctx.submit(app.cb, wait=False)
    return state["out"]


# --- what a pass cannot do without -------------------------------------------


def _triangles(case):
    if case["family"] == "grid":
        return 2 * case["cols"] * case["rows"]
    n = min(case["n"], 65536 * case["draws"]) if "draws" in case else case["n"]  # (zipf_counts' largest draw)
    return n + case.get("coarse", 0) + case.get("big", 0)


def work(case):
    """Geometry, texture and per-draw data read once, the attachments written
    once. Operations: about 60 per triangle (setup) and 36 per vertex (a
    matrix), and what shading every pixel once takes."""
    if case["family"] == "saxpy":
        return {"bytes": 12 * case["n"], "flops": 2 * case["n"]}
    f, n, px = case["family"], _triangles(case), case["width"] * case["height"]
    if f == "grid":
        geometry = 20 * (case["cols"] + 1) * (case["rows"] + 1) + 12 * n + 4 * case["tex"] ** 2
    else:
        geometry = 3 * n * {"phong": 24, "zipf": 28, "dynamic": 28, "camera": 28}.get(f, 32) + 68 * case.get("draws", 1)
    target = px * (36 if f == "phong" else 8)
    return {"bytes": geometry + target, "flops": n * (60 + 3 * 36) + px * (8 * 40 if f == "phong" else 30)}


def tolerance(case):
    """Coverage, depth and the stored bytes are fixed by the rules the driver
    follows (fixed-point edges, single-precision depth in a stated order),
    and a dispatch by its shader's operations."""
    return "exact"


# --- in 64 bits --------------------------------------------------------------

_SAMPLES = {1: ((8, 8),), 4: ((6, 2), (14, 6), (2, 10), (10, 14))}


def _clip_positions(s, device):
    """Clip-space positions of the scene's triangles, (n, 3, 4), 64 bits."""
    v = torch.from_numpy(s.vertices).to(device).double()
    if s.vs == g.VS_POS4_COLOR4:
        p = v[:, :4]
    else:
        p = torch.cat([v[:, :3], torch.ones_like(v[:, :1])], 1)
    if s.draws[0].get("mvp") is not None:
        m = torch.from_numpy(np.stack([dr["mvp"] for dr in s.draws])).to(device).double().reshape(-1, 4, 4)
        counts = torch.tensor([dr["count"] for dr in s.draws], device=device)
        per = torch.repeat_interleave(torch.arange(len(s.draws), device=device), counts)
        out = torch.empty(len(p), 4, dtype=torch.float64, device=device)
        for a in range(0, len(p), 1 << 22):
            out[a:a + (1 << 22)] = torch.matmul(p[a:a + (1 << 22), None, :], m[per[a:a + (1 << 22)]])[:, 0]
        p = out
    if s.indices is not None:
        p = p[torch.from_numpy(s.indices.astype(np.int64)).to(device)]
    return p.reshape(-1, 3, 4)


def _depth(s, device):
    """The depth attachment (LESS from 1.0, nothing clipped): positions
    snapped to 1/16 pixel, whole-number edges, depth in 64 bits."""
    p = _clip_positions(s, device)
    w = p[:, :, 3]
    half = torch.tensor([s.width * 0.5, s.height * 0.5], device=device)
    ndc = (p[:, :, :2] / w[:, :, None]).float()  # the viewport transform is single precision by rule
    xy = torch.round((ndc * half + half) * 16.0).long()
    z = p[:, :, 2] / w
    x, y = xy[:, :, 0], xy[:, :, 1]
    x0 = (x.amin(1) >> 4).clamp_min(0)
    x1 = (x.amax(1) >> 4).clamp_max(s.width - 1)
    y0 = (y.amin(1) >> 4).clamp_min(0)
    y1 = (y.amax(1) >> 4).clamp_max(s.height - 1)
    area = (x[:, 1] - x[:, 0]) * (y[:, 2] - y[:, 0]) - (x[:, 2] - x[:, 0]) * (y[:, 1] - y[:, 0])
    boxes = (x1 - x0 + 1).clamp_min(0) * (y1 - y0 + 1).clamp_min(0)
    keep = torch.nonzero((area != 0) & (boxes > 0))[:, 0]
    ends = boxes[keep].cumsum(0).cpu()
    depth = torch.ones(s.height * s.width * s.samples, dtype=torch.float64, device=device)
    a, step = 0, 1 << 24
    while a < len(keep):
        base = int(ends[a - 1]) if a else 0
        b = max(a + 1, int(torch.searchsorted(ends, base + step, right=True)))
        tri = keep[a:b]
        n = boxes[tri]
        t = torch.repeat_interleave(tri, n)
        k = torch.arange(len(t), device=device) - torch.repeat_interleave(n.cumsum(0) - n, n)
        bw = (x1 - x0 + 1)[t]
        px, py = x0[t] + k % bw, y0[t] + torch.div(k, bw, rounding_mode="floor")
        sign = torch.sign(area[t])
        for i, (ox, oy) in enumerate(_SAMPLES[s.samples]):
            inside = torch.ones_like(t, dtype=torch.bool)
            edge = []
            for c in range(3):  # from corner c to the next, positive inside, top and left edges included
                dx, dy = (x[t, (c + 1) % 3] - x[t, c]) * sign, (y[t, (c + 1) % 3] - y[t, c]) * sign
                e = dx * (py * 16 + oy - y[t, c]) - dy * (px * 16 + ox - x[t, c])
                inside &= (e > 0) | ((e == 0) & ((dy < 0) | ((dy == 0) & (dx > 0))))
                edge.append(e)
            inv = 1.0 / area[t].abs().double()
            zz = z[t, 0] + (edge[2] * inv) * (z[t, 1] - z[t, 0]) + (edge[0] * inv) * (z[t, 2] - z[t, 0])
            at = (py * s.width + px) * s.samples + i
            depth.scatter_reduce_(0, at[inside], zz[inside].clamp(0.0, 1.0), "amin")
        a = b
    return depth.reshape(s.height, s.width, s.samples)


def exact(case, seed):
    """Depth in 64 bits (colours are stored as bytes); none for the clipped
    scenes, whose cut triangles are a rule of their own."""
    device = "cuda" if torch.cuda.is_available() else "cpu"
    if case["family"] == "saxpy":
        x, y = _vectors(case, seed)
        return {"y": float(np.float32(A)) * x.double() + y.double()}
    if case["family"] == "camera":
        return None
    out = {"color": None, "depth": _depth(_scene(case, seed), device)}
    if case["family"] == "phong":
        out["resolved"] = None
    return out
