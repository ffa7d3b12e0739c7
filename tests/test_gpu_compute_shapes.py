"""Dispatches of odd, 2-D and 3-D workgroups over several dimensions, where a
block takes one workgroup and where it takes several (around the rule's line:
four blocks' worth of them along x), with and without a base workgroup: every
invocation sees its own ids and the dispatch's size, as it writes them itself.
Shaders that need many registers, whose blocks take fewer workgroups or one.
And a dispatch whose rows have more threads in all than a launch takes along x
in linear blocks."""
import numpy as np
import pytest

from kazan_amd.scenes import compute_shaders as cs
from kazan_amd.scenes import spirv as sp
from kazan_amd.scenes.compute import ComputeKernel, read_buffer
from test_compute_launch import held_values_shader

pytestmark = pytest.mark.gpu


def _ids_shader(local):
    """o[4 * (g.x + w * (g.y + h * g.z)) + k] = k-th of: workgroup id, local
    id, local index, number of workgroups (x + 4096 y + 2^24 z each); g the
    global id less the base's, (w, h, base x * local x) push constants."""

    def body(m, builtin):
        u, v3 = m.t_int(False), m.t_uvec(3)
        gid = builtin(sp.BuiltInGlobalInvocationId, "g")
        wid = builtin(sp.BuiltInWorkgroupId, "wg")
        lid = builtin(sp.BuiltInLocalInvocationId, "l")
        num = builtin(sp.BuiltInNumWorkgroups, "n")
        lix = m.variable(sp.StorageInput, u, "li")
        m.decorate(lix, sp.DecorationBuiltIn, sp.BuiltInLocalInvocationIndex)
        body.extra = lix
        out = cs._ssbo(m, u, 4, 0, "o")
        pc = cs._push_block(m, [u, u, u])
        f = sp.Function(m)
        c = lambda v: m.c_int(v, signed=False)
        add = lambda a, b: f.binop(sp.OpIAdd, u, a, b)
        mul = lambda a, b: f.binop(sp.OpIMul, u, a, b)
        push = [f.load(u, f.access_chain(m.t_ptr(sp.StoragePushConstant, u), pc, m.c_int(k))) for k in range(3)]

        def packed(v):
            x = f.load(v3, v)
            x, y, z = (f.extract(u, x, k) for k in range(3))
            return add(x, add(mul(y, c(4096)), mul(z, c(1 << 24))))

        g = f.load(v3, gid)
        gx, gy, gz = (f.extract(u, g, k) for k in range(3))
        at = add(f.binop(sp.OpISub, u, gx, push[2]), mul(push[0], add(gy, mul(push[1], gz))))
        for k, val in enumerate((packed(wid), packed(lid), f.load(u, lix), packed(num))):
            f.store(cs._elem(f, m, out, u, add(mul(at, c(4)), c(k))), val)
        f.ret()
        return f

    m = sp.Module()
    m.capability(sp.CapabilityShader)
    m.set_memory_model()
    iface = []

    def builtin(b, name):
        v = m.variable(sp.StorageInput, m.t_uvec(3), name)
        m.decorate(v, sp.DecorationBuiltIn, b)
        iface.append(v)
        return v

    f = body(m, builtin)
    m.entry_point(sp.ExecutionModelGLCompute, f.id, "main", iface + [body.extra])
    m.execution_mode(f.id, sp.ExecutionModeLocalSize, *local)
    return m.to_bytes()


def _expected(local, groups, base):
    w = [local[k] * groups[k] for k in range(3)]
    z, y, x = np.meshgrid(*(np.arange(n, dtype=np.uint32) for n in (w[2], w[1], w[0])), indexing="ij")
    pack = lambda a, b, c: a + 4096 * b + (1 << 24) * c
    lx, ly, lz = x % local[0], y % local[1], z % local[2]
    out = np.zeros((w[2], w[1], w[0], 4), np.uint32)
    out[..., 0] = pack(x // local[0] + base, y // local[1], z // local[2])
    out[..., 1] = pack(lx, ly, lz)
    out[..., 2] = lx + local[0] * (ly + local[1] * lz)
    out[..., 3] = pack(*groups)
    return out.ravel()


@pytest.mark.parametrize("local", [(64, 1, 1), (1, 1, 1), (3, 5, 2), (8, 8, 1), (1, 100, 1), (4, 4, 4), (2, 1, 33)])
def test_ids(ctx, local):
    most = max(1, 512 // (local[0] * local[1] * local[2]))
    k = ComputeKernel(ctx, _ids_shader(local), 1, push_bytes=12)
    try:
        for x in sorted({1, 4 * most - 1, 4 * most, 4 * most + 1, 5 * most}):
            for yz, base in (((1, 1), None), ((3, 2), None), ((1, 1), 7)):
                groups = (x,) + yz
                want = _expected(local, groups, base or 0)
                print("local %s groups %s base %s" % (local, groups, base), flush=True)
                ob = ctx.device_buffer_with(np.full(want.size + 64, 0xDEADBEEF, np.uint32))
                k.bind([(ob[0], want.nbytes)])
                k.run(groups, push=np.array([local[0] * x, local[1] * yz[0], (base or 0) * local[0]], np.uint32),
                      base=None if base is None else (base, 0, 0))
                got = read_buffer(ctx, ob[0], want.nbytes + 256, np.uint32)
                ctx.destroy_buffer(ob)
                np.testing.assert_array_equal(got[:want.size], want)
                assert (got[want.size:] == 0xDEADBEEF).all()
    finally:
        k.destroy()


@pytest.mark.parametrize("held", [4, 48, 100])
def test_many_registers(ctx, held):
    for groups in (1, 31, 33, 70):
        n = 64 * groups
        x = np.random.default_rng(groups).random((held, n), np.float32)
        s = x[0].copy()
        for y in x[1:]:
            s += y
        vb, ob = ctx.device_buffer_with(x), ctx.device_buffer_with(np.zeros(x.size + 64, np.float32))
        k = ComputeKernel(ctx, held_values_shader(held), 2, push_bytes=4)
        k.bind([(vb[0], x.nbytes), (ob[0], x.nbytes)])
        k.run((groups,), push=np.array([n], np.uint32))
        got = read_buffer(ctx, ob[0], x.nbytes + 256, np.float32)
        k.destroy()
        ctx.destroy_buffer(vb)
        ctx.destroy_buffer(ob)
        np.testing.assert_array_equal(got[:x.size].reshape(x.shape), x * s)
        assert (got[x.size:] == 0).all()


def test_long_rows_of_tall_workgroups(ctx):
    """2^24 workgroups of 1 x 256: 2^32 invocations, of which the last
    workgroup's write their index."""

    def body(m, builtin):
        u = m.t_int(False)
        gid = builtin(sp.BuiltInGlobalInvocationId, "g")
        lid = builtin(sp.BuiltInLocalInvocationId, "l")
        out = cs._ssbo(m, u, 4, 0, "o")
        f = sp.Function(m)
        gx = cs._gid_x(f, m, gid)
        then, merge = f.new_label(), f.new_label()
        f.selection_merge(merge)
        f.branch_cond(f.binop(sp.OpULessThan, m.t_bool(), m.c_int((1 << 24) - 2, signed=False), gx), then, merge)
        f.label(then)
        y = f.extract(u, f.load(m.t_uvec(3), lid), 1)
        f.store(cs._elem(f, m, out, u, y), f.binop(sp.OpIAdd, u, y, gx))
        f.branch(merge)
        f.label(merge)
        f.ret()
        return f

    k = ComputeKernel(ctx, cs._compute_module((1, 256, 1), body).to_bytes(), 1)
    ob = ctx.device_buffer_with(np.zeros(256, np.uint32))
    try:
        k.bind([(ob[0], 1024)])
        k.run((1 << 24,))
        got = read_buffer(ctx, ob[0], 1024, np.uint32)
        np.testing.assert_array_equal(got, np.arange(256) + (1 << 24) - 1)
    finally:
        k.destroy()
        ctx.destroy_buffer(ob)
