"""The launch of a dispatch (kazan_compute_launch, what vkCmdDispatch records):
every workgroup is in exactly one block, and no dimension has more threads than
a launch takes (2^32 - 1) where the workgroups' own shape has fewer. And the
workgroups a block takes of a shader that needs many registers: no more than
the waves its registers leave resident, and one where blocks of several would
make it spill."""
import ctypes

import numpy as np
import pytest

from kazan_amd import vk
from kazan_amd.scenes import compute_shaders as cs
from kazan_amd.scenes import spirv as sp

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


def held_values_shader(held):
    """o[g + n i] = v[g + n i] * (v[g] + v[g + n] + ...), i < held, n a push
    constant: an invocation holds all its values until its first store."""

    def body(m, builtin):
        u, fl = m.t_int(False), m.t_float()
        gid = builtin(sp.BuiltInGlobalInvocationId, "g")
        v, o = cs._ssbo(m, fl, 4, 0, "v"), cs._ssbo(m, fl, 4, 1, "o")
        pc = cs._push_block(m, [u])
        f = sp.Function(m)
        g = cs._gid_x(f, m, gid)
        n = f.load(u, f.access_chain(m.t_ptr(sp.StoragePushConstant, u), pc, m.c_int(0)))
        at = [f.binop(sp.OpIAdd, u, g, f.binop(sp.OpIMul, u, n, m.c_int(i, signed=False))) for i in range(held)]
        x = [f.load(fl, cs._elem(f, m, v, fl, a)) for a in at]
        s = x[0]
        for y in x[1:]:
            s = f.fadd(fl, s, y)
        for a, y in zip(at, x):
            f.store(cs._elem(f, m, o, fl, a), f.fmul(fl, y, s))
        f.ret()
        return f

    return cs._compute_module((64, 1, 1), body).to_bytes()


@pytest.mark.parametrize("held", [4, 48, 100])
def test_block_of_a_shader_with_many_registers(driver, tmp_path, monkeypatch, held):
    monkeypatch.setenv("KAZAN_PIPELINE_CACHE", str(tmp_path))
    w = np.frombuffer(held_values_shader(held), np.uint32).copy()
    rc, msg = vk.tool_call(driver, "kazan_compile_compute_spirv", w.ctypes.data_as(ctypes.c_void_p),
                           ctypes.c_size_t(w.size), b"main", ctypes.c_uint32(2))
    assert rc == 0, msg
    kv = {k: v for k, v in (t.split("=") for t in msg.split())}
    vgprs, per = int(kv["vgprs"]), int(kv["per_block"])
    assert int(kv["scratch"]) == 0  # (as a workgroup alone has it)
    waves = min(512 // vgprs, 8) * 4
    assert waves // per * per == waves or per == 1
    if held == 4:
        assert per == 8
    elif held == 100:
        assert vgprs > 256 and per == 1
