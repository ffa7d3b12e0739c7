"""Dispatches whose blocks take several workgroups (compute shaders without
workgroup memory and barriers: eight workgroups of 64 invocations a block):
workgroup counts around the rule's line (32) and around whole blocks, and with
a base workgroup. Every element is written exactly once: the results equal
numpy's, and the rest of the buffer keeps its values."""
import numpy as np
import pytest

from kazan_amd.scenes import compute_shaders as cs
from kazan_amd.scenes.compute import ComputeKernel, read_buffer

pytestmark = pytest.mark.gpu


def _saxpy(ctx, groups, base, n):
    size = 64 * 80
    rng = np.random.default_rng(groups)
    x, y = rng.random(size, np.float32), rng.random(size, np.float32)
    bx, by = ctx.device_buffer_with(x), ctx.device_buffer_with(y)
    k = ComputeKernel(ctx, cs.cs_saxpy(), 2, push_bytes=8)
    k.bind([(bx[0], 4 * size), (by[0], 4 * size)])
    k.run((groups,), push=np.array([np.float32(0.5).view(np.uint32), n], np.uint32), base=base)
    got = read_buffer(ctx, by[0], y.nbytes, np.float32)
    want = y.copy()
    at = np.arange(size)
    on = (at >= 64 * base[0]) & (at < min(n, 64 * (base[0] + groups)))
    want[on] = (np.float32(0.5) * x + y)[on]
    k.destroy()
    ctx.destroy_buffer(bx)
    ctx.destroy_buffer(by)
    np.testing.assert_array_equal(got, want)


@pytest.mark.parametrize("groups", [1, 8, 15, 31, 32, 33, 39, 40, 63, 64])
def test_saxpy_workgroup_counts(ctx, groups):
    _saxpy(ctx, groups, (0, 0, 0), 64 * groups - 3)


@pytest.mark.parametrize("groups", [3, 33, 65])
def test_saxpy_with_a_base(ctx, groups):
    _saxpy(ctx, groups, (5, 0, 0), 64 * 80)
