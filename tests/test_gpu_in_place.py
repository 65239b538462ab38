"""Applies and explicit steps on the callers' vectors in place against the
packed ones (CPMGPU_GROUP_GATHER=none): the apply to the bit, steps to a few
roundings (one step sums at most 64 products of weights whose absolute sum is
below 4, each operand off by a rounding or two: 1e-14 of the largest value)."""
import numpy as np
import pytest

import cpmgpu

pytestmark = pytest.mark.gpu


def _circle(order, btype):
    n = np.array([1.1, 1.234, 1.321])
    n /= np.linalg.norm(n)
    return cpmgpu.IBC("Circle3D", params=[np.sqrt(1 - 0.31 ** 2), *(0.31 * n), *n], boundary_order=order,
                      boundary_type=(btype, btype))


@pytest.mark.parametrize("dx,ibc", [(0.5, None), (0.31, None), (0.12, (2, 0)), (0.12, (1, 0)), (0.12, (2, 1)), (0.045, (2, 0))])
def test_in_place_equals_packed(gpu_ctx, monkeypatch, dx, ibc):
    print(f"case in place dx={dx} ibc={ibc}", flush=True)
    tube = cpmgpu.Tube(gpu_ctx, "Sphere", dx)
    if ibc is None:
        op = tube.operator(1.0, -1.0)
    else:
        c = _circle(*ibc)
        c.on_ibc_tolerance = 0.1 * dx * dx
        op = cpmgpu.Problem(tube, [c]).operator(1.0, -1.0)
    D = op.D
    rng = np.random.default_rng(3)
    u0, v0, g = rng.uniform(0.2, 1.0, D), rng.uniform(0.0, 0.5, D), rng.standard_normal(D)
    d = [gpu_ctx.alloc(8 * D) for _ in range(5)]
    p = cpmgpu.rd_params(dx, method=0)
    out = {}
    for mode in ("", "none"):
        monkeypatch.setenv("CPMGPU_GROUP_GATHER", mode)
        y = op.multiply(u0, 0.7, -1.3)
        gpu_ctx.h2d(d[0], u0)
        op.multiply_device(d[0], d[0], 0.7, -1.3)          # x and y the same vector
        same = gpu_ctx.d2h(np.zeros(D), d[0])
        gpu_ctx.h2d(d[0], u0)
        gpu_ctx.h2d(d[4], g)
        op.heat_step_device(0, 0.1 * dx * dx, d[4], d[0])
        h = gpu_ctx.d2h(np.zeros(D), d[0])
        for q, a in zip(d[:4], (u0, v0, v0, u0)):           # two fields
            gpu_ctx.h2d(q, a)
        op.rd_step_device(p, [d[0], d[2]], [d[1], d[3]], d[4], d[4])
        out[mode] = [y, same, h] + [gpu_ctx.d2h(np.zeros(D), q) for q in d[:4]]
    a, b = out[""], out["none"]
    assert np.array_equal(a[0], b[0]) and np.array_equal(a[1], b[1]) and np.array_equal(a[0], a[1])
    for x, y in zip(a[2:], b[2:]):
        assert np.abs(x - y).max() <= 1e-14 * np.abs(y).max()
    for q in d:
        gpu_ctx.free(q)
