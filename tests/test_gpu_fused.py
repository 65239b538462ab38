"""Iterations with finalisers folded into their kernels, and fused ones, end
bit for bit where the separate kernels end: batch and streamed solves of one
right-hand side (folded up to 2,560 row blocks, fused on tensor-product
operators) against request servers of one lane, which run the separate
kernels."""
import numpy as np
import pytest

import cpmgpu

pytestmark = pytest.mark.gpu


def _operator(ctx, monkeypatch, surface, dx, ibc, fmt):
    if fmt == "ell":
        monkeypatch.setenv("CPMGPU_OP_FORMAT", "ell")
    tube = cpmgpu.Tube(ctx, surface, dx)
    if not ibc:
        return tube.operator(1.0, -1.0)
    n = np.array([1.1, 1.234, 1.321])
    n /= np.linalg.norm(n)
    c = cpmgpu.IBC("Circle3D", params=[np.sqrt(1 - 0.31 ** 2), *(0.31 * n), *n], on_ibc_tolerance=0.1 * dx * dx)
    return cpmgpu.Problem(tube, [c]).operator(0.0, -1.0)


def _serve(ctx, op, d_b, d_x, o):
    s = cpmgpu.Server(ctx, 256 * op.D, lanes=1, o=o)
    assert s.submit(op, [d_b], [d_x], 7)
    while True:
        done, _ = s.run(16)
        if done:
            s.close()
            return done[0][1][0]


@pytest.mark.parametrize("surface,dx,ibc,fmt", [
    ("Sphere", 0.5, False, "tp"),        # fewer rows than one wave has partials
    ("Sphere", 0.1, True, "tp"),         # moved columns and identity rows, 43 blocks
    ("Sphere", 0.05, False, "tp"),       # 164 blocks
    ("Sphere", 0.0201, False, "tp"),     # a full first load of partials
    ("Sphere", 0.0199, False, "tp"),     # and a second one
    ("Sphere", 0.0126, False, "tp"),     # the most blocks that fold
    ("Sphere", 0.0125, False, "tp"),     # too many
    ("Sphere", 0.1, True, "ell"),        # folded, not fused
])
@pytest.mark.parametrize("precision", [cpmgpu.CPM_FP64, cpmgpu.CPM_FP32_REFINE])
def test_folded_iterations_equal_separate_kernels(gpu_ctx, monkeypatch, surface, dx, ibc, fmt, precision):
    print(f"case fused {surface} {dx} {ibc} {fmt} {precision}", flush=True)
    monkeypatch.setenv("CPMGPU_FP64_ROUTING", "0")
    op = _operator(gpu_ctx, monkeypatch, surface, dx, ibc, fmt)
    D = op.D
    assert op.format == fmt
    b = np.random.default_rng(31).standard_normal(D)
    d_b, d_x = gpu_ctx.alloc(8 * D), gpu_ctx.alloc(8 * D)
    gpu_ctx.h2d(d_b, b)
    o = cpmgpu.opts(tol=1e-9, precision=precision)
    if precision == cpmgpu.CPM_FP64:
        i1 = op.solve_device(d_b, d_x, o)
    else:   # the streamed start is the server's
        i1 = gpu_ctx.solve_stream_device(op, [d_b], [d_x], lanes=1, o=o)[0]
    x1 = gpu_ctx.d2h(np.zeros(D), d_x)
    i2 = _serve(gpu_ctx, op, d_b, d_x, o)
    x2 = gpu_ctx.d2h(np.zeros(D), d_x)
    print(f"D={D} iters={i1['iters']} updates={i1['updates']}", flush=True)
    assert (i1["status"], i1["iters"], i1["updates"], i1["fallback_iters"]) == (i2["status"], i2["iters"], i2["updates"], i2["fallback_iters"])
    assert np.array_equal(x1, x2)
    gpu_ctx.free(d_b)
    gpu_ctx.free(d_x)
