"""Batches over operators of both formats: each is gathered through its own
kernel (ELL, shared-stencil tiles, or rows where it has no tiles) and ends bit
for bit where it ends alone."""
import numpy as np
import pytest

import cpmgpu

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("order", ["etr", "rte", "teet", "er", "te"])
@pytest.mark.parametrize("n", [1, 2, 3, 8])
@pytest.mark.parametrize("precision", [cpmgpu.CPM_FP64, cpmgpu.CPM_FP32_REFINE])
def test_each_operator_as_alone(gpu_ctx, monkeypatch, order, n, precision):
    print(f"case mixed formats {order} n={n} precision={precision}", flush=True)
    monkeypatch.setenv("CPMGPU_FP64_ROUTING", "0")
    ops = []
    for k, f in enumerate(order):
        with monkeypatch.context() as m:
            if f == "e":
                m.setenv("CPMGPU_OP_FORMAT", "ell")
            if f == "r":
                m.setenv("CPMGPU_LDS_TILES", "0")
            ops.append(cpmgpu.Tube(gpu_ctx, "Sphere", (0.13, 0.061, 0.1, 0.25)[k]).operator(1.0, -(0.1 ** k)))
    rng = np.random.default_rng(n)
    bs = [[rng.standard_normal(op.D) for _ in range(n)] for op in ops]
    o = cpmgpu.opts(tol=1e-9, precision=precision)
    # the same right-hand sides of every operator, interleaved
    xs, infos = gpu_ctx.solve_batch([op for _ in range(n) for op in ops], [b[k] for k in range(n) for b in bs], o)
    for j, op in enumerate(ops):
        x1, i1 = gpu_ctx.solve_batch([op] * n, bs[j], o)
        for k in range(n):
            i = k * len(ops) + j
            assert infos[i]["status"] == "converged" and infos[i] == i1[k]
            assert np.array_equal(xs[i], x1[k]), (j, k)
