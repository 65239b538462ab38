"""Shared-stencil tiles built on the GPU: at the sizes where a tile, a run of
items or a wave ends, applies and solves through them end bit for bit where
the direct gather (CPMGPU_LDS_TILES=0) ends."""
import numpy as np
import pytest

import cpmgpu

pytestmark = pytest.mark.gpu


def _circle():
    n = np.array([1.1, 1.234, 1.321])
    n /= np.linalg.norm(n)
    return [np.sqrt(1 - 0.31 ** 2), *(0.31 * n), *n]


@pytest.mark.parametrize("surface,dx,ibc", [
    ("Sphere", 0.5, None),          # a few hundred rows: one partly filled run
    ("Sphere", 0.31, None),         # an odd spacing, a last tile that is nearly empty
    ("Sphere", 0.12, "circle"),     # moved columns, ghost rows, identity rows
    ("Sphere", 0.045, "circle"),    # full tiles of 256 items
    ("Torus", 0.05, None),          # 256 items a tile, another shape
    ("Sphere", 0.15, "point"),      # a point's ghost rows (lists of few, scattered rows)
])
def test_tiles_equal_direct_gather(gpu_ctx, monkeypatch, surface, dx, ibc):
    print(f"case tiles {surface} {dx} {ibc}", flush=True)
    monkeypatch.setenv("CPMGPU_FP64_ROUTING", "0")   # FP32 is tried on both operators, whatever fell back before
    tube = cpmgpu.Tube(gpu_ctx, surface, dx)
    if ibc is None:
        make = tube.operator
    else:
        c = cpmgpu.IBC("Circle3D", params=_circle()) if ibc == "circle" else cpmgpu.IBC("Point", params=[0.0, 0.6, 0.8],
                                                                                       boundary_order=1)
        c.on_ibc_tolerance = 0.1 * dx * dx
        make = cpmgpu.Problem(tube, [c]).operator
    ops = {}
    for mode in ("1", "0"):
        monkeypatch.setenv("CPMGPU_LDS_TILES", mode)
        ops[mode] = make(1.0, -1.0)
    D = ops["1"].D
    info = ops["1"].tile_info()
    print(f"D={D} {info}", flush=True)
    assert info["shared_stencil_tiles"] > 0
    assert ops["1"].gather_kernel(cpmgpu.CPM_FP64, 1) == "k_egather_grp<double,1>"
    assert ops["0"].gather_kernel(cpmgpu.CPM_FP64, 1) == "k_egather<double,1>"
    rng = np.random.default_rng(5)
    x = rng.standard_normal(D)
    assert np.array_equal(ops["1"].multiply(x, 0.5, -1.0), ops["0"].multiply(x, 0.5, -1.0))
    b = [rng.standard_normal(D) for _ in range(8)]
    for nb, prec in ((1, cpmgpu.CPM_FP64), (3, cpmgpu.CPM_FP64), (1, cpmgpu.CPM_FP32_REFINE), (2, cpmgpu.CPM_FP32_REFINE),
                     (4, cpmgpu.CPM_FP32_REFINE), (8, cpmgpu.CPM_FP32_REFINE)):
        o = cpmgpu.opts(tol=1e-14, max_iters=12, precision=prec)
        x1, i1 = gpu_ctx.solve_batch([ops["1"]] * nb, b[:nb], o)
        x0, i0 = gpu_ctx.solve_batch([ops["0"]] * nb, b[:nb], o)
        assert [i["iters"] for i in i1] == [i["iters"] for i in i0]
        assert all(np.array_equal(p, q) for p, q in zip(x1, x0)), (nb, prec)
