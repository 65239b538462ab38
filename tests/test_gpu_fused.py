"""Iterations with finalisers folded into their kernels, and fused ones, end
bit for bit where the separate kernels end: batch and streamed solves of one
right-hand side (folded up to 2,560 row blocks, fused on tensor-product
operators) against request servers of one lane that run the separate kernels
(CPMGPU_FOLD=0)."""
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
    return _serve_all(ctx, [(op, [(d_b, d_x)])], 1, o)[0]


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


def _dev(ctx, n, D, seed):
    d = []
    for k in range(n):
        d.append((ctx.alloc(8 * D), ctx.alloc(8 * D)))
        ctx.h2d(d[-1][0], np.random.default_rng([seed, k]).standard_normal(D))
    return d


def _serve_all(ctx, reqs, lanes, o, fold="0", chunks=(16,)):
    """reqs: (operator, [(d_b, d_x) ..]) each; the infos of every right-hand side in order."""
    with pytest.MonkeyPatch.context() as m:
        m.setenv("CPMGPU_FOLD", fold)
        s = cpmgpu.Server(ctx, sum(90 * lanes * (op.D + 64) for op, _ in reqs) + 4096, lanes=lanes, o=o)
        out, waiting, k = {}, list(enumerate(reqs)), 0
        while len(out) < len(reqs):
            for _ in range(len(reqs) if len(chunks) == 1 else 1):   # all at once, or one before each run
                if waiting:
                    tag, (op, d) = waiting.pop(0)
                    assert s.submit(op, [b for b, _ in d], [x for _, x in d], tag)
            out.update(dict(s.run(chunks[k % len(chunks)])[0]))
            k += 1
        s.close()
    return [i for tag in range(len(reqs)) for i in out[tag]]


@pytest.mark.parametrize("hs", [
    (0.1, 0.08, 0.13),       # three small segments, fused in both precisions
    (0.03, 0.0325),          # 833 row blocks in all: fused in both
    (0.0275, 0.028),         # 1,052: FP64 folded, mixed fused
    (0.0175, 0.018),         # 2,573: separate in both
])
@pytest.mark.parametrize("precision", [cpmgpu.CPM_FP64, cpmgpu.CPM_FP32_REFINE])
def test_several_operators_end_apart(gpu_ctx, monkeypatch, hs, precision):
    """One right-hand side on each of several operators whose systems end at different times: FP64
    against a server (separate kernels), mixed against iterations that are not fused."""
    print(f"case several operators {hs} {precision}", flush=True)
    monkeypatch.setenv("CPMGPU_FP64_ROUTING", "0")
    ops = [cpmgpu.Tube(gpu_ctx, "Sphere", h).operator(1.0, -c) for h, c in zip(hs, (1.0, 1e-4, 1e-2))]
    o = cpmgpu.opts(tol=1e-9, precision=precision)
    dev = [_dev(gpu_ctx, 1, op.D, k) for k, op in enumerate(ops)]
    read = lambda: [gpu_ctx.d2h(np.zeros(op.D), d[0][1]) for op, d in zip(ops, dev)]   # noqa: E731
    batch = lambda: gpu_ctx.solve_batch_device(ops, [d[0][0] for d in dev], [d[0][1] for d in dev], o)   # noqa: E731
    i1, x1 = batch(), read()
    if precision == cpmgpu.CPM_FP64:
        i2 = _serve_all(gpu_ctx, list(zip(ops, dev)), 1, o)
    else:
        monkeypatch.setenv("CPMGPU_PRECOND_FLY", "0")
        i2 = batch()
    x2 = read()
    print([i["iters"] for i in i1], flush=True)
    assert all(i["status"] == "converged" for i in i1) and len({i["iters"] for i in i1}) == len(ops)
    assert [(i["iters"], i["updates"], i["fallback_iters"]) for i in i1] == [(i["iters"], i["updates"], i["fallback_iters"]) for i in i2]
    assert all(np.array_equal(p, q) for p, q in zip(x1, x2))
    for d in dev:
        for p in d[0]:
            gpu_ctx.free(p)


@pytest.mark.parametrize("n,h", [
    (2, 0.0283), (2, 0.0279),     # 506 and 520 row blocks x 2 lanes
    (3, 0.0405), (3, 0.0395),     # 247 and 260 x 4
    (8, 0.057), (8, 0.0555),      # 125 and 132 x 8
])
@pytest.mark.parametrize("precision", [cpmgpu.CPM_FP64, cpmgpu.CPM_FP32_REFINE])
def test_folded_lanes_equal_separate_kernels(gpu_ctx, monkeypatch, n, h, precision):
    """Several right-hand sides of one operator on both sides of 1,024 lanes x row blocks, in batches
    (FP64; eight in the general format, which takes them in one group) and streams (mixed)."""
    print(f"case lanes {n} {h} {precision}", flush=True)
    monkeypatch.setenv("CPMGPU_FP64_ROUTING", "0")
    fp64 = precision == cpmgpu.CPM_FP64
    op = _operator(gpu_ctx, monkeypatch, "Sphere", h, False, "ell" if fp64 and n == 8 else "tp")
    lanes = 4 if n == 3 else n
    o = cpmgpu.opts(tol=1e-9, precision=precision)
    d = _dev(gpu_ctx, n, op.D, 5)
    bs, xs = [b for b, _ in d], [x for _, x in d]
    i1 = gpu_ctx.solve_batch_device([op] * n, bs, xs, o) if fp64 else gpu_ctx.solve_stream_device(op, bs, xs, lanes=lanes, o=o)
    x1 = [gpu_ctx.d2h(np.zeros(op.D), x) for x in xs]
    i2 = _serve_all(gpu_ctx, [(op, d)], lanes, o)
    x2 = [gpu_ctx.d2h(np.zeros(op.D), x) for x in xs]
    assert [(i["status"], i["iters"], i["updates"]) for i in i1] == [(i["status"], i["iters"], i["updates"]) for i in i2]
    assert all(np.array_equal(p, q) for p, q in zip(x1, x2))
    for p in bs + xs:
        gpu_ctx.free(p)


@pytest.mark.parametrize("hs,lanes,n", [
    ((0.1,), 1, 1),                     # one request: fused
    ((0.03, 0.0325, 0.2), 1, 1),        # fused while few are in, then folded (FP64)
    ((0.0175, 0.018, 0.1), 1, 1),       # past both lines while all are in
    ((0.1, 0.08, 0.13, 0.2), 4, 3),     # folded
    ((0.0405, 0.08), 4, 3),             # folded until both are in
])
@pytest.mark.parametrize("precision", [cpmgpu.CPM_FP64, cpmgpu.CPM_FP32_REFINE])
def test_servers_fold(gpu_ctx, monkeypatch, hs, lanes, n, precision):
    """Requests joining and leaving a server that folds or fuses where it may, with runs of odd
    lengths, against one that never does."""
    print(f"case servers fold {hs} {lanes} {precision}", flush=True)
    monkeypatch.setenv("CPMGPU_FP64_ROUTING", "0")
    reqs = []
    for k, h in enumerate(hs):
        op = cpmgpu.Tube(gpu_ctx, "Sphere", h).operator(1.0, -(0.1 ** (k % 3)))
        reqs.append((op, _dev(gpu_ctx, n, op.D, k)))
    o = cpmgpu.opts(tol=1e-9, precision=precision)
    res = []
    for fold in ("1", "0"):
        infos = _serve_all(gpu_ctx, reqs, lanes, o, fold, (3, 1, 16, 7))
        res.append((infos, [gpu_ctx.d2h(np.zeros(op.D), x) for op, d in reqs for _, x in d]))
    assert all(i["status"] == "converged" for i in res[0][0]) and res[0][0] == res[1][0]
    assert all(np.array_equal(p, q) for p, q in zip(res[0][1], res[1][1]))
    for _, d in reqs:
        for b, x in d:
            gpu_ctx.free(b)
            gpu_ctx.free(x)
