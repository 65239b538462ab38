"""Operators in the general sparse format at row widths around the rounds of
the E gather (32 and 8 slots, then one by one), applies and solves of 1 to 8
right-hand sides against dense numpy in FP64."""
import numpy as np
import pytest

import cpmgpu

pytestmark = pytest.mark.gpu

D = 601   # two full row blocks and a partial one


def _system(width, seed):
    """E with 1..width random columns a row (every 50th has all), L with a diagonal and 0..4 others, some identity rows."""
    rng = np.random.default_rng(seed)
    Ep, Ec, Ev, Lp, Lc, Lv = [0], [], [], [0], [], []
    ident = np.zeros(D, np.uint8)
    ident[rng.choice(D, 7, replace=False)] = 1
    E, L = np.zeros((D, D)), np.zeros((D, D))
    for r in range(D):
        n = width if r % 50 == 0 else int(rng.integers(1, width + 1))
        c, v = np.sort(rng.choice(D, n, replace=False)), rng.uniform(-1.0, 1.0, n) / n
        E[r, c] = v
        Ec += list(c)
        Ev += list(v)
        Ep.append(len(Ec))
        c = np.unique(np.append(rng.choice(D, int(rng.integers(0, 5)), replace=False), r))
        v = np.where(c == r, -4.0, rng.uniform(0.5, 1.0, len(c)))
        L[r, c] = v
        Lc += list(c)
        Lv += list(v)
        Lp.append(len(Lc))
    csr = lambda p, c, v: cpmgpu.CSR(np.array(p, np.int32), np.array(c, np.int32), np.array(v))   # noqa: E731
    return csr(Lp, Lc, Lv), csr(Ep, Ec, Ev), ident, L, E


@pytest.mark.parametrize("width", [1, 4, 7, 8, 9, 16, 25, 27, 31, 32, 33, 40, 41, 63, 64, 65, 125])
def test_row_widths(gpu_ctx, monkeypatch, width):
    print(f"case ell width={width}", flush=True)
    monkeypatch.setenv("CPMGPU_FP64_ROUTING", "0")
    Lm, Em, ident, L, E = _system(width, width)
    op = cpmgpu.Operator(gpu_ctx, Lm, Em, ident, 1.0, -0.5)
    assert op.format == "ell"
    diag = np.diag(np.diag(L))
    rng = np.random.default_rng(1)
    x = rng.standard_normal(D)

    def dense(m, n, E, L, diag, ident):
        A = m * np.eye(D) + n * (diag + (L - diag) @ np.where(ident[:, None] != 0, np.eye(D), E))
        return np.where(ident[:, None] != 0, np.eye(D), A)

    y = op.multiply(x, 0.7, -1.3)
    scale = dense(0.7, 1.3, abs(E), abs(L), abs(diag), ident) @ abs(x)
    assert np.all(abs(y - dense(0.7, -1.3, E, L, diag, ident) @ x) <= (width + 16) * 2.3e-16 * scale)
    A = dense(1.0, -0.5, E, L, diag, ident)
    b = rng.standard_normal((8, D))
    xs = np.linalg.solve(A, b.T).T
    limit = 1e-12 * np.linalg.cond(A) + 1e-13   # solves stop at a relative residual of 1e-12
    for prec in (cpmgpu.CPM_FP64, cpmgpu.CPM_FP32_REFINE):
        for n in (1, 2, 3, 8):
            got, infos = gpu_ctx.solve_batch([op] * n, list(b[:n]), cpmgpu.opts(tol=1e-12, precision=prec, max_iters=2000))
            assert all(i["status"] == "converged" for i in infos), infos
            for k in range(n):
                assert np.linalg.norm(got[k] - xs[k]) <= limit * np.linalg.norm(xs[k])
