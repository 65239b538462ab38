"""The breadth-first walk of a curve's tagging subset where its frontier is
wide (levels over the whole GPU), narrow again, and where its members exceed
the room first set aside."""
import numpy as np
import pytest

import cpmgpu
import orc

pytestmark = pytest.mark.gpu


def _spiral(turns, z0, z1, n=800):
    """From height z0 to z1 on the unit sphere."""
    t = np.linspace(0.0, 1.0, n)
    z = np.cos(np.arccos(z0) + t * (np.arccos(z1) - np.arccos(z0)))
    q = np.sqrt(1.0 - z * z)
    return np.stack([q * np.cos(2 * np.pi * turns * t), q * np.sin(2 * np.pi * turns * t), z], 1)


@pytest.mark.parametrize("dx,turns,z0,z1,point", [
    (0.1, 3, 0.98, -0.98, False),     # hardly wide
    (0.06, 4, 0.98, -0.98, False),    # wide from near one pole to near the other
    (0.05, 3, 0.98, 0.45, True),      # wide on a cap, with a point's narrow walk in the same launch
])
def test_wide_frontier_matches_oracle(gpu_ctx, dx, turns, z0, z1, point):
    print(f"case wide walk dx={dx} turns={turns}", flush=True)
    ibcs = [dict(type="Polyline", verts=_spiral(turns, z0, z1), on_ibc_tolerance=0.1 * dx * dx)]
    if point:
        ibcs.insert(0, dict(type="Point", params=[0.0, 0.28, -0.96], boundary_order=1, on_ibc_tolerance=0.1 * dx * dx))
    P = orc.IBCProblem("Sphere", dx, ibcs=[orc.IBC(**k) for k in ibcs])
    Q = cpmgpu.Problem(cpmgpu.Tube(gpu_ctx, "Sphere", dx), [cpmgpu.IBC(**k) for k in ibcs])
    for c in range(len(ibcs)):
        so, co, _ = P.subset(c, 0)
        sg, cg, _ = Q.subset(c, 0)
        print(f"curve {c}: {len(sg)} members", flush=True)
        assert np.array_equal(sg, so)                 # the same nodes in the same breadth-first order
        assert np.abs(cg - co).max() <= 1e-14


def test_members_past_the_first_room(gpu_ctx):
    """Degree 4 on a thin ellipsoid, whose tube also holds its inside: a point's members are more than
    the room set aside (204 x 16), and the walk starts again with more."""
    print("case walk room", flush=True)
    dx, p = 0.05, np.array([0.0, 0.0, 0.2])
    tube = cpmgpu.Tube(gpu_ctx, "Ellipsoid", dx, params=[1.0, 1.0, 0.2], bbox=(-1.0, 1.0), p=4)
    Q = cpmgpu.Problem(tube, [cpmgpu.IBC("Point", params=list(p), boundary_order=1, on_ibc_tolerance=0.1 * dx * dx)])
    t = tube.export()
    near = np.linalg.norm(t["x"] - p, axis=1) < 2 * 1.0001 * np.sqrt(2 * 2.5 ** 2 + 3.5 ** 2) * dx
    order, seen, front = [], np.zeros(tube.N, bool), [int(np.argmin(np.linalg.norm(t["x"] - p, axis=1)))]
    while front:                                      # the start node is not marked at first
        new = []
        for i in front:
            for j in t["nbr"][i]:
                if j >= 0 and near[j] and not seen[j]:
                    seen[j] = True
                    new.append(int(j))
        order += new
        front = new
    s, cp, _ = Q.subset(0, 0)
    assert len(order) > 204 * 16
    assert np.array_equal(s, order) and np.array_equal(cp, np.broadcast_to(p, cp.shape))


def test_room_of_a_circle_with_negative_radius(gpu_ctx):
    """The first room is guessed from the curve's length, which a signed radius must not turn into a
    failing allocation: such a circle's closest points lie opposite, and its subset is empty."""
    print("case walk negative radius", flush=True)
    n = np.array([1.1, 1.234, 1.321])
    n /= np.linalg.norm(n)
    tube = cpmgpu.Tube(gpu_ctx, "Sphere", 0.05)
    with pytest.raises(cpmgpu.CpmError, match="tagging subset is empty"):
        cpmgpu.Problem(tube, [cpmgpu.IBC("Circle3D", params=[-np.sqrt(1 - 0.31 ** 2), *(0.31 * n), *n], on_ibc_tolerance=0.1 * 0.05 ** 2)])
