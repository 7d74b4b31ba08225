"""grid_projection builds unrotated grids on the device (grid.device_view):
the rays are generate_projection_grid's bit for bit over the arguments it
takes, and everything else -- rotations, float32 extents, odd shapes, bad
arguments -- stays with numpy, with the same results and errors."""
import re

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

import vortrace_amd as vt  # noqa: E402
from vortrace_amd import grid  # noqa: E402

TAKEN = [
    dict(extent=[0.0, 10.0], nres=1, bounds=[0.0, 10.0]),
    dict(extent=[0, 10], nres=(1, 7), bounds=[0, 10]),
    dict(extent=np.array([1, 9]), nres=(33, 2), bounds=np.array([10.0, 0.0])),
    dict(extent=[[0.1, 9.7], [2.3, 2.9]], nres=[31, np.int64(17)], bounds=(0.3, 9.1)),
    dict(extent=[3.0, 3.0], nres=3, bounds=[0.0, 10.0]),
    dict(extent=[9.0, 1.0], nres=(64, 65), bounds=[10.0, 0.0], proj="xy"),
    dict(extent=[0.0, 10.0], nres=(5, 4), bounds=[0.0, 10.0], proj="yz"),
    dict(extent=[0.0, 10.0], nres=(40, 41), bounds=[0.0, 10.0], center=[5.0, 4.1, 5.3]),
    dict(extent=[-3.0, 10.0], nres=6, bounds=[0, 10], center=np.array([1, 2, 3]), proj="xy"),
    dict(extent=[1e-9, 3e-9], nres=(3, 4), bounds=np.array([0.0, 10.0], np.float32)),
]
KEPT = [
    dict(extent=np.array([0.0, 10.0], np.float32), nres=4, bounds=[0.0, 10.0]),
    dict(extent=[0.0, 10.0], nres=4, bounds=[0.0, 10.0], center=[5.0, 5.0, 5.0], yaw=0.3),
    dict(extent=[0.0, 10.0, 0.0, 10.0], nres=4, bounds=[0.0, 10.0]),
    dict(extent=[0.0, 10.0], nres=(4, 4.5), bounds=[0.0, 10.0]),
    dict(extent=[0.0, 10.0], nres=0, bounds=[0.0, 10.0]),
    dict(extent=[0.0, 1.0, 2.0], nres=4, bounds=[0.0, 10.0]),
    dict(extent=[0.0, np.inf], nres=4, bounds=[0.0, 10.0]),
]


@pytest.mark.parametrize("v", TAKEN)
def test_same_rays(v):
    view = grid.device_view(**v)
    assert view is not None
    s, e, _ = grid._rays_of([view], "cuda")
    ns, ne = grid.generate_projection_grid(**v)
    np.testing.assert_array_equal(s.cpu().numpy().reshape(ns.shape), ns)
    np.testing.assert_array_equal(e.cpu().numpy().reshape(ne.shape), ne)


@pytest.mark.parametrize("v", TAKEN[:9] + KEPT)
def test_same_projection(v, monkeypatch):
    rng = np.random.default_rng(2)
    pos = 10.0 * rng.random((500, 3))
    pc = vt.ProjectionCloud(pos, rng.random(500), boundbox=[0.0, 10.0] * 3, periodic=True)

    def project():
        try:
            return pc.grid_projection(**v)
        except Exception as ex:  # noqa: BLE001 -- whatever numpy raises
            # Whichever failing ray reports first is named.
            return type(ex).__name__, re.sub(r"^Ray \d+", "Ray", str(ex))
    assert (grid.device_view(**v) is None) == any(v is k for k in KEPT)
    with np.errstate(all="ignore"):
        got = project()
        monkeypatch.setattr(grid, "device_view", lambda *a, **k: None)
        want = project()
    np.testing.assert_array_equal(got, want)
