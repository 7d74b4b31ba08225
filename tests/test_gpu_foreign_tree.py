"""Trees whose cuts do not bound the cloud's points.

vt_cloud_load_tree takes any well-formed dump over as many points, also one
saved before the points moved, and periodic clouds take NaN coordinates.  The
reference then answers with what its searches find through that tree, and the
ray engine (help_events = 0) repeats it; a march over lists and boxes of the
points themselves finds other cells.  Such clouds must not be marched.
"""
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

import vortrace_amd as vt  # noqa: E402
from vortrace_amd import synthetic  # noqa: E402

BB = [0.0, 100.0] * 3


def _both(pc, s, e):
    saved = vt.tuning.get_tuning()
    out = []
    try:
        for he in (0, 128):
            vt.tuning.set_tuning(help_events=he)
            print(f"  help_events {he}", flush=True)
            sys.stdout.flush()
            try:
                out.append(pc.traced_projection(s, e, flatten=True))
            except (RuntimeError, ValueError) as ex:
                out.append(type(ex))
    finally:
        vt.tuning.set_tuning(**saved)
    return out


def _same(a, b):
    assert type(a) is type(b)
    if isinstance(a, tuple):
        for x, y in zip(a, b):
            np.testing.assert_array_equal(x, y)


def _rays(n, seed):
    xy = 100.0 * np.random.default_rng(seed).random((n, 2))
    return (np.column_stack([xy, np.full(n, 0.5)]), np.column_stack([xy, np.full(n, 99.5)]))


@pytest.mark.filterwarnings("ignore::UserWarning")
@pytest.mark.parametrize("periodic", [False, True])
def test_tree_of_points_that_moved(periodic):
    pos, rho = synthetic.uniform_mesh(8000, seed=71)
    old = vt.ProjectionCloud(pos, rho, boundbox=BB, periodic=periodic)
    moved = np.clip(pos + 0.4 * np.random.default_rng(72).standard_normal(pos.shape), 0.0, 100.0)
    pc = vt.ProjectionCloud(moved, rho, boundbox=BB, periodic=periodic)
    pc.load_tree_bytes(old.save_tree_bytes())
    a, b = _both(pc, *_rays(400, 73))
    _same(a, b)
    # The cloud's own tree again: marched again, and the engine's bits.
    pc.load_tree_bytes(vt.ProjectionCloud(moved, rho, boundbox=BB,
                                          periodic=periodic).save_tree_bytes())
    a, b = _both(pc, *_rays(400, 73))
    assert isinstance(a, tuple)
    _same(a, b)


@pytest.mark.filterwarnings("ignore::UserWarning")
def test_nan_points():
    pos, rho = synthetic.uniform_mesh(3000, seed=74)
    pos[[5, 700, 2999]] = np.nan
    pos[1200, 1] = np.nan
    a, b = _both(vt.ProjectionCloud(pos, rho, boundbox=BB, periodic=True), *_rays(200, 75))
    _same(a, b)
