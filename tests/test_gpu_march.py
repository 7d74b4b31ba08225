"""GPU tests of the march (march.hip) against the ray engine.

help_events = 0 runs every ray in the engine, which repeats the reference's
steps one by one; the default marches the rays and leaves to the engine what
the march cannot vouch for.  Both must give the same bits and raise the same
errors: clouds of one cell up to a few list lengths, lists that end before a
cell's exit (a dense clump beside sparse cells), periodic boxes whose cells
are large against the box, near-coincident generators, rays
that start outside the box, end inside their first cell or graze ties, and
ray counts around the groups and waves of the kernels.
"""
import sys

import numpy as np
import pytest

from oracle import port

pytestmark = pytest.mark.gpu

import vortrace_amd as vt  # noqa: E402
from vortrace_amd import synthetic  # noqa: E402


def _say(msg):
    print(msg, flush=True)
    sys.stdout.flush()


@pytest.fixture()
def tuning():
    saved = vt.tuning.get_tuning()
    yield
    vt.tuning.set_tuning(**saved)


def _traced(pc, s, e, mode):
    try:
        return pc.traced_projection(s, e, reduction=mode, flatten=len(s) > 1)
    except (RuntimeError, ValueError) as ex:
        return type(ex).__name__, str(ex)


def _compare(pc, s, e, name, modes=("sum", "max")):
    """Projection and traced projection by the march and by the engine."""
    out = {}
    for he in (0, 128):
        vt.tuning.set_tuning(help_events=he)
        _say(f"  {name}: {len(s)} rays, help_events {he}")
        out[he] = [_traced(pc, s, e, m) for m in modes]
        try:
            out[he].append((pc.projection(s, e),))
        except (RuntimeError, ValueError) as ex:
            out[he].append((type(ex).__name__, str(ex)))
    for a, b in zip(out[128], out[0]):
        assert len(a) == len(b), (a, b)
        for x, y in zip(a, b):
            np.testing.assert_array_equal(x, y, err_msg=name)
    return out[128]


def _cloud(pos, box, periodic, f=None):
    f = 1.0 + np.arange(len(pos), dtype=np.float64) if f is None else f
    kw = {} if periodic else {"vol": np.full(len(pos), box ** 3 / len(pos))}
    return vt.ProjectionCloud(pos, f, boundbox=[0.0, box] * 3, periodic=periodic, **kw)


def _chords(n, seed, lo, hi):
    rng = np.random.default_rng(seed)
    return rng.uniform(lo, hi, (n, 3)), rng.uniform(lo, hi, (n, 3))


@pytest.mark.filterwarnings("ignore::UserWarning")
@pytest.mark.parametrize("periodic", [False, True])
@pytest.mark.parametrize("n", [1, 2, 3, 10, 11, 64, 65, 66, 500])
def test_small_clouds(tuning, n, periodic):
    rng = np.random.default_rng(100 + n)
    pos = 10.0 * rng.random((n, 3))
    pc = _cloud(pos, 10.0, periodic)
    for m in (1, 3, 17):
        s, e = _chords(m, n + m, 0.0, 10.0)
        _compare(pc, s, e, f"{n} cells, periodic {periodic}")


@pytest.mark.parametrize("rays", [1, 5, 63, 65, 1000, 4097, 20_000])
def test_ray_counts(tuning, rays):
    pos, rho = synthetic.uniform_mesh(20_000, seed=31)
    pc = vt.ProjectionCloud(pos, rho, boundbox=[0.0, 100.0] * 3, periodic=True)
    rng = np.random.default_rng(rays)
    xy = 100.0 * rng.random((rays, 2))
    s = np.column_stack([xy, np.zeros(rays)])
    e = np.column_stack([xy, np.full(rays, 100.0)])
    got = _compare(pc, s, e, "axis rays", modes=("sum",))
    k = min(rays, 500)
    oc = port.OracleCloud(pos, rho, [0.0, 100.0] * 3, periodic=True)
    np.testing.assert_array_equal(got[-1][0][:k], oc.project(s[:k], e[:k])[:, 0])


@pytest.mark.parametrize("periodic,rays", [(False, 16_383), (False, 16_384), (False, 65_535),
                                           (False, 65_536), (True, 16_384), (True, 196_607),
                                           (True, 196_608)])
def test_lanes_per_ray(tuning, periodic, rays):
    """Ray counts on both sides of each change of a ray's lanes (256 CUs)."""
    rng = np.random.default_rng(rays)
    pos = rng.uniform(0, 1, (3000, 3))
    if not periodic:
        pos[:700] = rng.normal(0.4, 0.003, (700, 3))
    pc = _cloud(pos, 1.0, periodic)
    s, e = _chords(rays, 7, 0.0, 1.0)
    if periodic:  # views, 0.9 of the box deep: oblique chords may have no unique split point
        s[:, 2] = 0.05
        e[:] = s + [0.0, 0.0, 0.9]
    got = []
    for he in (0, 128):
        vt.tuning.set_tuning(help_events=he)
        _say(f"  {rays} rays, periodic {periodic}, help_events {he}")
        got.append(pc.projection(s, e))
    np.testing.assert_array_equal(got[0], got[1])


@pytest.mark.parametrize("rays,outside", [(64, 0), (64, 32), (64, 33), (3072, 3072),
                                          (3073, 3073)])
def test_few_rays_that_leave_the_box(tuning, rays, outside):
    """Both sides of the choice between engine and march for a few rays."""
    pos, rho = synthetic.uniform_mesh(100_000, seed=61)
    pc = vt.ProjectionCloud(pos, rho, boundbox=[0.0, 100.0] * 3, periodic=False)
    s, e = _chords(rays, 9, 1.0, 99.0)
    s[:outside, 2] = -20.0
    _compare(pc, s, e, f"{outside} of {rays} rays leave the box")


@pytest.mark.parametrize("periodic", [False, True])
def test_clump_beside_void(tuning, periodic):
    """Lists full of a clump's generators do not reach across the void."""
    rng = np.random.default_rng(5)
    d = rng.standard_normal((6000, 3))
    d /= np.linalg.norm(d, axis=1)[:, None]
    clump = 50.0 + 0.5 * rng.random(6000)[:, None] * d
    pos = np.concatenate([clump, 100.0 * rng.random((400, 3))])
    pc = _cloud(pos, 100.0, periodic)
    if periodic:
        xy = 50.0 + rng.uniform(-3.0, 3.0, (600, 2))
        s = np.column_stack([xy, np.zeros(600)])
        e = np.column_stack([xy, np.full(600, 100.0)])
    else:
        s, e = _chords(600, 6, 0.0, 100.0)
        e[:300] = clump[:300]
    got = _compare(pc, s, e, f"clump, periodic {periodic}")
    oc = port.OracleCloud(pos, 1.0 + np.arange(len(pos), dtype=np.float64), [0.0, 100.0] * 3,
                          vol=None if periodic else np.full(len(pos), 1e6 / len(pos)),
                          periodic=periodic)
    np.testing.assert_array_equal(got[-1][0], oc.project(s, e)[:, 0])


def test_near_ties_and_odd_rays(tuning):
    """Near-coincident generators, lattice planes, tiny and outside rays."""
    rng = np.random.default_rng(9)
    pos = 10.0 * rng.random((3000, 3))
    pos[100:120] = pos[200:220] + 1e-5 * rng.standard_normal((20, 3))
    pos[300:310] = np.round(pos[300:310])
    pos[310:320] = pos[300:310] + [0.0, 0.0, 1.0]
    pc = _cloud(pos, 10.0, False)
    s, e = _chords(400, 10, -5.0, 15.0)
    s[:40], e[:40] = pos[100:140] - [0.3, 0.2, 0.1], pos[100:140] + [0.3, 0.2, 0.1]
    s[40:60] = pos[300:320] - [0.5, 0.0, 0.0]
    e[40:60] = pos[300:320] + [0.5, 0.0, 0.0]
    s[60:80] = pos[500:520]
    e[60:80] = s[60:80] + 1e-7
    e[80:90] = s[80:90] + [0.0, 0.0, 2e-6]
    _compare(pc, s, e, "near ties and odd rays", modes=("sum", "min"))


def test_periodic_rays_leave_the_box(tuning):
    """Rotated views: rays start and end up to most of a box outside."""
    pos, rho = synthetic.clustered_mesh(30_000, seed=41, n_clumps=12)
    pc = vt.ProjectionCloud(pos, rho, boundbox=[0.0, 100.0] * 3, periodic=True)
    views = synthetic.camera_rays(42, 3, sizes=(24, 40), extent_range=(60.0, 100.0))
    s = np.concatenate([v[0] for v in views])
    e = np.concatenate([v[1] for v in views])
    _compare(pc, s, e, "rotated views", modes=("sum",))
