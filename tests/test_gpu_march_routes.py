"""Which rays are marched, and how many the march leaves to the ray engine.

Equal bits alone do not show that the march did anything: these tests read how
many rays it took and left.  Ordinary meshes leave next to none; ties, lattices
and cells that are large against a periodic box are left.
"""
import sys

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

import vortrace_amd as vt  # noqa: E402
from vortrace_amd import _lib, synthetic  # noqa: E402

BB = [0.0, 100.0] * 3


def _say(msg):
    print(msg, flush=True)
    sys.stdout.flush()


def _routes(pc, s, e):
    """(rays marched, rays left) of a projection, checked against the engine;
    called often enough that the cloud's lists are built."""
    s, e = [torch.from_numpy(np.ascontiguousarray(x)).cuda() for x in (s, e)]
    for _ in range(60):
        got = pc.projection_tensor(s, e)
        st = _lib.last_march_stats()
        if st.rays:
            break
    pc._cloud.set_march_limit(0)
    want = pc.projection_tensor(s, e)
    assert _lib.last_march_stats().rays == 0
    pc._cloud.set_march_limit(None)
    assert torch.equal(got, want)
    _say(f"  {st.rays} of {len(s)} rays marched, {st.left} left")
    return st.rays, st.left


def _axis(n, seed, box=100.0):
    xy = box * np.random.default_rng(seed).random((n, 2))
    return np.column_stack([xy, np.zeros(n)]), np.column_stack([xy, np.full(n, box)])


def _chords(n, seed, lo=1.0, hi=99.0):
    rng = np.random.default_rng(seed)
    return rng.uniform(lo, hi, (n, 3)), rng.uniform(lo, hi, (n, 3))


@pytest.mark.filterwarnings("ignore::UserWarning")
@pytest.mark.parametrize("periodic", [False, True])
@pytest.mark.parametrize("mesh", ["uniform", "clustered"])
def test_ordinary_meshes_leave_next_to_none(mesh, periodic):
    pos, rho = (synthetic.uniform_mesh(20_000, seed=31) if mesh == "uniform" else
                synthetic.clustered_mesh(60_000, seed=32, n_clumps=30))
    pc = vt.ProjectionCloud(pos, rho, boundbox=BB, periodic=periodic)
    for n in (1, 100, 20_000):
        marched, left = _routes(pc, *(_axis(n, n) if periodic else _chords(n, n)))
        assert marched == n and left <= 1 + n // 1000


def test_ties_are_left():
    rng = np.random.default_rng(9)
    pos = 10.0 * rng.random((3000, 3))
    pos[:500] = np.round(pos[:500])
    pc = vt.ProjectionCloud(pos, rng.random(3000), boundbox=[0.0, 10.0] * 3,
                            vol=np.full(3000, 1.0 / 3))
    s = np.repeat(pos[:200], 5, axis=0) + 0.4 * rng.standard_normal((1000, 3))
    e = np.repeat(np.round(pos[200:400]), 5, axis=0)
    marched, left = _routes(pc, s, e)
    assert marched == 1000 and left > 0


@pytest.mark.parametrize("cells,rays,outside,marched", [
    (100_000, 64, 0, True), (100_000, 64, 1, False), (100_000, 64, 64, False),
    (100_000, 3072, 1, False), (100_000, 3073, 1, True), (99_999, 64, 1, True)])
def test_few_rays_that_leave_an_open_box(cells, rays, outside, marched):
    """Both sides of engine_sooner's lines (12 rays per CU, 256 CUs)."""
    pos, rho = synthetic.uniform_mesh(cells, seed=61)
    pc = vt.ProjectionCloud(pos, rho, boundbox=BB, periodic=False,
                            vol=np.full(cells, 1e6 / cells))
    # The lists are built by a call that is marched.
    assert _routes(pc, *_chords(5000, 1))[0] == 5000
    s, e = _chords(rays, 9)
    s[:outside, 2] = -20.0
    assert _routes(pc, s, e)[0] == (rays if marched else 0)


def test_own_tree_loaded_is_marched():
    """A tree that bounds the points is marched through also when loaded, one
    that does not is not."""
    pos, rho = synthetic.uniform_mesh(8000, seed=71)
    pc = vt.ProjectionCloud(pos, rho, boundbox=BB, periodic=True)
    own = pc.save_tree_bytes()
    pc.load_tree_bytes(own)
    assert _routes(pc, *_axis(400, 73))[0] == 400
    moved = np.clip(pos + 0.4 * np.random.default_rng(72).standard_normal(pos.shape), 0.0, 100.0)
    q = vt.ProjectionCloud(moved, rho, boundbox=BB, periodic=True)
    q.load_tree_bytes(own)
    for _ in range(3):
        try:
            q.projection(*_axis(100, 73))
        except ValueError:  # searches through such a tree may find nothing
            pass
        assert _lib.last_march_stats().rays == 0


@pytest.mark.filterwarnings("ignore::UserWarning")
@pytest.mark.parametrize("cells,box,rays,marched", [
    (200, 1.0, 500, False), (300, 1.0, 500, True),          # cells large against the box
    (200_000, 100.0, 1000, True), (200_000, 1.0, 1000, False),  # a ray or two would be left
    (200_000, 1.0, 8192, False), (200_000, 1.0, 8193, True),    # (32 rays per CU, 256 CUs)
    (600_000, 1.0, 2900, False), (600_000, 1.0, 3100, True),    # (7e6 rays x cells per CU)
    (200_000, 1.0, 100, True), (100_000, 0.03, 20_000, False)])  # next to none; most
def test_where_a_march_does_not_pay(cells, box, rays, marched):
    """Both sides of march_pays's lines, in periodic boxes."""
    pos, rho = synthetic.uniform_mesh(cells, seed=63)
    pc = vt.ProjectionCloud(box * (pos / 100.0), rho, boundbox=[0.0, box] * 3, periodic=True)
    if cells >= 200_000:
        assert _routes(pc, *_axis(20_000, 1, box))[0] == 20_000  # the lists are built
    assert _routes(pc, *_axis(rays, 2, box))[0] == (rays if marched else 0)


def test_lattice_is_left():
    """Split points on the cells' faces: every ray is left, in the order it had."""
    g = (np.arange(24) + 0.5) / 24
    pos = np.stack(np.meshgrid(g, g, g, indexing="ij"), -1).reshape(-1, 3)
    pc = vt.ProjectionCloud(pos, np.random.default_rng(1).random(len(pos)) + 0.5,
                            boundbox=[0.0, 1.0] * 3, vol=np.full(len(pos), 24.0 ** -3))
    x = (np.arange(100) + 0.5) / 100
    xy = np.stack(np.meshgrid(x, x, indexing="ij"), -1).reshape(-1, 2)
    z = np.zeros(len(xy))
    assert _routes(pc, np.column_stack([xy, z]), np.column_stack([xy, z + 1.0])) == (10_000, 10_000)


def test_rows_of_more_than_640_cells():
    """Clouds of more than 11M cells: rows of 704 cells, 512 intervals a wave in the
    march's check."""
    n = 11_500_000
    pos, rho = synthetic.uniform_mesh(n, seed=65)
    pc = vt.ProjectionCloud(pos, rho, boundbox=BB, periodic=True)
    marched, left = _routes(pc, *_axis(500_000, 3))
    assert marched == 500_000 and left < 500  # (some ten meet a near-tie)


def test_autotune_times_marched_calls():
    """A few rays through a large cloud: lists are built before anything is timed."""
    pos, rho = synthetic.uniform_mesh(600_000, seed=67)
    pc = vt.ProjectionCloud(pos, rho, boundbox=BB, periodic=True)
    saved = vt.tuning.get_tuning()
    marched = []
    try:
        project = pc.projection_tensor

        def seen(*a, **kw):
            out = project(*a, **kw)
            marched.append((vt.tuning.get_tuning()["help_events"], _lib.last_march_stats().rays))
            return out
        pc.projection_tensor = seen
        out = vt.tuning.autotune(pc, *_axis(64, 5), stride=1, walk_batches=(32,),
                                 leaf_batches=(32,), ray_parts=(8,), help_events=(0, 128),
                                 repeats=2, cache=False)
    finally:
        vt.tuning.set_tuning(**saved)
    assert [r for r in marched[-4:]] == [(0, 0), (0, 0), (128, 64), (128, 64)]
    assert len(out["results"]) == 2
