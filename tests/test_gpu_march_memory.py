"""The march's device memory is optional: a call that finds no room for it runs
in smaller batches or in the ray engine, and an allocation that a call cannot
do without gets it back -- whichever cloud holds it.
"""
import sys
import threading

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

import vortrace_amd as vt  # noqa: E402
from vortrace_amd import synthetic  # noqa: E402

BB = [0.0, 100.0] * 3
GIB = 1 << 30


def _say(msg):
    print(msg, flush=True)
    sys.stdout.flush()


def _grid(nx, ny):
    x, y = np.meshgrid((np.arange(nx) + 0.5) * (100.0 / nx), (np.arange(ny) + 0.5) * (100.0 / ny),
                       indexing="ij")
    s = np.column_stack([x.ravel(), y.ravel(), np.zeros(nx * ny)])
    return (torch.from_numpy(s).cuda(),
            torch.from_numpy(s + [0.0, 0.0, 100.0]).cuda())


def _cloud(n, seed):
    pos, rho = synthetic.uniform_mesh(n, seed=seed)
    return vt.ProjectionCloud(pos, rho, boundbox=BB, periodic=True)


def _engine(pc, s, e):
    pc._cloud.set_march_limit(0)
    out = pc.projection_tensor(s, e)
    pc._cloud.set_march_limit(None)
    return out


def _hog(leave):
    """A tensor over all free device memory but `leave` bytes."""
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    free, _ = torch.cuda.mem_get_info()
    return torch.empty(max(1, free - leave), dtype=torch.uint8, device="cuda")


def test_rows_do_not_fit():
    """A million rays' rows are 4 GiB; 3 GiB are free."""
    pc = _cloud(200_000, 91)
    s, e = _grid(1024, 1024)
    saved = vt.tuning.get_tuning()
    try:
        vt.tuning.set_tuning(help_events=0)
        want = pc.projection_tensor(s, e)
    finally:
        vt.tuning.set_tuning(**saved)
    _say("filling the device's memory")
    hog = _hog(3 * GIB)
    _say("projecting")
    got = pc.projection_tensor(s, e)
    del hog
    torch.cuda.empty_cache()
    assert torch.equal(got, want)


def test_clouds_give_memory_back():
    """A cloud that fits only into what an idle cloud's march holds."""
    a = _cloud(2_000_000, 92)
    s, e = _grid(512, 512)
    want = a.projection_tensor(s, e)
    pos, rho = synthetic.uniform_mesh(6_000_000, seed=93)
    b = vt.PointCloud()
    b.loadPoints(pos, rho, BB, periodic=True)
    _say("filling the device's memory")
    hog = _hog(int(0.6 * GIB))
    _say("uploading the second cloud")
    b.buildTree()  # 0.7 GiB
    _say("projecting through both")
    p = vt.Projection(s[:5000], e[:5000])
    got = p.project_tensor(b)
    assert torch.equal(a.projection_tensor(s[:5000], e[:5000]), want[:5000])
    del hog
    torch.cuda.empty_cache()
    b.set_march_limit(0)
    assert torch.equal(got, p.project_tensor(b))


@pytest.mark.parametrize("rays", [1, 1000, 16_384, 100_000])
def test_limits(rays):
    """Every limit gives the same bits: no lists, no rows, small batches, all."""
    pc = _cloud(30_000, 94)
    s, e = _grid(400, 250)
    s, e = s[:rays], e[:rays]
    want = _engine(pc, s, e)
    lists = 280 * 30_000
    for limit in (None, 10 ** 12, lists * 2 + 120 * 10 ** 6, lists * 2 + 60 * 10 ** 6, lists * 2,
                  1000, 0, None):
        _say(f"{rays} rays, limit {limit}")
        pc._cloud.set_march_limit(limit)
        assert torch.equal(pc.projection_tensor(s, e), want)
    with pytest.raises(ValueError):
        pc._cloud.set_march_limit(-1)


def test_threads_share_rows():
    """Calls on several clouds at once lease blocks of their own."""
    sizes = [(5_000, (64, 48)), (60_000, (300, 200)), (20_000, (7, 5))]
    work = []
    for k, (n, g) in enumerate(sizes):
        pc = _cloud(n, 95 + k)
        s, e = _grid(*g)
        work.append((pc, s, e, _engine(pc, s, e)))
    torch.cuda.synchronize()
    bad = []

    def run(pc, s, e, want):
        stream = torch.cuda.Stream()
        with torch.cuda.stream(stream):
            for _ in range(10):
                if not torch.equal(pc.projection_tensor(s, e), want):
                    bad.append(len(s))
    threads = [threading.Thread(target=run, args=w) for w in work]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad


def test_lists_wait_for_rays_that_pay_for_them():
    """A cloud that is uploaded and queried holds its tree alone; a few rays run
    without lists until they have cost as much, with the same bits throughout."""
    n = 1_000_000
    pos, rho = synthetic.uniform_mesh(n, seed=99)
    cloud = vt.PointCloud()
    cloud.loadPoints(pos, rho, BB, periodic=True)
    torch.cuda.synchronize()
    free0 = torch.cuda.mem_get_info()[0]
    cloud.buildTree()
    _say("queries")
    ids, _ = cloud.query_tensor(torch.rand(1000, 3, dtype=torch.float64) * 100.0, 2)
    assert ids.shape == (1000, 2)
    assert free0 - torch.cuda.mem_get_info()[0] < 200 * n + (1 << 30), "lists before any ray"
    s, e = _grid(3, 5)
    p = vt.Projection(s, e)
    first = p.project_tensor(cloud)
    free1 = torch.cuda.mem_get_info()[0]
    for _ in range(40):
        assert torch.equal(p.project_tensor(cloud), first)
    assert free1 - torch.cuda.mem_get_info()[0] > 200 * n, "no lists after forty calls"


def test_lists_dropped_while_other_clouds_project():
    """One thread takes lists away as a failing allocation would, others project."""
    work = []
    for k, n in enumerate((4_000, 9_000)):
        pc = _cloud(n, 110 + k)
        s, e = _grid(60, 40)
        work.append((pc, s, e, _engine(pc, s, e)))
    torch.cuda.synchronize()
    stop, bad = threading.Event(), []

    def run(pc, s, e, want):
        with torch.cuda.stream(torch.cuda.Stream()):
            for _ in range(60):
                if not torch.equal(pc.projection_tensor(s, e), want):
                    bad.append(len(s))

    def hog():
        c = vt.PointCloud()
        c.loadPoints(np.random.default_rng(0).random((500, 3)), np.ones(500),
                     [0.0, 1.0] * 3, periodic=True)
        c.buildTree()
        q = torch.rand(64, 3, dtype=torch.float64, device="cuda")
        first = c.query_tensor(q, 2)[0]
        refused = 0
        while not stop.is_set():
            try:
                c.set_ray_order(order)  # a copy of 4 GiB: the library frees what it can
            except RuntimeError:
                refused += 1
            # The refusal is not the next call's.
            if not torch.equal(c.query_tensor(q, 2)[0], first):
                bad.append("query")
        taken.append(refused)
    taken = []
    _say("filling the device's memory")
    order = torch.zeros(1 << 30, dtype=torch.int32, device="cuda")
    hog_mem = _hog(3 * GIB)
    threads = [threading.Thread(target=run, args=w) for w in work]
    taker = threading.Thread(target=hog)
    _say("projecting")
    taker.start()
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    stop.set()
    taker.join()
    del hog_mem, order
    torch.cuda.empty_cache()
    assert not bad
    assert taken and taken[0] > 0
