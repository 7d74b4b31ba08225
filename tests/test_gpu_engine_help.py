"""The ray engine's helping, with no march before it.

A march limit of 0 runs every ray of a cloud in the engine, whose idle lanes
walk intervals of busy lanes' rays and record up to help_events boundaries of
each.  Every setting must give the bits of the plain walk: 0 (no helping), 1
and 3 (almost every interval is handed back), 128; by the kernels that project,
count, list segments and feed the adjoint.  Launches of more rays than
workgroups, so that the recorded boundaries are as many as help_events says.
"""
import sys

import numpy as np
import pytest
import torch

from oracle import port

pytestmark = pytest.mark.gpu

import vortrace_amd as vt  # noqa: E402
from vortrace_amd import _lib, synthetic  # noqa: E402

BB = [0.0, 100.0] * 3
RAYS = 3000


def _say(msg):
    print(msg, flush=True)
    sys.stdout.flush()


@pytest.fixture()
def tuning():
    saved = vt.tuning.get_tuning()
    yield
    vt.tuning.set_tuning(**saved)


def _cloud(periodic, nf):
    if periodic:
        pos, rho = synthetic.clustered_mesh(60_000, seed=13, n_clumps=30)
        xy = 100.0 * np.random.default_rng(5).random((RAYS, 2))
        s = np.column_stack([xy, np.zeros(RAYS)])
        e = np.column_stack([xy, np.full(RAYS, 100.0)])
    else:
        pos, rho = synthetic.uniform_mesh(30_000, seed=11)
        rng = np.random.default_rng(12)
        s, e = rng.uniform(0.0, 100.0, (RAYS, 3)), rng.uniform(0.0, 100.0, (RAYS, 3))
    f = np.stack([rho, rho * rho, np.sqrt(rho)], axis=1)[:, :nf]
    kw = {} if periodic else {"vol": np.full(len(pos), 1e6 / len(pos))}
    pc = vt.ProjectionCloud(pos, f if nf > 1 else rho, boundbox=BB, periodic=periodic, **kw)
    pc._cloud.set_march_limit(0)
    oracle = port.OracleCloud(pos, f, BB, periodic=periodic, **kw)
    return pc, oracle, s, e


def _stats(out, key):
    st = _lib.last_call_stats()
    assert _lib.last_march_stats().rays == 0, "marched"
    out[key] = (st.intervals, st.intervals_back)


@pytest.mark.parametrize("periodic,nf", [(False, 1), (True, 1), (True, 3)])
def test_every_setting_gives_the_same_bits(tuning, periodic, nf):
    pc, oracle, s, e = _cloud(periodic, nf)
    ds, de = torch.from_numpy(s).cuda(), torch.from_numpy(e).cuda()
    g = torch.from_numpy(np.random.default_rng(7).standard_normal((RAYS, nf))).cuda()
    res, shared = {}, {}
    for he in (0, 1, 3, 128):
        vt.tuning.set_tuning(help_events=he)
        _say(f"periodic {periodic}, {nf} fields, help_events {he}")
        out, st = {}, {}
        for m in ("sum", "max", "min"):
            out[m] = pc.projection(s, e, reduction=m)
            _stats(st, m)
        p = vt.Projection(ds, de)
        out["traced"] = [x.cpu().numpy() for x in p.segments_tensor(pc._cloud, vt.ReductionMode.Sum)]
        _stats(st, "fill")
        out["adjoint"] = p.adjoint_tensor(pc._cloud, g).cpu().numpy()
        _stats(st, "segs")
        res[he], shared[he] = out, st
    for he in (1, 3, 128):
        for k, want in res[0].items():
            for a, b in zip(res[he][k], want) if k == "traced" else [(res[he][k], want)]:
                np.testing.assert_array_equal(a, b, err_msg=f"{k}, help_events {he}")
    for k in shared[0]:
        assert shared[0][k] == (0, 0), k
        assert shared[128][k][0] > 0, f"{k}: no interval was given"
        assert min(shared[1][k]) > 0, f"{k}: no interval came back at help_events 1"
    want = oracle.project(s, e, "sum")
    np.testing.assert_array_equal(res[128]["sum"], want if nf > 1 else want[:, 0])


def test_recorded_forward(tuning):
    """The kernels that record their segments help too."""
    pc, _, s, e = _cloud(True, 1)
    fields = torch.from_numpy(np.asarray(pc.fields_orig, dtype=np.float64).reshape(-1)).cuda()
    ds, de = torch.from_numpy(s).cuda(), torch.from_numpy(e).cuda()
    res = []
    for he in (0, 1, 128):
        vt.tuning.set_tuning(help_events=he)
        _say(f"recorded, help_events {he}")
        f = fields.clone().requires_grad_(True)
        for _ in range(2):  # the second pass has its record pool sized
            f.grad = None
            img = pc.projection_grad(ds, de, f, reduction="sum")
            (img * img).sum().backward()
        assert _lib.last_march_stats().rays == 0
        assert (pc._forward_stats.intervals > 0) == (he > 0)
        res.append((img.detach(), f.grad))
    for img, grad in res[1:]:
        assert torch.equal(img, res[0][0]) and torch.equal(grad, res[0][1])


def test_left_rays_are_walked_once(tuning):
    """Rays of some 240 cells, 160 of them in a dense slab, many left by the march:
    an interval that its walker has no room for is handed back and walked again,
    by every giver above it, so the leftovers need room for whole intervals."""
    rng = np.random.default_rng(17)
    h = 2e-3
    g = np.stack(np.meshgrid(np.arange(24), np.arange(24), np.arange(110), indexing="ij"), -1)
    slab = 50.0 + h * (g.reshape(-1, 3) + 0.25 + 0.5 * rng.random((24 * 24 * 110, 3)))
    pos = np.concatenate([slab, 100.0 * rng.random((400_000, 3))])
    pc = vt.ProjectionCloud(pos, rng.random(len(pos)), boundbox=BB, periodic=True)
    x = 50.0 + h * (2.0 + 20.0 * (np.arange(64) + 0.5) / 64)
    xy = np.stack(np.meshgrid(x, x, indexing="ij"), -1).reshape(-1, 2)
    s = torch.from_numpy(np.column_stack([xy, np.zeros(4096)])).cuda()
    e = s + torch.tensor([0.0, 0.0, 100.0], dtype=torch.float64, device="cuda")
    for _ in range(40):  # until the lists are built
        got = pc.projection_tensor(s, e)
        m = _lib.last_march_stats()
        if m.rays:
            break
    st = _lib.last_call_stats()
    given, back = st.intervals - m.intervals, st.intervals_back - m.intervals_back
    _say(f"  {m.left} of {m.rays} rays left, {given} intervals given, {back} handed back")
    assert m.left >= 512, "fewer rays than workgroups"
    assert 200 <= st.segments / len(s) <= 300, "rays of other lengths than meant"
    assert given > 0 and back == 0
    vt.tuning.set_tuning(help_events=0)
    assert torch.equal(pc.projection_tensor(s, e), got)
