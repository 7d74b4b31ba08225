"""Exits that a float key cannot tell apart.

Generators in close pairs and triples (1e-7 to 1e-5 apart in a unit box): the keys
of two exits are then often the same float, and every lane of a ray's group has
to take the same one for the nearer -- the group reads that generator's list and
searches around its exit together.  The rays start far outside, so cells' lists
seldom reach their exits.  Ray counts for 16, 8 and 4 lanes a ray.
"""
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

import vortrace_amd as vt  # noqa: E402


def _say(msg):
    print(msg, flush=True)
    sys.stdout.flush()


def _cloud(rng, n, gap, periodic):
    pos = rng.random((n, 3))
    k = n // 2
    pos[:k] = pos[rng.integers(k, n, k)] + gap * rng.standard_normal((k, 3))
    pos = np.clip(pos, 0.0, 1.0)
    kw = {} if periodic else {"vol": np.full(n, 1.0 / n)}
    return vt.ProjectionCloud(pos, rng.random(n) + 0.5, boundbox=[0.0, 1.0] * 3,
                              periodic=periodic, **kw)


@pytest.mark.filterwarnings("ignore::UserWarning")
@pytest.mark.parametrize("periodic", [False, True])
@pytest.mark.parametrize("rays", [4000, 20_000, 70_000])
@pytest.mark.parametrize("gap", [1e-7, 1e-6, 1e-5])
def test_pairs_of_generators(rays, gap, periodic):
    rng = np.random.default_rng(int(rays / gap) % 1_000_003 + periodic)
    saved = vt.tuning.get_tuning()
    try:
        for n in (40, 240, 1500) if not periodic else (600, 1500):
            pc = _cloud(rng, n, gap, periodic)
            if periodic:
                s = np.column_stack([rng.random((rays, 2)), np.full(rays, 0.02)])
                e = s + [0.0, 0.0, 0.9]
            else:
                s, e = rng.uniform(-3.0, 4.0, (2, rays, 3))
            got = []
            for he in (0, 128):
                vt.tuning.set_tuning(help_events=he)
                _say(f"  {n} cells, pairs {gap}, {rays} rays, help_events {he}")
                for _ in range(1 if he == 0 else 3):  # (the lists are built)
                    out = pc.projection(s, e)
                got.append(out)
            np.testing.assert_array_equal(got[1], got[0], err_msg=f"{n} cells")
    finally:
        vt.tuning.set_tuning(**saved)
