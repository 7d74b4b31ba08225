"""Which grids grid.device_view hands to the device generator (no GPU).

The device computes a view in FP64 alone (grid_ray in vt_hip.hip); numpy
computes it in the types it is given.  Every grid that device_view takes must
come out the same, over the kinds of extent, resolution, bounds and centre a
caller can pass: narrow and unsigned integers divide and wrap in their own
type, long doubles round once instead of twice.
"""
import itertools

import numpy as np
import pytest

from vortrace_amd import grid


def _device_grid(v):
    """The rays of a view record, as the device computes them: FP64, every
    operation rounded on its own (numpy.linspace's steps; fused products with
    the identity's zeros and ones are exact)."""
    def centres(lo, hi, n):
        d = (hi - lo) / n
        a, b = lo + 0.5 * d, hi - 0.5 * d
        if n == 1:
            return np.array([0.0 * (b - a) + a])
        i = np.arange(n, dtype=np.float64)
        step = (b - a) / (n - 1)
        x = i * step + a if step != 0.0 else (i / (n - 1)) * (b - a) + a
        x[-1] = b
        return x
    e = [np.float64(x) for x in v.extent]
    x, y = centres(e[0], e[1], int(v.nx)), centres(e[2], e[3], int(v.ny))
    out = np.empty((2, int(v.nx), int(v.ny), 3))
    out[..., 0] = x[:, None]
    out[..., 1] = y[None, :]
    out[0, ..., 2], out[1, ..., 2] = v.bounds[0], v.bounds[1]
    if v.rotate:
        c = np.array(list(v.center))
        assert list(v.rot) == np.eye(3).ravel().tolist()
        out = (out - c) + c
    return out[0], out[1]


EXTENTS = [
    [0.0, 10.0], [0, 10], (3, 7.5), [10.0, 0.0], [[0.1, 9.7], [2.3, 2.9]], [-3, 2 ** 51],
    [1e-310, 3e-310], np.array([0.0, 10.0]), np.array([[0, 10], [5, 1]]),
    np.array([-100, 100], np.int8), np.array([0, 10], np.int16), np.array([10, 0], np.uint8),
    np.array([7, 3], np.uint16), np.array([0, 10], np.int32),
    np.array([-2_000_000_000, 2_000_000_000], np.int32), np.array([10, 0], np.uint32),
    np.array([10, 0], np.uint64), np.array([0.0, 10.0], np.float32),
    np.array([0.0, 10.0], np.float16), np.array([0.0, 10.0], np.longdouble),
]
BOUNDS = [
    [0.0, 10.0], (10, 0), np.array([0.0, 10.0], np.float32), np.array([200, 0], np.uint8),
    np.array([-100, 100], np.int8), np.array([0, 2 ** 63], np.uint64),
    np.array([0.1, 10.1], np.longdouble) / 3,
]
CENTRES = [
    None, [5.0, 5.0, 5.0], (1, 2, 3), np.array([5, 4, 3], np.int8),
    np.array([0.3, 0.1, 0.7], np.float32), np.array([1, 1, 1], np.longdouble) / 3,
]


@pytest.mark.parametrize("extent", EXTENTS, ids=lambda e: f"{np.asarray(e).dtype}-{e!r}"[:40])
def test_taken_grids_equal_numpy(extent):
    taken = 0
    for bounds, centre, nres, proj in itertools.product(
            BOUNDS, CENTRES, (1, 7, (3, np.int64(5)), [2, np.int8(9)]), (None, "xy", "yx")):
        with np.errstate(all="ignore"):
            try:
                view = grid.device_view(extent, nres, bounds, centre, proj=proj)
            except Exception as ex:  # noqa: BLE001 -- numpy must raise the same
                with pytest.raises(type(ex)):
                    grid.generate_projection_grid(extent, nres, bounds, centre, proj=proj)
                continue
            if view is None:
                continue
            taken += 1
            want = grid.generate_projection_grid(extent, nres, bounds, centre, proj=proj)
            got = _device_grid(view)
        for a, b in zip(got, want):
            np.testing.assert_array_equal(a, b, err_msg=f"{extent!r} {bounds!r} {centre!r} {nres}")
    if np.asarray(extent).dtype in (np.float64, np.int64):
        assert taken, "an ordinary grid is not built on the device"
