"""What a march leaves behind in its cloud.

A call that is refused half way -- under stream capture its kernels and clears
are recorded and never run -- must leave nothing that a later call counts on:
the later call clears its counters itself.
"""
import ctypes as C
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


def _hip():
    """The HIP runtime that torch has loaded."""
    with open("/proc/self/maps") as f:
        path = next(line.split()[-1] for line in f if "libamdhip64" in line)
    hip = C.CDLL(path)
    hip.hipStreamBeginCapture.argtypes = [C.c_void_p, C.c_int]
    hip.hipStreamEndCapture.argtypes = [C.c_void_p, C.POINTER(C.c_void_p)]
    hip.hipGraphDestroy.argtypes = [C.c_void_p]
    return hip


def test_first_call_refused_under_capture():
    # Clumps: many starts are left to the search, so their list is used.
    pos, rho = synthetic.clustered_mesh(30_000, seed=81, n_clumps=12)
    pc = vt.ProjectionCloud(pos, rho, boundbox=BB, periodic=True)
    xy = 100.0 * np.random.default_rng(82).random((3000, 2))
    s = torch.from_numpy(np.column_stack([xy, np.zeros(3000)])).cuda()
    e = torch.from_numpy(np.column_stack([xy, np.full(3000, 100.0)])).cuda()
    out = torch.zeros(3000, dtype=torch.float64, device="cuda")
    hip, stream = _hip(), torch.cuda.Stream()
    torch.cuda.synchronize()
    _say("a first call while its stream is captured")
    assert hip.hipStreamBeginCapture(stream.cuda_stream, 2) == 0  # relaxed: may allocate
    rc = _lib.lib().vt_project(pc._cloud._handle(), s.data_ptr(), e.data_ptr(), 3000, 0,
                               out.data_ptr(), stream.cuda_stream)
    graph = C.c_void_p()
    hip.hipStreamEndCapture(stream.cuda_stream, C.byref(graph))
    if graph.value:
        hip.hipGraphDestroy(graph)
    hip.hipGetLastError()
    assert rc != 0, "a call that waits for its result cannot be captured"
    _say("the same call, run")
    got = pc.projection_tensor(s, e).cpu().numpy()
    saved = vt.tuning.get_tuning()
    try:
        vt.tuning.set_tuning(help_events=0)
        want = pc.projection_tensor(s, e).cpu().numpy()
    finally:
        vt.tuning.set_tuning(**saved)
    np.testing.assert_array_equal(got, want)
