"""Contexts closed and graphs dropped with a replay still running on a
caller's stream: the replay's results arrive whole."""
import numpy as np
import pytest

from ddfmm_amd import geometry
from ddfmm_amd._lib import Hip
from ddfmm_amd.wave3d import MIXED, Mlib3d, Wave3d

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("end", ["close", "graph off"])
def test_replay_in_flight(oplib, end):
    K, N = 8.0, 20000
    den = np.ascontiguousarray(np.atleast_2d(geometry.densities(N, 35)))
    ml = Mlib3d()
    ml.setup({"-mlib3d_ldname": oplib[0], "-mlib3d_hdname": oplib[1]})
    w = Wave3d()
    w.posptr, w.mlibptr = geometry.sphere(N, K, 34), ml
    w.setup({"-wave3d_ACCU": 2, "-wave3d_K": K, "-wave3d_maxlevel": 12}, precision=MIXED)
    ref = w.eval(den)
    w.set_graph(True)
    hip = Hip()
    st = hip.stream()
    dd, vd = hip.to_device(den), hip.malloc(den.nbytes)
    try:
        for _ in range(4):
            w.eval_device(dd, vd, 1, st)
        if end == "close":
            w.close()
        else:
            w.set_graph(False)
        hip.stream_sync(st)
        assert np.array_equal(hip.to_host(vd, np.empty_like(den)), ref)
    finally:
        w.close()
        hip.free(dd)
        hip.free(vd)
        hip.stream_destroy(st)
