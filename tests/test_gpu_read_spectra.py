"""ddfmm_read_buffer on the V-list spectra, whose right-hand sides lie side by side: each
right-hand side of a pass of three reads as the same one evaluated alone."""
import numpy as np
import pytest

from ddfmm_amd import geometry
from ddfmm_amd._lib import DdfmmError
from ddfmm_amd.wave3d import FP64, MIXED, Mlib3d, Wave3d

pytestmark = pytest.mark.gpu

BUF_SPEC, BUF_TSPEC = 10, 12      # plan.hpp numbering


@pytest.mark.parametrize("precision", [FP64, MIXED])
def test_spectra_by_right_hand_side(oplib, precision):
    K, N = 4.0, 6000
    den = geometry.densities(N, 37, nrhs=3)
    ml = Mlib3d()
    ml.setup({"-mlib3d_ldname": oplib[0], "-mlib3d_hdname": oplib[1]})
    w = Wave3d()
    w.posptr, w.mlibptr = geometry.sphere(N, K, 36), ml
    w.setup({"-wave3d_ACCU": 2, "-wave3d_K": K, "-wave3d_maxlevel": 12}, nrhs_max=3, precision=precision)
    read = lambda b, r: w.read_buffer(b, 1728 + 5, 3 * 1728, r)
    alone = []
    for d in den:
        w.eval(d)
        alone.append([read(b, 0) for b in (BUF_SPEC, BUF_TSPEC)])
    w.eval(den)
    for r in range(3):
        for b, ref in zip((BUF_SPEC, BUF_TSPEC), alone[r]):
            assert np.abs(ref).max() > 0
            assert np.array_equal(read(b, r), ref), (b, r)
    w.eval(den[0])
    with pytest.raises(DdfmmError, match="last pass"):
        read(BUF_SPEC, 1)
    w.close()
