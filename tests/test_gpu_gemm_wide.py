"""Every tile-height limit at 16 and 33 right-hand sides, where FP32 waves are blocks of their
own and, with three products (e^{ikr}/r) at 33, take two column blocks: each right-hand side
keeps the bits that it has at the planner's heights.  Limits 1 to 7 reach tiles of 1 to 7 row
blocks for e^{ikr}/r, of 1 to 5 and 7 for e^{ikr} (no operator of its library splits into 6)."""
import numpy as np
import pytest

from ddfmm_amd import geometry
from ddfmm_amd.wave3d import MIXED, Kernel3d, Mlib3d, Wave3d

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kernel", [0, 1])
def test_heights_keep_bits_at_many_rhs(oplib, oplib_expr, kernel):
    K, N = 8.0, 30011
    ops = oplib_expr if kernel else oplib
    den = geometry.densities(N, 64, nrhs=33)
    ml = Mlib3d()
    ml.setup({"-mlib3d_ldname": ops[0], "-mlib3d_hdname": ops[1]})
    w = Wave3d()
    w.posptr, w.mlibptr, w.kernel = geometry.sphere(N, K, 63), ml, Kernel3d(kernel)
    w.setup({"-wave3d_ACCU": 2, "-wave3d_K": K, "-wave3d_maxlevel": 12}, nrhs_max=33, precision=MIXED)
    ref = w.eval(den)
    for mb in range(1, 8):
        w.set_tiles([mb] * len(w.tiles()[0]))
        assert np.array_equal(w.eval(den), ref), mb
        assert np.array_equal(w.eval(den[:16]), ref[:16]), mb
    w.close()
