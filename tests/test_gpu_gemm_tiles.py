"""The GEMM kernel at every tile height, which sets how many units of k a pipeline step holds:
a column's order of k is the same at each, so FP64 and mixed potentials keep their bits, at 1
and 5 right-hand sides, for both kernels (three or four real products)."""
import numpy as np
import pytest

from ddfmm_amd import geometry
from ddfmm_amd.wave3d import FP64, MIXED, Kernel3d, Mlib3d, Wave3d

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [FP64, MIXED])
@pytest.mark.parametrize("kernel", [0, 1])
def test_heights_keep_bits(oplib, oplib_expr, kernel, precision):
    K, N = 4.0, 6007
    ops = oplib_expr if kernel else oplib
    den = geometry.densities(N, 62, nrhs=5)
    ml = Mlib3d()
    ml.setup({"-mlib3d_ldname": ops[0], "-mlib3d_hdname": ops[1]})
    w = Wave3d()
    w.posptr, w.mlibptr, w.kernel = geometry.sphere(N, K, 61), ml, Kernel3d(kernel)
    w.setup({"-wave3d_ACCU": 2, "-wave3d_K": K, "-wave3d_maxlevel": 12}, nrhs_max=5, precision=precision)
    ref = w.eval(den)
    table, _ = w.tiles()
    for mb in range(1, 8):
        w.set_tiles([mb] * len(table))
        assert np.array_equal(w.eval(den), ref), mb
        assert np.array_equal(w.eval(den[4]), ref[4]), mb
    w.close()
