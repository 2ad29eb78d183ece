"""The translation GEMM's forms at the counts where the launch changes: one or two column
blocks per wave (32 right-hand sides up, K not blocked, large stages), partial column tiles
and planned tiles whose columns do not fill whole waves.  The form never changes a column's
order of summation, so a right-hand side keeps its bits in every batch, and the mixed mode
stays within its FP32 distance (3e-6, the bound of the other mixed-mode tests) of FP64 FMM."""
import numpy as np
import pytest

from ddfmm_amd import geometry
from ddfmm_amd.wave3d import FP64, MIXED, Kernel3d, Mlib3d, Wave3d

pytestmark = pytest.mark.gpu


def _wave(pos, K, ops, precision, nrhs_max, kernel):
    ml = Mlib3d()
    ml.setup({"-mlib3d_ldname": ops[0], "-mlib3d_hdname": ops[1]})
    w = Wave3d()
    w.posptr, w.mlibptr, w.kernel = pos, ml, Kernel3d(kernel)
    w.setup({"-wave3d_ACCU": 2, "-wave3d_K": K, "-wave3d_maxlevel": 12}, nrhs_max=nrhs_max, precision=precision)
    return w


@pytest.mark.parametrize("kernel", [0, 1])
def test_counts_keep_bits(oplib, oplib_expr, kernel):
    K, N = 8.0, 45007
    ops = oplib_expr if kernel else oplib
    pos = geometry.sphere(N, K, 51)
    den = geometry.densities(N, 52, nrhs=65)
    w = _wave(pos, K, ops, MIXED, 65, kernel)
    full = w.eval(den)
    for lo, hi in ((0, 1), (1, 32), (0, 32), (32, 65), (1, 65)):      # 1, 31, 32, 33, 64
        got = w.eval(den[lo] if hi - lo == 1 else den[lo:hi])
        assert np.array_equal(np.atleast_2d(got), full[lo:hi]), (lo, hi)
    w.close()
    w = _wave(pos, K, ops, FP64, 2, kernel)
    ref = w.eval(den[[0, 64]])
    w.close()
    d = float(np.linalg.norm(full[[0, 64]] - ref) / np.linalg.norm(ref))
    print(f"kernel {kernel}: mixed vs FP64 {d:.2e}", flush=True)
    assert d < (1e-4 if kernel else 3e-6)
