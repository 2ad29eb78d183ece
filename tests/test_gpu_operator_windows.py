"""The operator table made in many small pieces (a budget of the tables and one right-hand
side: each piece is at most that one's buffers) against the pieces of an unlimited context,
and both against the oracle's direct sum: the same bits in every precision and for both
kernels, one pass of two right-hand sides or two passes of one."""
import numpy as np
import pytest

from ddfmm_amd import geometry
from ddfmm_amd.wave3d import FP64, FP64_FUSED, MIXED, MIXED_SPLIT, Kernel3d, Mlib3d, Wave3d, direct_sum

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [FP64, MIXED, FP64_FUSED, MIXED_SPLIT])
@pytest.mark.parametrize("kernel", [0, 1])
def test_small_windows_keep_bits(oplib, oplib_expr, kernel, precision):
    K, N = 4.0, 6003
    ld, hd = oplib_expr if kernel else oplib
    pos, den = geometry.sphere(N, K, 91), geometry.densities(N, 92, nrhs=2)
    ml = Mlib3d()
    ml.setup({"-mlib3d_ldname": ld, "-mlib3d_hdname": hd})

    def wave(budget):
        w = Wave3d()
        w.posptr, w.mlibptr, w.kernel = pos, ml, Kernel3d(kernel)
        w.setup({"-wave3d_ACCU": 2, "-wave3d_K": K, "-wave3d_maxlevel": 12, "-wave3d_hbm_budget": budget / 2**30},
                nrhs_max=2, precision=precision)
        return w

    w = wave(0)
    ref, m = w.eval(den), w.memory()
    w.close()
    w = wave(m["fixed_bytes"] + m["per_rhs_bytes"] + 1024)
    b = w.memory()
    print(f"kernel {kernel} precision {precision}: setup {m['setup_bytes']} -> {b['setup_bytes']}", flush=True)
    assert b["slab"] == 1 and b["setup_bytes"] < 0.6 * m["setup_bytes"]
    assert np.array_equal(w.eval(den), ref)
    w.close()
    chk = geometry.check_targets(N, 200, 93)
    exact = direct_sum(pos[chk], pos, den, kernel)
    err = float(np.linalg.norm(ref[:, chk] - exact) / np.linalg.norm(exact))
    assert err < (0.1 if kernel else 1e-5), err      # e^{ikr}: the method's own limit is about 5e-2
