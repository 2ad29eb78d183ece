"""The FP64 kernel function of the pair loops against long double, from distances of 1e-6 to
1e7 wavelengths and for coincident points, through the kernel matrix and the direct sum (a
unit density, whose sum over one source is the kernel value itself).

Error of |G| r (kernel 0) or |G| (kernel 1), u = 2^-53: r^2 is three roundings (1.5 u of r), the
root one more, times the phase 2 pi r; sin, cos, 1/r and their product a few u each."""
import numpy as np
import pytest

from ddfmm_amd.wave3d import Kernel3d, direct_sum

pytestmark = pytest.mark.gpu

U = 2.0 ** -53


@pytest.mark.parametrize("kernel", [0, 1])
@pytest.mark.parametrize("scale", [1e-6, 1e-2, 1.0, 40.0, 1e7])
def test_values(scale, kernel):
    rng = np.random.default_rng(7)
    t = rng.uniform(-scale, scale, (257, 3))
    s = rng.uniform(-scale, scale, (65, 3))
    s[0] = t[0]
    g = Kernel3d(kernel).kernel(t.T, s.T)
    d = (t[:, None] - s[None]).astype(np.longdouble)
    r = np.sqrt((d ** 2).sum(-1))
    r[r ** 2 < 1e-16] = 1
    a = np.longdouble("6.28318530717958647692528676655900577") * (r - np.floor(r))
    ref = np.cos(a) + 1j * np.sin(a)
    if kernel == 0:
        ref = ref / r
    err = np.abs(g - ref) * (r if kernel == 0 else 1) / ((2.5 * 2 * np.pi * r + 8) * U)
    print(f"scale {scale:g} kernel {kernel}: {float(err.max()):.2f} of the bound", flush=True)
    assert err.max() < 1
    for j in (0, 64):
        assert np.array_equal(direct_sum(t, s[j:j + 1], np.ones(1), kernel), g[:, j]), j
