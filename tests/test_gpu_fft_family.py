"""The FFT kernel family chosen on a prepared target (ddscat_hip_set_fft_kernels):
every pass of the next MATVEC is of that family, also on small grids, where one
kernel replaces passes 2 to 4.  With the LDS-staged family the products are, bit
for bit, those of a target prepared with it; back at the register family, those
from before.  The two families agree within the rounding of FP32 transforms
(5e-7)."""
import numpy as np
import pytest

from ddscat_hip import BACKEND_FFT3D, BACKEND_SLICES

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("backend", [BACKEND_FFT3D, BACKEND_SLICES])
@pytest.mark.parametrize("n,plane", [(32, 1), (60, 0)])
def test_family_on_prepared_target(lib, n, plane, backend):
    rng = np.random.default_rng(n)
    iocc = np.ones(n ** 3, np.int16)
    cx = lambda s: (s * (rng.normal(size=3 * n ** 3) + 1j * rng.normal(size=3 * n ** 3))).astype(np.complex64)
    args = cx(1.0), cx(1.0), cx(0.3)
    try:
        lib.set_backend(backend)
        lib.prepare_green(n, n, n, iocc, (0.3, 0.0, 0.0))
        assert lib.info()["plane_kernel"] == plane
        reg = lib.apply("N", *args)
        lib.set_fft_kernels(1)
        assert lib.info()["plane_kernel"] == 0
        staged = lib.apply("N", *args)
        lib.set_fft_kernels(0)
        assert lib.info()["plane_kernel"] == plane
        assert np.array_equal(lib.apply("N", *args), reg)
        lib.set_fft_kernels(1)
        lib.prepare_green(n, n, n, iocc, (0.3, 0.0, 0.0))
        assert np.array_equal(lib.apply("N", *args), staged)
        assert 0 < np.linalg.norm(staged - reg) < 5e-7 * np.linalg.norm(reg)
    finally:
        lib.set_fft_kernels(0)
        lib.release()
        lib.set_backend(BACKEND_FFT3D)
