"""The convolution returns its input's product with G at a scale of one: the part
of the error that lies along the result itself, |<y, Gx> / <Gx, Gx> - 1| for a
random x, stays under 3e-8 (half the distance of 1 from the next FP32 value
below), where the rounded twiddle factors of three axes alone would leave up to
2e-7.  Register kernels, the plane kernel, LDS-staged passes one at a time and
all together, both backends."""
import numpy as np
import pytest

from ddscat_hip import BACKEND_FFT3D, BACKEND_SLICES
from oracle import ddscat_oracle as O

pytestmark = pytest.mark.gpu

DIMS = [(200, 200, 4), (4, 200, 200), (128, 8, 128), (162, 6, 162), (75, 75, 20), (48, 48, 48), (54, 54, 54), (50, 50, 50),
        (12, 12, 12), (10, 10, 10), (8, 256, 64), (12, 384, 15), (7, 280, 7), (256, 6, 6)]


@pytest.mark.parametrize("dims", DIMS)
def test_scale(lib, dims):
    nx, ny, nz = dims
    nat = nx * ny * nz
    rng = np.random.default_rng(nat)
    x = (rng.normal(size=3 * nat) + 1j * rng.normal(size=3 * nat)).astype(np.complex64)
    zero = np.zeros(3 * nat, np.complex64)
    iocc = np.ones(nat, np.int16)
    akd = 0.126
    ref = O.matvec_fft("N", x, zero, zero, O.green_octant(nx, ny, nz, np.float64(np.float32(akd))), nx, ny, nz, iocc)

    def gain(what):
        y = lib.apply("N", x, zero, zero).astype(np.complex128)
        g = np.vdot(ref, y - ref).real / np.vdot(ref, ref).real
        print(f"{dims} {what}: {g:+.2e}")
        assert abs(g) < 3e-8, what

    try:
        for backend in (BACKEND_FFT3D, BACKEND_SLICES):
            lib.set_backend(backend)
            lib.prepare_green(nx, ny, nz, iocc, (akd, 0.0, 0.0))
            gain(f"backend {backend}")
            lib.set_fft_kernels(1)
            gain(f"backend {backend}, LDS-staged")
            lib.set_fft_kernels(0)
            if backend == BACKEND_FFT3D:
                for p in (3, 5, 1, 2, 4):
                    lib.set_pass_kernel(p, -1)
                    gain(f"passes up to {p} LDS-staged")
    finally:
        lib.set_fft_kernels(0)
        lib.release()
        lib.set_backend(BACKEND_FFT3D)
