"""Where the row support is in use (ddscat_hip_info): on sparse targets whose x
spectra pass 256 MiB and whose y kernels honour it, not on a full block of the
same grid, not on a target whose spectra fit 256 MiB, not with y lengths whose
kernels do not honour it, and not while any of passes 1, 2, 4 and 5 or the whole
family is LDS-staged; it comes back with the register kernels."""
import numpy as np
import pytest

from ddscat_hip import BACKEND_FFT3D, BACKEND_SLICES

pytestmark = pytest.mark.gpu


def target(dims, shape):
    nx, ny, nz = dims
    if shape == "block":
        return np.ones(nx * ny * nz, np.int16)
    z, y, x = np.meshgrid(np.arange(nz), np.arange(ny), np.arange(nx), indexing="ij")
    occ = (((x - nx / 2) / (0.5 * nx)) ** 2 + ((y - 0.45 * ny) / (0.4 * ny)) ** 2 + ((z - 0.4 * nz) / (0.3 * nz)) ** 2) < 1
    if shape == "holes":
        occ &= (x + y) % 7 != 0
    return occ.astype(np.int16).reshape(-1)


@pytest.fixture
def slot(lib):
    yield lib
    lib.set_fft_kernels(0)
    lib.release()
    lib.set_backend(BACKEND_FFT3D)


@pytest.mark.parametrize("dims,backend,shape", [((80, 384, 192), BACKEND_FFT3D, "interval"),
                                                ((128, 256, 200), BACKEND_FFT3D, "holes"),
                                                ((250, 256, 100), BACKEND_FFT3D, "interval"),
                                                ((96, 256, 256), BACKEND_SLICES, "holes")])
def test_in_use(slot, dims, backend, shape):
    slot.set_backend(backend)
    slot.prepare_green(*dims, target(dims, shape), (0.2, 0.0, 0.0))
    assert slot.info()["row_support"] == 1
    slot.set_fft_kernels(1)
    assert slot.info()["row_support"] == 0
    slot.set_fft_kernels(0)
    assert slot.info()["row_support"] == 1
    if backend == BACKEND_FFT3D:
        for p in (1, 2, 4, 5):
            kind = slot.info()[f"kernel_pass{p}"]
            slot.set_pass_kernel(p, -1)
            assert slot.info()["row_support"] == 0, p
            slot.set_pass_kernel(p, kind)
            assert slot.info()["row_support"] == 1, p
    slot.prepare_green(*dims, target(dims, "block"), (0.2, 0.0, 0.0))
    assert slot.info()["row_support"] == 0


@pytest.mark.parametrize("dims", [(16, 256, 64), (128, 250, 216)])
def test_not_in_use(slot, dims):
    slot.prepare_green(*dims, target(dims, "interval"), (0.2, 0.0, 0.0))
    assert slot.info()["row_support"] == 0
