"""The LDS-staged y passes: y axes without a register kernel on targets of few
planes, where a workgroup's columns cross kx planes, and of plane counts just
under, at and over whole tiles, with a row of the last workgroup left empty,
both products, a batch and SLICES, against the oracle under the bar of every
MATVEC test (1e-5 relative L2)."""
import numpy as np
import pytest

from ddscat_hip import BACKEND_FFT3D, BACKEND_SLICES
from oracle import ddscat_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims", [(5, 280, 1), (12, 294, 2), (3, 400, 3), (25, 1, 1), (24, 2, 5), (9, 7, 7), (30, 10, 12),
                                  (7, 9, 15), (8, 5, 16), (6, 6, 18), (5, 280, 20), (4, 8, 35), (2, 1024, 3)])
def test_against_oracle(lib, dims):
    import torch
    nx, ny, nz = dims
    rng = np.random.default_rng(nx * 10007 + ny * 101 + nz)
    nat = nx * ny * nz
    iocc = (rng.random(nat) < 0.8).astype(np.int16)
    iocc[0] = 1
    cx = lambda s: (s * (rng.normal(size=3 * nat) + 1j * rng.normal(size=3 * nat)) * np.tile(iocc != 0, 3)).astype(np.complex64)
    x, adia, aoff = cx(1.0), cx(1.0), cx(0.3)
    akd = 0.29
    goct = O.green_octant(nx, ny, nz, np.float64(np.float32(akd)))
    rel = lambda a, b: float(np.linalg.norm(a - b) / np.linalg.norm(b))
    occ = np.flatnonzero(iocc)
    comp = lambda v: np.ascontiguousarray(v.reshape(3, -1)[:, occ].reshape(-1))
    dev = lambda a: torch.from_numpy(a.view(np.float32)).cuda()
    try:
        for backend in (BACKEND_FFT3D, BACKEND_SLICES):
            lib.set_backend(backend)
            lib.prepare_green(nx, ny, nz, iocc, (akd, 0.0, 0.0))
            assert lib.info()["kernel_pass2"] == -1
            for cw in ("N", "C"):
                y = lib.apply(cw, x, adia, aoff)
                assert rel(y, O.matvec_fft(cw, x, adia, aoff, goct, nx, ny, nz, iocc)) < 1e-5
            y = comp(lib.apply("N", x, adia, aoff))
            xb = dev(np.concatenate([comp(x), comp(-x)]))
            ab, ob = (dev(np.tile(comp(v), 2)) for v in (adia, aoff))
            yb = torch.empty_like(xb)
            torch.cuda.synchronize()
            lib.apply_batch("N", 2, xb.data_ptr(), yb.data_ptr(), ab.data_ptr(), ob.data_ptr())
            lib.sync()
            yb = yb.cpu().numpy().view(np.complex64).reshape(2, -1)
            assert np.array_equal(yb[0], y) and np.array_equal(yb[1], -y)
    finally:
        lib.release()
        lib.set_backend(BACKEND_FFT3D)
