"""The LDS-staged x passes: x axes without a register kernel, from a single site
(2 points) to the longest (2,048), with row counts that leave the last workgroup
part-filled and tiles that cross z runs, targets whose rows are no intervals,
both products, both layouts and a batch, against the oracle under the bar of
every MATVEC test (1e-5 relative L2).  A workgroup's rows give every thread an
element, and at axes of 560 to 800 points as many rows as half the LDS holds,
where the target has rows for 512 workgroups of them."""
import numpy as np
import pytest

from ddscat_hip import BACKEND_FFT3D, BACKEND_SLICES
from oracle import ddscat_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims", [(1, 6, 5), (1, 40, 36), (2, 18, 16), (3, 15, 12), (4, 9, 60), (5, 10, 9), (6, 15, 14),
                                  (7, 7, 7), (8, 16, 18), (9, 30, 27), (10, 10, 10), (280, 5, 4), (294, 4, 3), (400, 3, 20),
                                  (675, 5, 3), (1024, 2, 3)])
@pytest.mark.parametrize("holes", [False, True])
def test_against_oracle(lib, dims, holes):
    import torch
    nx, ny, nz = dims
    rng = np.random.default_rng(nx * 10007 + ny * 101 + nz)
    nat = nx * ny * nz
    iocc = (rng.random(nat) < 0.8).astype(np.int16) if holes else np.ones(nat, np.int16)
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
            assert lib.info()["kernel_pass1"] == -1
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


@pytest.mark.parametrize("dims,rows", [((2, 128, 128), 64), ((8, 60, 60), 16), ((280, 64, 64), 7), ((400, 64, 64), 5)])
def test_rows_per_workgroup(lib, dims, rows):
    lib.prepare_green(*dims, np.ones(dims[0] * dims[1] * dims[2], np.int16), (0.2, 0.0, 0.0))
    assert lib.info()["rx_fwd"] >= rows and lib.info()["rx_inv"] >= rows
