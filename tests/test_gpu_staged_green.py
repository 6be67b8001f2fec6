"""The LDS-staged Green pass: z axes without a register kernel, from a single
plane (2 points) to the longest (2,048), with column counts that leave the last
workgroup part-filled and tiles that cross kx planes, both products, a batch, a
periodic target's whole-grid Green tensor and SLICES, against the oracle under
the bar of every MATVEC test (1e-5 relative L2).  A workgroup has 256 threads:
its columns give every one of them an element."""
import numpy as np
import pytest

from ddscat_hip import BACKEND_FFT3D, BACKEND_SLICES
from oracle import ddscat_oracle as O

pytestmark = pytest.mark.gpu


def case(dims):
    nx, ny, nz = dims
    rng = np.random.default_rng(nx * 10007 + ny * 101 + nz)
    nat = nx * ny * nz
    iocc = (rng.random(nat) < 0.8).astype(np.int16)
    iocc[0] = 1
    cx = lambda s: (s * (rng.normal(size=3 * nat) + 1j * rng.normal(size=3 * nat)) * np.tile(iocc != 0, 3)).astype(np.complex64)
    return iocc, cx(1.0), cx(1.0), cx(0.3)


def rel(a, b):
    return float(np.linalg.norm(a - b) / np.linalg.norm(b))


@pytest.mark.parametrize("backend", [BACKEND_FFT3D, BACKEND_SLICES])
@pytest.mark.parametrize("dims", [(5, 6, 1), (40, 36, 1), (16, 18, 2), (45, 30, 2), (12, 15, 3), (21, 20, 4),
                                  (9, 10, 5), (14, 15, 6), (7, 9, 7), (18, 16, 8), (30, 27, 9), (24, 20, 10),
                                  (5, 4, 294), (7, 6, 400), (3, 5, 675), (2, 3, 1024)])
def test_against_oracle(lib, dims, backend):
    nx, ny, nz = dims
    iocc, x, adia, aoff = case(dims)
    akd = 0.29
    try:
        lib.set_backend(backend)
        lib.prepare_green(nx, ny, nz, iocc, (akd, 0.0, 0.0))
        info = lib.info()
        assert info["kernel_pass3"] == -1
        assert info["cz"] * info["gz"] >= 256
        goct = O.green_octant(nx, ny, nz, np.float64(np.float32(akd)))
        for cw in ("N", "C"):
            assert rel(lib.apply(cw, x, adia, aoff), O.matvec_fft(cw, x, adia, aoff, goct, nx, ny, nz, iocc)) < 1e-5
    finally:
        lib.release()
        lib.set_backend(BACKEND_FFT3D)


@pytest.mark.parametrize("dims", [(36, 40, 1), (15, 16, 3), (20, 18, 10), (5, 6, 280)])
def test_batch_equals_single(lib, dims):
    import torch
    iocc, x, adia, aoff = case(dims)
    lib.prepare_green(*dims, iocc, (0.29, 0.0, 0.0))
    occ = np.flatnonzero(iocc)
    comp = lambda v: np.ascontiguousarray(v.reshape(3, -1)[:, occ].reshape(-1))
    dev = lambda a: torch.from_numpy(a.view(np.float32)).cuda()
    xb = dev(np.concatenate([comp(x), comp(x.conj()), comp(1j * x).astype(np.complex64)]))
    ab, ob = (dev(np.tile(comp(v), 3)) for v in (adia, aoff))
    yb = torch.empty_like(xb)
    torch.cuda.synchronize()
    lib.apply_batch("N", 3, xb.data_ptr(), yb.data_ptr(), ab.data_ptr(), ob.data_ptr())
    lib.sync()
    yb = yb.cpu().numpy().view(np.complex64).reshape(3, -1)
    for r, v in enumerate((x, x.conj(), (1j * x).astype(np.complex64))):
        assert np.array_equal(yb[r], comp(lib.apply("N", v, adia, aoff)))


@pytest.mark.parametrize("dims", [(6, 5, 1), (20, 18, 2), (9, 8, 10)])
def test_whole_grid_green(lib, dims):
    nx, ny, nz = dims
    iocc, x, adia, aoff = case(dims)
    ak, pyd, pzd, gamma = (0.4, 0.1, 0.0), float(ny), float(nz) + 3.0, 0.3
    lib.prepare_green(nx, ny, nz, iocc, ak, ipbc=1, gamma=gamma, pyd=pyd, pzd=pzd)
    g = lib.get_green().reshape(6, 2 * nz, 2 * ny, 2 * nx)
    y = lib.apply("N", x, adia, aoff)
    yref = O.matvec_fft("N", x, adia, aoff, g.astype(np.complex128), nx, ny, nz, iocc, ipbc=1)
    assert rel(y, yref) < 1e-5
