"""The plane kernel (y, z, Green and inverse transforms of a kx plane in LDS)
at every padded y length and every padded z length it has, on planes as unlike
as they fit, with both products and a batch of right-hand sides, against the
oracle under the bar of every MATVEC test (1e-5 relative L2); the whole-grid
Green tensor of a periodic target and planes just too large go to other tests.
The kernel is checked to be the one that runs: selecting a kernel for pass 2
returns to the separate passes, and both agree within the rounding of FP32
transforms (5e-7)."""
import numpy as np
import pytest

from oracle import ddscat_oracle as O

pytestmark = pytest.mark.gpu

LENGTHS = [12, 14, 15, 16, 18, 20, 21, 24, 25, 27, 28, 30, 32, 35, 36, 40, 42, 45, 48, 49, 50, 54]


def check(lib, dims, nrhs=3):
    import torch
    nx, ny, nz = dims
    rng = np.random.default_rng(nx * 10000 + ny * 100 + nz)
    nat = nx * ny * nz
    iocc = (rng.random(nat) < 0.7).astype(np.int16)
    iocc[0] = 1
    cx = lambda s: (s * (rng.normal(size=3 * nat) + 1j * rng.normal(size=3 * nat)) * np.tile(iocc != 0, 3)).astype(np.complex64)
    x, adia, aoff = cx(1.0), cx(1.0), cx(0.3)
    akd = 0.31
    lib.prepare_green(nx, ny, nz, iocc, (akd, 0.0, 0.0))
    goct = O.green_octant(nx, ny, nz, np.float64(np.float32(akd)))
    rel = lambda a, b: float(np.linalg.norm(a - b) / np.linalg.norm(b))
    for cw in ("N", "C"):
        y = lib.apply(cw, x, adia, aoff)
        assert rel(y, O.matvec_fft(cw, x, adia, aoff, goct, nx, ny, nz, iocc)) < 1e-5, (dims, cw)
    occ = np.flatnonzero(iocc)
    comp = lambda v: np.ascontiguousarray(v.reshape(3, -1)[:, occ].reshape(-1))
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a).view(np.float32)).cuda()
    xb = dev(np.concatenate([comp(x) * np.complex64(1j ** r) for r in range(nrhs)]))
    yb = torch.empty_like(xb)
    ab, ob = (dev(np.tile(comp(v), nrhs)) for v in (adia, aoff))
    torch.cuda.synchronize()
    lib.apply_batch("N", nrhs, xb.data_ptr(), yb.data_ptr(), ab.data_ptr(), ob.data_ptr())
    lib.sync()
    yb = yb.cpu().numpy().view(np.complex64).reshape(nrhs, -1)
    yn = comp(lib.apply("N", x, adia, aoff))
    for r in range(nrhs):
        assert rel(yb[r], yn * np.complex64(1j ** r)) < 5e-7, (dims, r)
    assert np.array_equal(yb[0], yn)
    lib.set_pass_kernel(2, lib.info()["kernel_pass2"])
    ys = lib.apply("N", x, adia, aoff)
    err = rel(comp(ys), yn)
    assert 0 < err < 5e-7, (dims, err)


@pytest.mark.parametrize("n", LENGTHS)
def test_y_lengths(lib, n):
    check(lib, (5 if n <= 36 else 48, n, 12 if n % 2 else 15))


@pytest.mark.parametrize("n", LENGTHS)
def test_z_lengths(lib, n):
    check(lib, (6, 12 if n % 2 else 15, n))


@pytest.mark.parametrize("dims", [(7, 12, 54), (9, 54, 12), (4, 36, 36), (16, 45, 45), (48, 54, 54), (50, 48, 54)])
def test_plane_sizes(lib, dims):
    check(lib, dims)
