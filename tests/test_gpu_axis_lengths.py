"""FFT3D MATVEC at every padded axis length with a register kernel of its own
(2N for N = 2^a 3^b 5^c from 12 to 256, and the lengths above), on each axis in
turn, against the oracle: tiles whose columns or rows end inside a workgroup,
z runs with and without padding, plans whose stages leave lanes idle.
Tolerance: 1e-5 relative L2, the bar of every MATVEC test (FP32 transforms of
up to 768 points round at a few 1e-7)."""
import numpy as np
import pytest

from oracle import ddscat_oracle as O

pytestmark = pytest.mark.gpu

SMOOTH = [n for n in range(12, 257) if all(f in (2, 3, 5) for f in
                                           [p for p in range(2, n + 1) if n % p == 0 and all(p % q for q in range(2, p))])]
LONG = [270, 288, 300, 320, 324, 360, 375, 384]


@pytest.mark.parametrize("axis", [0, 1, 2])
@pytest.mark.parametrize("n", SMOOTH + LONG)
def test_axis_length_matches_oracle(lib, n, axis):
    dims = [(n, 5, 7), (6, n, 5), (7, 6, n)][axis]
    nx, ny, nz = dims
    rng = np.random.default_rng(1000 * axis + n)
    nat = nx * ny * nz
    iocc = (rng.random(nat) < 0.7).astype(np.int16)
    iocc[0] = 1
    cx = lambda s: (s * (rng.normal(size=3 * nat) + 1j * rng.normal(size=3 * nat)) * np.tile(iocc != 0, 3)).astype(np.complex64)
    x, adia, aoff = cx(1.0), cx(1.0), cx(0.3)
    akd = 0.31
    lib.prepare_green(nx, ny, nz, iocc, (akd, 0.0, 0.0))
    info = lib.info()
    passes = [(1, 5), (2, 4), (3,)][axis]
    assert all(info[f"kernel_pass{p}"] >= 0 for p in passes)  # a register kernel, not the LDS-staged one
    goct = O.green_octant(nx, ny, nz, np.float64(np.float32(akd)))
    y = lib.apply("N", x, adia, aoff)
    yref = O.matvec_fft("N", x, adia, aoff, goct, nx, ny, nz, iocc)
    err = float(np.linalg.norm(y - yref) / np.linalg.norm(yref))
    assert err < 1e-5, (dims, err)
