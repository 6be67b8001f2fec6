"""Far-field sums on the matrix cores at the edges of their tiles: rows of odd
and even length below and above one stage of 64 site pairs, row counts that
leave a group of 8 or a chunk of 32 unfilled, rows with holes, empty rows, and
direction counts around the 16 of a wave and the 128 of a workgroup, against
the FP64 oracle on the same polarizations.

Tolerances: the sums are FP64, so the Mueller elements carry only the rounding
of the phases, 4 x 2.2e-16 x |k.r| (|k.r| < 200 here), grown by at most ten
through cancellation and doubled by the product: 1e-11 of the largest element.
The amplitudes are rounded to complex64: 2e-7."""
import numpy as np
import pytest

from oracle import ddscat_oracle as O
from oracle import scattering as SC

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims,ndir,shape", [
    ((2, 3, 1), 1, "block"), ((3, 5, 7), 15, "holes"), ((9, 4, 10), 16, "sphere"), ((12, 35, 2), 17, "holes"),
    ((25, 8, 8), 128, "block"), ((20, 7, 15), 129, "sphere"), ((128, 6, 5), 33, "holes"),
    ((135, 5, 9), 40, "sphere"), ((135, 5, 9), 40, "holes"), ((160, 3, 4), 300, "block"), ((270, 4, 3), 20, "holes")])
def test_farfield_tiles_match_oracle(lib, dims, ndir, shape):
    import torch
    nx, ny, nz = dims
    rng = np.random.default_rng(nx + 7 * ny + ndir)
    z, y, x = np.meshgrid(*(np.linspace(-1, 1, n) if n > 1 else np.zeros(1) for n in (nz, ny, nx)), indexing="ij")
    iocc = {"block": np.ones(nx * ny * nz, bool), "holes": rng.random(nx * ny * nz) < 0.4,
            "sphere": (x * x + y * y + z * z <= 1.0).reshape(-1)}[shape].astype(np.int16)
    iocc[nx // 2] = 1
    occ = np.flatnonzero(iocc)
    kd = 0.25
    lib.prepare_green(nx, ny, nz, iocc, (kd, 0.0, 0.0))
    P = (rng.normal(size=(2, 3 * occ.size)) + 1j * rng.normal(size=(2, 3 * occ.size))).astype(np.complex64)
    f32 = lambda a: np.asarray(a, np.float32)
    ks = f32(kd * (lambda v: v / np.linalg.norm(v, axis=1, keepdims=True))(rng.normal(size=(ndir, 3))))
    em1, em2 = f32(rng.normal(size=(ndir, 3))), f32(rng.normal(size=(ndir, 3)))
    x0 = f32([-0.5 * (nx + 1), -3.25, 0.4])
    k, e1, e2 = np.array([1.0, 0, 0]), np.array([0, 1, 0], complex), np.array([0, 0, 1], complex)
    Pd = torch.from_numpy(P).cuda()
    torch.cuda.synchronize()
    f, M = lib.scat_matrix(Pd.data_ptr(), 1, [kd * k], [[e1, e2]], [ks], [em1], [em2], x0)
    S = [O.farfield_sums(P[j], occ, nx, ny, (1, 1, 1), np.float64(x0), ks) for j in range(2)]
    fr = [SC.amplitudes(S[j], kd * k, np.float64(em1), np.float64(em2)) for j in range(2)]
    fref = np.stack([fr[0][0], fr[0][1], fr[1][0], fr[1][1]], axis=1)
    Mref = SC.mueller(*SC.amplitude_matrix(*fref.T, e1, e2, k, np.float64(em2)))
    ferr = np.max(np.abs(f[0] - fref)) / np.max(np.abs(fref))
    merr = np.max(np.abs(M[0] - Mref)) / np.max(np.abs(Mref))
    print(f"{dims} {shape} {ndir}: amplitudes {ferr:.2e}, Mueller {merr:.2e}")
    assert ferr < 2e-7 and merr < 1e-11
    lib.release()
