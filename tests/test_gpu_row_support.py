"""Compact MATVECs that leave the rows outside the target's y range alone in the
FFT work arrays (targets whose x spectra pass 256 MiB) against full-lattice
MATVECs, which transform every row with the same kernels: equal values at every
occupied site.  A full-lattice product of NaNs comes first, so that a read of an
unwritten row would show.  Grids: y lengths of 512 and 768 points, z pitches of whole and of half lines, empty z runs, a union whose rows
are no intervals, and the slabs of SLICES."""
import numpy as np
import pytest

from ddscat_hip import BACKEND_FFT3D, BACKEND_SLICES

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims,backend,rows", [((80, 384, 192), BACKEND_FFT3D, "interval"),
                                               ((128, 256, 200), BACKEND_FFT3D, "holes"),
                                               ((250, 256, 100), BACKEND_FFT3D, "interval"),
                                               ((96, 256, 256), BACKEND_SLICES, "holes")])
def test_support_equals_whole_lattice(lib, dims, backend, rows):
    import torch
    nx, ny, nz = dims
    z, y, x = np.meshgrid(np.arange(nz), np.arange(ny), np.arange(nx), indexing="ij")
    occ = (((x - nx / 2) / (0.5 * nx)) ** 2 + ((y - 0.45 * ny) / (0.4 * ny)) ** 2 + ((z - 0.4 * nz) / (0.3 * nz)) ** 2) < 1
    if rows == "holes":
        occ &= (x + y) % 7 != 0
    iocc = occ.astype(np.int16).reshape(-1)
    sites = torch.from_numpy(np.flatnonzero(iocc)).cuda()
    n0 = int(iocc.sum())
    gen = torch.Generator(device="cuda").manual_seed(nx)
    full = [torch.zeros((3, nx * ny * nz), dtype=torch.complex64, device="cuda") for _ in range(3)]
    comp = [s * torch.randn((3, n0), dtype=torch.complex64, generator=gen, device="cuda") for s in (1.0, 1.0, 0.3)]
    for f, c in zip(full, comp):
        f[:, sites] = c
    try:
        lib.set_backend(backend)
        lib.prepare_green(nx, ny, nz, iocc, (0.2, 0.0, 0.0))

        def apply(cw, layout, v):
            out = torch.zeros_like(v[0])
            torch.cuda.synchronize()
            lib.apply_device(cw, v[0].data_ptr(), out.data_ptr(), v[1].data_ptr(), v[2].data_ptr(), layout=layout)
            lib.sync()
            return out

        nan = torch.full_like(full[0], float("nan"))
        for cw in ("N", "C"):
            apply(cw, 0, [nan, full[1], full[2]])
            got = apply(cw, 1, comp)
            want = apply(cw, 0, full)[:, sites]
            assert torch.isfinite(torch.view_as_real(got)).all()
            assert torch.equal(got, want)
    finally:
        lib.release()
        lib.set_backend(BACKEND_FFT3D)
