"""SLICES over several slabs of kx planes (grids above one slab, with a last
slab of fewer planes) against FFT3D, on compact and full vectors, both
products, the register and the LDS-staged kernels and the whole-grid Green
tensor of a periodic target.  Both back ends run the same kernels on the same
values, plane by plane, so the products are equal bit for bit."""
import numpy as np
import pytest

from ddscat_hip import BACKEND_FFT3D, BACKEND_SLICES

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims,generic,ipbc", [((75, 100, 96), 0, 0), ((75, 100, 96), 1, 0), ((84, 90, 98), 0, 0),
                                               ((64, 128, 96), 0, 1), ((162, 180, 160), 0, 0), ((180, 162, 180), 0, 0)])
def test_slabs_equal_fft3d(lib, dims, generic, ipbc):
    import torch
    nx, ny, nz = dims
    rng = np.random.default_rng(nx)
    nat = nx * ny * nz
    iocc = (rng.random(nat) < 0.6).astype(np.int16)
    iocc[0] = 1
    n0 = int(iocc.sum())
    dev = lambda n, s: torch.from_numpy((s * rng.normal(size=2 * n)).astype(np.float32)).cuda()
    ops = {1: [dev(3 * n0, s) for s in (1.0, 1.0, 0.3)],
           0: [dev(3 * nat, s) for s in (1.0, 1.0, 0.3)] if not generic else None}
    out = {}
    try:
        lib.set_fft_kernels(generic)
        for backend in (BACKEND_FFT3D, BACKEND_SLICES):
            lib.release()
            lib.set_backend(backend)
            kw = dict(ipbc=1, gamma=0.05, pyd=float(ny), pzd=float(nz)) if ipbc else {}
            lib.prepare_green(nx, ny, nz, iocc, (0.2, 0.0, 0.0), **kw)
            for layout, v in ops.items():
                for cw in ("N", "C") if v else ():
                    y = torch.zeros_like(v[0])
                    torch.cuda.synchronize()
                    lib.apply_device(cw, v[0].data_ptr(), y.data_ptr(), v[1].data_ptr(), v[2].data_ptr(),
                                     layout=layout)
                    lib.sync()
                    out[backend, layout, cw] = y
        for (b, layout, cw), y in out.items():
            if b == BACKEND_SLICES:
                assert torch.isfinite(y).all() and float(y.abs().max()) > 0
                assert torch.equal(y, out[BACKEND_FFT3D, layout, cw]), (layout, cw)
    finally:
        lib.release()
        lib.set_backend(BACKEND_FFT3D)
        lib.set_fft_kernels(0)
