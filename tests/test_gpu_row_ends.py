"""Row passes whose last workgroup has waves without rows: grids of few rows,
with the output and the input at the front of larger tensors."""
import numpy as np
import pytest

import oracle as O
from fwix_testutil import TOL_WFLD, crand, dims_of, grid, rel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("quad", [0, 1])
@pytest.mark.parametrize("nx,ny,nw", [(8, 8, 1), (12, 24, 3), (16, 12, 1), (64, 24, 1), (128, 8, 1), (384, 12, 1)])
def test_waves_without_rows_touch_nothing(dev, nx, ny, nw, quad):
    import torch
    from pyfwix_amd import _lib
    from pyfwix_amd.ops import FWIX_NSPS, FWIX_PSPI, FFT2d, OneStep, Scatter
    rng = np.random.default_rng(nx + ny)
    g = grid(nx, ny, nw, 1, nz=1)
    shape, n, mark = (1, nw, ny, nx), nw * ny * nx, 7.0 - 3.0j

    def front(a=None):
        """A tensor of the wavefield's shape at the front of one with 64 k marked elements behind it."""
        big = torch.full((n + 65536,), mark, dtype=torch.complex64, device=dev)
        big[:n] = 0 if a is None else torch.from_numpy(a.astype(np.complex64).ravel()).to(dev)
        return big, big[:n].view(shape)

    sref = (1.0 / rng.uniform(1500, 3000, (1, 3, nw)) ** 2).astype(np.complex64)
    lab = rng.integers(0, 3, (1, nw, ny, nx)).astype(np.uint8)
    slow = np.full((1, nw, ny, nx), 1 / 2000.0 ** 2, np.complex64)
    x, y = crand(rng, shape), crand(rng, shape)
    s64, l64 = sref[0].astype(np.complex128), lab[0].astype(np.int64)
    before = _lib.lib.fwix_tune_scratch_layout_get(ny)
    try:
        _lib.call("fwix_tune_scratch_layout_set", ny, quad)
        for what in ("fft", FWIX_PSPI, FWIX_NSPS, "scatter"):
            if what == "fft":
                op = FFT2d(dims_of(g))
                want = np.fft.fft2(x, norm="ortho"), np.fft.ifft2(y, norm="ortho")
            elif what == "scatter":
                op = Scatter(dims_of(g), taylor=1, eps_scat=0.04)
                op.set_slow(torch.from_numpy(slow).to(dev))
                op.set_depth(0)
                s = slow[0].astype(np.complex128)
                want = O.scatter_forward(x, s, g, g.dz, 0.04, 1), O.scatter_adjoint(y, s, g, g.dz, 0.04, 1)
            else:
                op = OneStep(what, dims_of(g), nref=3, taperx=2, tapery=2)
                op.set_refs(torch.from_numpy(sref).to(dev), torch.from_numpy(lab).to(dev))
                op.set_depth(0)
                if what == FWIX_PSPI:
                    want = O.pspi_forward(x, s64, l64, g, g.dz, 0.0, 2, 2), O.pspi_adjoint(y, s64, l64, g, g.dz, 0.0, 2, 2)
                else:
                    want = O.nsps_forward(x, s64, l64, g, g.dz, 0.0), O.nsps_adjoint(y, s64, l64, g, g.dz, 0.0)
            for add in (False, True):
                (bm, m), (bf, f), (bd, d), (ba, a) = front(x), front(), front(y), front()
                op.forward(add, m, f)
                op.adjoint(add, a, d)
                torch.cuda.synchronize()
                for b in (bm, bf, bd, ba):
                    assert torch.all(b[n:] == mark), (what, add)
                assert rel(f.cpu().numpy(), want[0]) < TOL_WFLD, (what, add)
                assert rel(a.cpu().numpy(), want[1]) < TOL_WFLD, (what, add)
    finally:
        _lib.call("fwix_tune_scratch_layout_set", ny, before)
