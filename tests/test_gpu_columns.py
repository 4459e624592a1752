"""Column transforms at every supported length: the plain 2-D FFT, and the
fused steps, whose last tile of columns is partly beyond the grid (NX = 12,
rows of the presence masks with references absent), against float64."""
import numpy as np
import pytest

import oracle as O
from fwix_testutil import TOL_WFLD, crand, dims_of, grid, rel

pytestmark = pytest.mark.gpu

SIZES = (8, 12, 16, 24, 32, 48, 64, 96, 128, 192, 256, 384, 512, 768, 1024)


def _t(a, dev, dtype=np.complex64):
    import torch
    return torch.from_numpy(np.ascontiguousarray(a.astype(dtype))).to(dev)


@pytest.mark.parametrize("ny", SIZES)
def test_fft_of_every_column_length(dev, ny):
    """Rounding of a radix-16 or smaller plan: a few 2^-24 per stage (at most
    7 stages over both axes), so 1e-6 in the relative L2 norm."""
    import torch
    from pyfwix_amd.ops import FFT2d
    rng = np.random.default_rng(ny)
    g = grid(12, ny, 2, 1, nz=1)
    x = crand(rng, (1, 2, ny, 12)).astype(np.complex64)
    op = FFT2d(dims_of(g))
    f, b = torch.zeros_like(_t(x, dev)), _t(x, dev)
    op.forward(False, _t(x, dev), f)
    op.adjoint(True, b, _t(x, dev))  # added to x
    x64 = x.astype(np.complex128)
    assert rel(f.cpu().numpy(), np.fft.fft2(x64, norm="ortho")) < 1e-6
    assert rel(b.cpu().numpy(), x64 + np.fft.ifft2(x64, norm="ortho")) < 1e-6


@pytest.mark.parametrize("eps", [0.0, 0.02])
@pytest.mark.parametrize("ny", SIZES)
def test_steps_of_every_column_length(dev, ny, eps):
    import torch
    from pyfwix_amd.ops import FWIX_NSPS, FWIX_PSPI, OneStep
    rng = np.random.default_rng(100 + ny)
    nref, shape = 5, (1, 3, ny, 12)
    g = grid(12, ny, 3, 1, nz=1)
    sref = (1.0 / rng.uniform(1500, 3000, (1, nref, 3)) ** 2).astype(np.complex64)
    lab = np.zeros((1, 3, ny, 12), np.uint8)
    lab[0, 0] = rng.integers(0, nref, (ny, 12))       # every reference
    lab[0, 1, ny // 3:, 5:] = nref - 1                # two references, one in some rows only
    x, y = crand(rng, shape), crand(rng, shape)
    s64, l64 = sref[0].astype(np.complex128), lab[0].astype(np.int64)
    for method in (FWIX_PSPI, FWIX_NSPS):
        op = OneStep(method, dims_of(g), nref=nref, taperx=2, tapery=3, eps=eps)
        op.set_refs(_t(sref, dev), _t(lab, dev, np.uint8))
        op.set_depth(0)
        f, a = _t(0 * x, dev), _t(0 * y, dev)
        op.forward(False, _t(x, dev), f)
        op.adjoint(False, a, _t(y, dev))
        if method == FWIX_PSPI:
            rf, ra = O.pspi_forward(x, s64, l64, g, g.dz, eps, 2, 3), O.pspi_adjoint(y, s64, l64, g, g.dz, eps, 2, 3)
        else:
            rf, ra = O.nsps_forward(x, s64, l64, g, g.dz, eps), O.nsps_adjoint(y, s64, l64, g, g.dz, eps)
        torch.cuda.synchronize()
        assert rel(f.cpu().numpy(), rf) < TOL_WFLD, method
        assert rel(a.cpu().numpy(), ra) < TOL_WFLD, method


@pytest.mark.parametrize("ny", [24, 64, 96, 192, 256, 384, 512])
def test_float64_columns_of_every_kind(dev, ny):
    """The float64 scattering arithmetic (its own column plans) at the lengths
    that the large-grid tests leave out."""
    from pyfwix_amd.ops import FWIX_PREC_F64_SCATTER
    from test_gpu_born import _born_vs_oracle
    errs, _ = _born_vs_oracle(dev, (48, ny, 2, 40, ny - 8), 6.0, precision=FWIX_PREC_F64_SCATTER)
    assert max(errs) < TOL_WFLD, errs


@pytest.mark.parametrize("nx,ny", [(16, 12), (96, 64), (128, 192), (256, 256), (384, 384), (512, 768), (48, 1024)])
@pytest.mark.parametrize("masks", [True, False])
def test_small_launches_split_their_terms(dev, nx, ny, masks):
    """A plane on its own (few waves: its references shared out over
    workgroups, thread groups or waves) and among so many that nothing is split: the
    same step up to the order in which the references' spectra are added
    (2^-24 per addition; 1e-6 relative).  nref = 40 runs without presence masks."""
    import torch
    from pyfwix_amd.ops import FWIX_NSPS, FWIX_PSPI, OneStep
    rng = np.random.default_rng(nx + ny)
    nref = 5 if masks else 40
    many = max(2, min(400, (6 << 20) // (nx * ny)))
    sref = (1.0 / rng.uniform(1500, 3000, (1, nref, 1)) ** 2).astype(np.complex64)
    lab = rng.integers(0, nref, (1, 1, ny, nx)).astype(np.uint8)
    lab[0, 0, : ny // 2] = nref - 1
    x = crand(rng, (1, 1, ny, nx))
    for method in (FWIX_PSPI, FWIX_NSPS):
        out = []
        for nw in (1, many):
            op = OneStep(method, dims_of(grid(nx, ny, nw, 1, nz=1, dw=0.0)), nref=nref, taperx=2, tapery=3)
            op.set_refs(_t(np.repeat(sref, nw, 2), dev), _t(np.repeat(lab, nw, 1), dev, np.uint8))
            op.set_depth(0)
            u = _t(np.repeat(x, nw, 1), dev)
            f, a = torch.zeros_like(u), torch.zeros_like(u)
            op.forward(False, u, f)
            op.adjoint(False, a, u)
            out.append((f[0, -1].cpu().numpy(), a[0, -1].cpu().numpy()))
        assert rel(out[0][0], out[1][0]) < 1e-6 and rel(out[0][1], out[1][1]) < 1e-6, method
