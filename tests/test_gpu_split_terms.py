"""Launches of few waves, which share a step's references out over workgroups,
thread groups or waves, against float64: a narrow plane on its own at column
lengths of every kind of split fan-in, every reference in some row and most
absent from others, with the presence masks (5 references) and without (40)."""
import numpy as np
import pytest

import oracle as O
from fwix_testutil import TOL_WFLD, crand, dims_of, grid, rel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny", [(16, 12), (96, 64), (128, 192), (256, 256), (48, 384), (48, 512), (256, 512),
                                   (48, 768), (24, 768), (48, 1024)])
@pytest.mark.parametrize("nref", [5, 40])
def test_one_plane_matches_oracle(dev, nx, ny, nref):
    import torch
    from pyfwix_amd.ops import FWIX_NSPS, FWIX_PSPI, OneStep
    rng = np.random.default_rng(nx + ny + nref)
    g = grid(nx, ny, 1, 1, nz=1)
    sref = (1.0 / rng.uniform(1500, 3000, (1, nref, 1)) ** 2).astype(np.complex64)
    lab = rng.integers(0, nref, (1, 1, ny, nx)).astype(np.uint8)
    lab[0, 0, : ny // 3] = nref - 1
    lab[0, 0, ny // 3: ny // 2, : nx // 2] = 1
    x, y = crand(rng, (1, 1, ny, nx)), crand(rng, (1, 1, ny, nx))
    s64, l64 = sref[0].astype(np.complex128), lab[0].astype(np.int64)
    t = lambda a: torch.from_numpy(a.astype(np.complex64)).to(dev)  # noqa: E731
    for method in (FWIX_PSPI, FWIX_NSPS):
        op = OneStep(method, dims_of(g), nref=nref, taperx=2, tapery=3)
        op.set_refs(torch.from_numpy(sref).to(dev), torch.from_numpy(lab).to(dev))
        op.set_depth(0)
        f, a = t(0 * x), t(0 * y)
        op.forward(False, t(x), f)
        op.adjoint(False, a, t(y))
        if method == FWIX_PSPI:
            want = O.pspi_forward(x, s64, l64, g, g.dz, 0.0, 2, 3), O.pspi_adjoint(y, s64, l64, g, g.dz, 0.0, 2, 3)
        else:
            want = O.nsps_forward(x, s64, l64, g, g.dz, 0.0), O.nsps_adjoint(y, s64, l64, g, g.dz, 0.0)
        assert rel(f.cpu().numpy(), want[0]) < TOL_WFLD, method
        assert rel(a.cpu().numpy(), want[1]) < TOL_WFLD, method


@pytest.mark.parametrize("nx,ny", [(16, 12), (128, 96), (192, 192), (256, 256), (48, 512), (48, 1024)])
@pytest.mark.parametrize("present", [1, 2, 3, 5])
def test_split_by_references_present(dev, nx, ny, present):
    """Six references of which the first plane holds one and the second `present`
    (not the lowest numbers): parts of a launch with no term of a plane, and
    planes of a launch with more terms than others."""
    import torch
    from pyfwix_amd.ops import FWIX_NSPS, FWIX_PSPI, OneStep
    rng = np.random.default_rng(nx + ny + present)
    g = grid(nx, ny, 2, 1, nz=1)
    sref = (1.0 / rng.uniform(1500, 3000, (1, 6, 2)) ** 2).astype(np.complex64)
    lab = np.full((1, 2, ny, nx), 4, np.uint8)
    lab[0, 1] = rng.permutation(6)[:present][rng.integers(0, present, (ny, nx))]
    x, y = crand(rng, (1, 2, ny, nx)), crand(rng, (1, 2, ny, nx))
    s64, l64 = sref[0].astype(np.complex128), lab[0].astype(np.int64)
    t = lambda a: torch.from_numpy(a.astype(np.complex64)).to(dev)  # noqa: E731
    for method in (FWIX_PSPI, FWIX_NSPS):
        op = OneStep(method, dims_of(g), nref=6, taperx=2, tapery=3)
        op.set_refs(torch.from_numpy(sref).to(dev), torch.from_numpy(lab).to(dev))
        op.set_depth(0)
        f, a = t(0 * x), t(0 * y)
        op.forward(False, t(x), f)
        op.adjoint(False, a, t(y))
        if method == FWIX_PSPI:
            want = O.pspi_forward(x, s64, l64, g, g.dz, 0.0, 2, 3), O.pspi_adjoint(y, s64, l64, g, g.dz, 0.0, 2, 3)
        else:
            want = O.nsps_forward(x, s64, l64, g, g.dz, 0.0), O.nsps_adjoint(y, s64, l64, g, g.dz, 0.0)
        assert rel(f.cpu().numpy(), want[0]) < TOL_WFLD, method
        assert rel(a.cpu().numpy(), want[1]) < TOL_WFLD, method
