"""How many planes a step's launches hold: as the caller says, or chosen, with
the same results."""
import numpy as np
import pytest

from fwix_testutil import crand, dims_of, grid, rel

pytestmark = pytest.mark.gpu


def _launches(run):
    """Launches of every timed pass in run()."""
    import torch
    from pyfwix_amd import _lib
    torch.cuda.synchronize()
    _lib.timing_reset()
    _lib.timing_select(None, 1)
    _lib.timing_enable(256)
    try:
        run()
        torch.cuda.synchronize()
    finally:
        _lib.timing_disable()
        p = _lib.timing_collect()
        _lib.timing_reset()
    return {k: v["total_launches"] for k, v in p.items()}


def _steps(dev, n, nw, nref, chunk, method, seed=5):
    """A step with every reference in every row, its input and the operator."""
    import torch
    from pyfwix_amd.ops import OneStep
    rng = np.random.default_rng(seed)
    sref = (1.0 / rng.uniform(1500, 3000, (1, nref, 1)) ** 2).astype(np.complex64)
    sref = torch.from_numpy(sref).to(dev).expand(1, nref, nw).contiguous()
    lab = torch.from_numpy(rng.integers(0, nref, (1, 1, n, n)).astype(np.uint8)).to(dev).expand(1, nw, n, n).contiguous()
    op = OneStep(method, dims_of(grid(n, n, nw, 1, nz=1, dw=0.5)), nref=nref, taperx=4, tapery=4, planes_per_chunk=chunk)
    op.set_refs(sref, lab)
    op.set_depth(0)
    x = torch.from_numpy(crand(rng, (1, 1, n, n)).astype(np.complex64)).to(dev).expand(1, nw, n, n).contiguous()
    return op, x


@pytest.mark.parametrize("n,nw,nref", [(512, 24, 10), (768, 12, 8), (1024, 8, 6)])
def test_given_planes_per_launch_are_taken(dev, n, nw, nref):
    """planes_per_chunk is taken as given however many references the rows hold,
    and the step is the same, bit for bit, as with launches of the automatic size."""
    import torch
    from pyfwix_amd.ops import FWIX_NSPS, FWIX_PSPI
    for method in (FWIX_PSPI, FWIX_NSPS):
        outs = []
        for chunk in (0, nw, 5):
            op, x = _steps(dev, n, nw, nref, chunk, method)
            f, a = torch.zeros_like(x), torch.zeros_like(x)

            def run():
                op.forward(False, x, f)
                op.adjoint(False, a, x)
            got = _launches(run)
            if chunk:
                want = -(-nw // chunk)
                assert got["cols_fanout"] == got["cols_fanin"] == want, got
                assert got["rows_select"] == got["rows_fanout"] == want, got
            outs.append((f, a))
        for f, a in outs[1:]:
            assert torch.equal(f, outs[0][0]) and torch.equal(a, outs[0][1])


@pytest.mark.parametrize("n,nw,nref,want", [(256, 96, 12, 3), (512, 24, 2, 1), (512, 24, 4, 1), (512, 24, 8, 2),
                                            (512, 24, 12, 3), (768, 16, 8, 4), (1024, 8, 4, 1), (1024, 8, 8, 3),
                                            (1024, 8, 12, 4)])
def test_automatic_launches_fit_the_cache(dev, n, nw, nref, want):
    """A launch whose K and W (every reference in every row) fit in 256 MiB and
    which fills the chip, with 1024-point columns only from 7 references on."""
    import torch
    from pyfwix_amd.ops import FWIX_PSPI
    op, x = _steps(dev, n, nw, nref, 0, FWIX_PSPI)
    y = torch.zeros_like(x)
    got = _launches(lambda: op.forward(False, x, y))
    assert got["cols_fanout"] == got["rows_select"] == want, got


@pytest.mark.parametrize("method", ["pspi", "nsps"])
def test_chained_recursion_with_launches_of_changing_size(dev, method):
    """Downward over depths of 10, 2, 7 and 4 references per row, so that the
    row spectra left by one depth's launches are read by the next in
    launches of another size: the unchained steps, and launches of all planes,
    to float rounding (1e-6)."""
    import torch
    from pyfwix_amd.ops import FWIX_NSPS, FWIX_PSPI, OneWay
    rng = np.random.default_rng(11)
    n, nw, nref, present = 512, 22, 10, (10, 2, 7, 4, 1)
    g = grid(n, n, nw, 1, nz=len(present), dw=0.5)
    sref = (1.0 / rng.uniform(1500, 3000, (g.nz, nref, 1)) ** 2).astype(np.complex64)
    sref = torch.from_numpy(sref).to(dev).expand(g.nz, nref, nw).contiguous()
    lab = np.stack([rng.integers(0, k, (1, n, n)) for k in present]).astype(np.uint8)
    lab = torch.from_numpy(lab).to(dev).expand(g.nz, nw, n, n).contiguous()
    x = torch.from_numpy(crand(rng, (1, nw, n, n)).astype(np.complex64)).to(dev)
    outs, launches = [], []
    for chunk, chain in ((0, True), (0, False), (nw, True)):
        op = OneWay(0, FWIX_PSPI if method == "pspi" else FWIX_NSPS, dims_of(g), nref=nref, taperx=4, tapery=4,
                    planes_per_chunk=chunk)
        op.set_refs(sref, lab)
        op.set_step_chaining(chain)
        f, a = torch.zeros_like(x), torch.zeros_like(x)

        def run():
            op.forward(False, x, f)
            op.adjoint(False, a, x)
        launches.append(_launches(run))
        outs.append((f.cpu().numpy(), a.cpu().numpy()))
        del op
    assert launches[0]["cols_fanout"] > launches[2]["cols_fanout"] + 2, launches
    for f, a in outs[1:]:
        assert rel(f, outs[0][0]) < 1e-6 and rel(a, outs[0][1]) < 1e-6
