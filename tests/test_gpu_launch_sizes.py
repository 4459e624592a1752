"""How many planes a step's launches hold: as the caller says, or chosen, with
the same results."""
import numpy as np
import pytest

from fwix_testutil import crand, dims_of, grid

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
