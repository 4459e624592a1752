"""What a unitary transform adds to the energy of its input, which a recursion of depth steps
raises to the power of its transforms."""
import pytest

pytestmark = pytest.mark.gpu


def test_1024_point_transforms_keep_the_energy(dev):
    """Random planes through the 2-D transform and back at 1024^2, where the
    scales are exact: the gain of the rounded twiddles and constants, computed in
    float64, is -1.0e-8 (columns) and -2.5e-8 (rows) per transform, -7.0e-8 over
    the four, and was -2.35e-7; bounded by half of that."""
    import torch
    from pyfwix_amd.ops import FFT2d, make_dims
    n, nw = 1024, 4
    op = FFT2d(make_dims(n, n, nw, 1, n, n, 0.0, 10.0, 0.0, 10.0, 5.0, 1.0, 0.0, 10.0, 1))
    g = torch.Generator(device=dev)
    g.manual_seed(3)
    x = torch.view_as_complex(torch.randn((1, nw, n, n, 2), generator=g, device=dev))
    f, b = torch.empty_like(x), torch.empty_like(x)
    op.forward(False, x, f)
    op.adjoint(False, b, f)
    e = [float(torch.view_as_real(t).double().square().sum()) for t in (x, b)]
    assert abs(e[1] / e[0] - 1) < 1.2e-7
