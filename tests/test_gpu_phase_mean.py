"""Phase retrieval of a constant image: every sum of the transforms is exact (the
lengths are powers of two, the value has few digits), and the factor over its
maximum is 1 at zero frequency, so what is left is the rounding of the product
with 1 / (Ny Nx) in its few terms: at most a last place, 2^-23 of the value.  The
same at a regularisation so large that the factor is subnormal everywhere."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('alpha', [1e-4, 1e-3, 3e-3, 0.7, 1e38])
@pytest.mark.parametrize('dy,dz', [(20, 60), (128, 256), (300, 700), (1024, 1024)])
def test_constant_image(dy, dz, alpha):
    from tomocupy_amd.retrieve_phase import PhasePlan
    plan = PhasePlan(dy, dz, 'paganin', pixel_size=1e-4, dist=5.0, energy=20.0, alpha=alpha)
    d = torch.full((1, dy, dz), 0.75, device='cuda')
    plan.apply(d)
    err = float((d.double() / 0.75 - 1).abs().max())
    print((dy, dz), 'alpha %g error %.3g of 2^-23' % (alpha, err * 2.0**23))
    plan.free()
    assert err <= 2.0**-23
