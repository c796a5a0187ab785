"""Rounding error of the separate filter on smooth float32 rows whose result is
their high frequencies, at lengths of a run-time plan: multiples of large primes
(127, 101, 79) and of 5, 9 and 17.

Tolerance: a rounding at each of the log2(ne) levels of the transform, about 0.41
units (2^-24; 0.29 of a last place, whose size relative to the value is between
one and two units) of the row's rms, white over the frequencies, then times the
ramp: relative to the result 0.41 sqrt(log2 ne) 2^-24 G with G the ramp's gain
for white noise over its gain for the row.  Twiddles and constants add a few
tenths of that in quadrature: asserted at 0.55."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _ellipses(nz, nproj, ne, seed):
    rng = np.random.default_rng(seed)
    t = np.arange(ne) - ne / 2
    rows = np.zeros((nz, nproj, ne))
    for z in range(nz):
        for p in range(nproj):
            for _ in range(10):
                a, c = rng.uniform(0.05, 0.4) * ne / 2, rng.uniform(-0.5, 0.5) * ne / 2
                rows[z, p] += rng.uniform(0.1, 0.8) * np.sqrt(np.clip(1 - ((t - c) / a)**2, 0, None))
    return rows.astype(np.float32)


@pytest.mark.parametrize('ne', [1016, 2448, 4000, 8888, 9792, 12324])
def test_smooth_rows(ne):
    from tomocupy_amd.fbp_filter import FBPFilter
    nz, nproj = 2, 5
    rows = _ellipses(nz, nproj, ne, ne)
    ramp = np.arange(ne // 2 + 1) / ne
    ref = np.fft.irfft(np.fft.rfft(rows.astype(np.float64)) * ramp, n=ne)
    flt = FBPFilter(ne, nproj, nz, n_unpadded=ne // 4 * 2)
    d = torch.from_numpy(rows).cuda()
    w = torch.from_numpy(ramp.astype(np.complex64)).cuda().expand(nz, -1).contiguous()
    flt.filter(d, w)
    got = d.cpu().numpy().astype(np.float64) / ne  # (the inverse transform is unnormalised)
    err = np.linalg.norm(got - ref) / np.linalg.norm(ref)
    gain = np.linalg.norm(rows) * np.sqrt(1 / 12) / np.linalg.norm(ref)
    bound = 0.55 * np.sqrt(np.log2(ne)) * 2.0**-24 * gain
    print('ne=%d error %.3g bound %.3g' % (ne, err, bound))
    assert err <= bound
