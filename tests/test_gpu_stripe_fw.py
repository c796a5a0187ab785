"""Fourier-wavelet stripe removal at the edges of its kernels, against the FP64
oracle: widths below, at and past the 16, 32 and 128 columns of a tile, a wave
and a workgroup, odd widths (element-wise loads), a width whose rows do not
fit the LDS, fewer angles than one 32-angle step, angle groups left empty, term
counts that need one, two and three blocks of 32 and more than fit the LDS, a
sigma that keeps no frequency.

Tolerance: the result is x_0 + d_0 rounded to float32 (6e-8 of x_0); the
correction's own error is below that (24-bit products, FP64 sums), so the
relative error is at most a few roundings: 5e-7.  After -log of
transmissions between 0.2 and 1 an absolute error of 3e-7 is at most 2e-6 of
the sinograms (whose rms is above 0.3)."""
import numpy as np
import pytest
import torch

from oracle import preproc_fp64 as pp

pytestmark = pytest.mark.gpu

CASES = [  # nproj, nz, n, wavelet, level, sigma
    (5, 1, 3, 'sym16', 3, 1.0),
    (31, 2, 15, 'sym5', 2, 1.0),
    (33, 1, 17, 'sym16', 7, 1.0),
    (257, 3, 127, 'db5', 3, 1.0),
    (64, 2, 129, 'haar', 2, 1.0),
    (300, 2, 130, 'sym16', 1, 1.0),
    (120, 4, 1664, 'sym16', 4, 1.0),
    (200, 2, 260, 'db5', 4, 3.0),
    (24, 1, 11000, 'db5', 2, 1.0),
    (40, 1, 64, 'sym16', 2, 0.01),
]


def _transmission(nproj, nz, n, seed):
    rng = np.random.default_rng(seed)
    y, x = np.arange(nproj)[:, None, None], np.arange(n)[None, None, :]
    t = 0.55 + 0.25 * np.sin(y / 9.0 + x / 11.0) + 0.02 * rng.standard_normal((nproj, nz, n))
    return t * (1 + 0.03 * (rng.random((1, nz, n)) < 0.1))


@pytest.mark.parametrize('nproj,nz,n,wname,level,sigma', CASES)
def test_in_place_chunk(nproj, nz, n, wname, level, sigma):
    from tomocupy_amd import ProcFunctions
    data = _transmission(nproj, nz, n, 1).astype(np.float32)
    ref = pp.remove_stripe_fw(data, sigma, wname, level)
    pf = ProcFunctions(nproj, nz, n, 1, 1, remove_stripe_method='fw', fw_sigma=sigma,
                       fw_filter=wname, fw_level=level)
    d = torch.from_numpy(data).cuda()
    pf.remove_stripe_fw(d)
    err = np.linalg.norm(d.cpu().numpy() - ref) / np.linalg.norm(ref)
    print('in place', (nproj, nz, n, wname, level, sigma), 'rel-L2 %.3g' % err)
    assert err <= 5e-7


@pytest.mark.parametrize('flat_linear', [False, True])
@pytest.mark.parametrize('nproj,nz,n,wname,level,sigma', [CASES[i] for i in (0, 2, 3, 6, 7)])
def test_counts_to_sinograms(nproj, nz, n, wname, level, sigma, flat_linear):
    from tomocupy_amd import ProcFunctions
    rng = np.random.default_rng(2)
    gain, dark0 = rng.uniform(20000, 60000, (nz, n)), rng.uniform(90, 110, (nz, n))
    data = np.clip(_transmission(nproj, nz, n, 2) * gain + dark0, 0, 65535).astype(np.uint16)
    dark = rng.poisson(dark0, (3, nz, n)).astype(np.uint16)
    flat = np.clip(rng.poisson(gain + dark0, (7, nz, n)), 0, 65535).astype(np.uint16)
    ref = pp.proc_chain(data, dark, flat, stripe='fw', fw_sigma=sigma, fw_filter=wname,
                        fw_level=level, flat_linear=flat_linear)
    pf = ProcFunctions(nproj, nz, n, 3, 7, flat_linear=flat_linear, remove_stripe_method='fw',
                       fw_sigma=sigma, fw_filter=wname, fw_level=level)
    out = pf.proc_chunk(*(torch.from_numpy(a).cuda() for a in (data, dark, flat)))
    err = np.linalg.norm(out.cpu().numpy() - ref) / np.linalg.norm(ref)
    print('counts', (nproj, nz, n, wname, level, sigma, flat_linear), 'rel-L2 %.3g' % err)
    assert err <= 2e-6
