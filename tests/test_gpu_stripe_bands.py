"""Fourier-wavelet stripe removal of scans of few angles and many columns, which run
band by band, and a change of settings from one form to the other within a plan,
against the FP64 oracle: each filter length, notches of up to 8, 16 and 32
frequencies, odd widths, both outputs.

Tolerance: a chain of at most 4 level filters of 32 taps each way in float32 on the
correction alone, which is a few per cent of x_0, and x_0 + d_0 rounded once
(6e-8): below 3e-7, asserted at 5e-7; after -log of transmissions between 0.2 and
1 at 2e-6, as for the low-rank form."""
import numpy as np
import pytest
import torch

from oracle import preproc_fp64 as pp

pytestmark = pytest.mark.gpu

CASES = [  # nproj, nz, n, wavelet, level, sigma
    (16, 24, 2048, 'sym16', 7, 3.0),
    (9, 80, 1023, 'sym16', 3, 1.0),
    (24, 32, 2047, 'sym16', 2, 2.0),
    (16, 64, 1400, 'db5', 4, 1.0),
    (33, 96, 1026, 'sym5', 4, 2.0),
    (8, 260, 600, 'haar', 7, 1.0),
    (16, 160, 515, 'haar', 3, 3.0),
    (80, 64, 2048, 'sym16', 7, 8.0),
]


def _transmission(nproj, nz, n, seed):
    rng = np.random.default_rng(seed)
    y, x = np.arange(nproj)[:, None, None], np.arange(n)[None, None, :]
    t = 0.55 + 0.25 * np.sin(y / 9.0 + x / 11.0) + 0.02 * rng.standard_normal((nproj, nz, n))
    return t * (1 + 0.03 * (rng.random((1, nz, n)) < 0.1))


def _rel(a, b):
    return float(np.linalg.norm(a - b) / np.linalg.norm(b))


def _ran(call, kernel):
    """The call's result and whether it launched the kernel."""
    from tomocupy_amd import _lib
    _lib.prof_enable(True)
    _lib.prof_reset()
    out = call()
    torch.cuda.synchronize()
    count = _lib.prof_read(kernel)[1]
    _lib.prof_enable(False)
    return out, count > 0


@pytest.mark.parametrize('nproj,nz,n,wname,level,sigma', CASES)
def test_in_place_chunk(nproj, nz, n, wname, level, sigma):
    from tomocupy_amd import ProcFunctions
    data = _transmission(nproj, nz, n, 1).astype(np.float32)
    ref = pp.remove_stripe_fw(data, sigma, wname, level)
    pf = ProcFunctions(nproj, nz, n, 1, 1, remove_stripe_method='fw', fw_sigma=sigma,
                       fw_filter=wname, fw_level=level)
    d = torch.from_numpy(data).cuda()
    _, bands = _ran(lambda: pf.remove_stripe_fw(d), 'k_fw_syn_rows')
    err = _rel(d.cpu().numpy(), ref)
    print('in place', (nproj, nz, n, wname, level, sigma), 'rel-L2 %.3g' % err)
    assert bands and err <= 5e-7


@pytest.mark.parametrize('flat_linear', [False, True])
@pytest.mark.parametrize('nproj,nz,n,wname,level,sigma', [CASES[i] for i in (1, 3, 6)])
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
    args = [torch.from_numpy(a).cuda() for a in (data, dark, flat)]
    out, bands = _ran(lambda: pf.proc_chunk(*args), 'k_fw_syn_rows')
    err = _rel(out.cpu().numpy(), ref)
    print('counts', (nproj, nz, n, wname, level, sigma, flat_linear), 'rel-L2 %.3g' % err)
    assert bands and err <= 2e-6


def test_settings_change():
    # wide and narrow notches in turn: bands, low rank, bands again, twice
    from tomocupy_amd import ProcFunctions
    nproj, nz, n = 40, 48, 2048
    data = _transmission(nproj, nz, n, 3).astype(np.float32)
    pf = ProcFunctions(nproj, nz, n, 1, 1, remove_stripe_method='fw')
    seen = []
    for sigma in (8.0, 1.0, 8.0, 8.0):
        pf.fw_sigma = sigma
        d = torch.from_numpy(data).cuda()
        _, bands = _ran(lambda: pf.remove_stripe_fw(d), 'k_fw_syn_rows')
        seen.append(bands)
        assert _rel(d.cpu().numpy(), pp.remove_stripe_fw(data, sigma, 'sym16', 7)) <= 5e-7
    assert seen == [True, False, True, True]
