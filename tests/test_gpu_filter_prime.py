"""Rounding error of the separate filter on padded float32 sinogram rows, smooth with
a little noise, at lengths 8 p with a prime p above 17: not above that of the plain
sum over the prime's inputs, each multiplied by one entry of the length's table,
which is emulated here operation by operation in float32.

Tolerance: both errors are rms values over rows x length independent roundings
(20000 at least, of which the ramp lets an eighth count), so they scatter by
1/sqrt(2 x 2500) = 1.4 percent each, their ratio by 2 percent.  Asserted at 5 percent."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
C8, F4 = np.complex64, np.float32


def _mul(a, w):
    re = (a.real * w.real - a.imag * w.imag).astype(F4)
    return (re + 1j * (a.real * w.imag + a.imag * w.real).astype(F4)).astype(C8)


def _dft8(x):
    """Radix-8 butterflies over axis 0, three rounds of sums and differences."""
    s, d = x[:4] + x[4:], x[:4] - x[4:]
    r = F4(np.sqrt(0.5))
    d = np.stack([d[0], _mul(d[1], C8(r - 1j * r)), -1j * d[2], _mul(d[3], C8(-r - 1j * r))])
    out = []
    for h in (s, d.astype(C8)):
        a, b, c, e = h[0] + h[2], h[1] + h[3], h[0] - h[2], (h[1] - h[3]) * C8(-1j)
        out.append([a + b, c + e, a - b, c - e])
    return np.stack([out[k % 2][k // 2] for k in range(8)])


def _fft(x, p):
    """Float32 transform of the rows of x, length 8 p: the radix-8 pass, then the sum."""
    n = 8 * p
    tab = np.exp(-2j * np.pi * np.arange(n) / n).astype(C8)
    a = _dft8(x.reshape(len(x), 8, p).transpose(1, 0, 2).astype(C8))  # a[k][row][r]
    k = np.arange(8)
    y = np.empty((len(x), n), C8)
    for q in range(p):
        re = np.zeros((8, len(x)), F4)
        im = re.copy()
        for r in range(p):
            w, v = tab[r * (k + 8 * q) % n][:, None], a[:, :, r]
            vr = v.real.astype(np.float64)
            re = re + (vr * w.real - v.imag * w.imag).astype(F4)  # one product is rounded,
            im = im + (vr * w.imag + v.imag * w.real).astype(F4)  # the other goes in exactly
        y[:, k + 8 * q] = (re + 1j * im).T
    return y


@pytest.mark.parametrize('p', [19, 31, 71, 127])
def test_no_worse_than_the_sum(p):
    from tomocupy_amd.fbp_filter import FBPFilter
    ne, pairs = 8 * p, 20000 // (8 * p) + 1
    rng = np.random.default_rng(p)
    n = ne // 4
    pad, t = ne // 2 - n // 2, np.arange(n) - n / 2
    rows = np.zeros((2, pairs, n))
    for z in range(2):
        for i in range(pairs):
            for _ in range(10):
                a, c = rng.uniform(0.05, 0.4) * n / 2, rng.uniform(-0.6, 0.6) * n / 2
                h = rng.uniform(0.05, 0.4) * rng.uniform(0.1, 0.8)
                rows[z, i] += 2 * h * np.sqrt(np.clip(1 - ((t - c) / a)**2, 0, None))
    rows += rng.standard_normal(rows.shape) * np.exp(0.5 * rows) / 173
    rows = np.pad(rows, ((0, 0), (0, 0), (pad, ne - pad - n)), mode='edge').astype(F4)
    ramp = np.minimum(np.arange(ne), ne - np.arange(ne)) / ne
    ref = np.fft.ifft(np.fft.fft(rows.astype(np.float64)) * ramp).real * ne
    z = _fft((rows[0] + 1j * rows[1]).astype(C8), p) * ramp.astype(F4)
    z = np.conj(_fft(np.conj(z).astype(C8), p))
    emulated = np.linalg.norm(np.stack([z.real, z.imag]) - ref)
    flt = FBPFilter(ne, pairs, 2, n_unpadded=n)
    d = torch.from_numpy(rows).cuda()
    w = torch.from_numpy(ramp[:ne // 2 + 1].astype(C8)).cuda().expand(2, -1).contiguous()
    flt.filter(d, w)
    got = np.linalg.norm(d.cpu().numpy().astype(np.float64) - ref)
    print('p=%d error %.3g of the sum %.3g' % (p, got, emulated))
    assert got <= 1.05 * emulated


@pytest.mark.parametrize('ne', [9804, 10184, 14964, 15544, 15776, 16376])
def test_twelve_and_sixteen_pairs(ne):
    """Lengths whose prime passes take 12 or 16 output pairs a wave, white rows.  Two
    transforms of at most five passes, each about 1e-7 of the values: 1e-7 sqrt(10)."""
    from tomocupy_amd.fbp_filter import FBPFilter
    rng = np.random.default_rng(ne)
    rows = rng.standard_normal((2, 5, ne)).astype(F4)
    gain = rng.uniform(0.5, 1, ne // 2 + 1) * np.exp(1j * rng.uniform(-3, 3, ne // 2 + 1))
    gain[0] = gain[-1] = 1
    gain = gain.astype(C8)
    ref = np.fft.irfft(np.fft.rfft(rows.astype(np.float64)) * gain, n=ne) * ne
    flt = FBPFilter(ne, 5, 2, n_unpadded=ne // 8 * 2)
    d = torch.from_numpy(rows).cuda()
    flt.filter(d, torch.from_numpy(gain).cuda().expand(2, -1).contiguous())
    err = np.linalg.norm(d.cpu().numpy() - ref) / np.linalg.norm(ref)
    print('ne=%d error %.3g' % (ne, err))
    assert err <= 1e-7 * np.sqrt(10)
