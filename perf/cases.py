"""What the framework is timed on: reconstructions, stripe removal, a resident scan, the
gradient of the projector, phase retrieval and a batch, through the public entry points.

A case is a dict of plain values with a ``kind``:

* ``rec``    fused FBP filter + backprojection of one chunk of sinograms
             (``BackprojFunctions.fbp_filter_backprojection``), the step every
             reconstruction repeats for each chunk;
* ``split``  the same in the two calls a program ported from the reference makes
             (``fbp_filter_center`` in place, then ``FourierRec.backprojection``);
* ``prep``   detector counts to sinograms (``ProcFunctions.proc_chunk``): dark/flat,
             Fourier-wavelet stripe removal or none, -log, swap;
* ``scan``   a whole resident volume, counts to images, chunk by chunk
             (``GPURec.recon_resident``);
* ``grad``   one step of an iterative or learned reconstruction: the forward projection and
             the gradient of the squared residual (``autograd.project`` and its backward);
* ``phase``  Paganin phase retrieval of a block of projections (``paganin_filter``);
* ``batch``  independent reconstructions of several sizes as one captured graph
             (``BatchRec(grid='batched')``).

Inputs are projections of random ellipses (total optical depth up to about 2) with counting
noise, as float sinograms or uint16 counts with dark and flat frames and column-gain stripes.
``exact`` restates each path in 64 bits with torch and numpy only.
"""
import math

import numpy as np
import torch

DEV = 'cuda'
DTYPES = {'float32': torch.float32, 'float16': torch.float16, 'bfloat16': torch.bfloat16}
BYTES = {'float32': 4, 'float16': 2, 'bfloat16': 2}
NDARK, NFLAT = 10, 20
FW_LEVEL, FW_SIGMA = 7, 1.0
PAGANIN = dict(pixel_size=1.17e-4, dist=6.0, energy=20.0, alpha=1e-4)  # cm, cm, keV


# ---- the cases -----------------------------------------------------------------------


def listed():
    return [
        # one slice pair of a small region of interest, as the try mode repeats it while the
        # rotation centre is searched: latency and launches
        dict(name='rec_256', kind='rec', n=256, nproj=180, nz=2, dtype='float32',
             filter='parzen', shift=0.0),
        # a laboratory scan: 512 columns, two groups of slices in a chunk
        dict(name='rec_512', kind='rec', n=512, nproj=720, nz=16, dtype='float32',
             filter='parzen', shift=0.5),
        # the benchmark's chunk: 2048 columns, 1500 angles, 8 slices
        dict(name='rec_2048', kind='rec', n=2048, nproj=1500, nz=8, dtype='float32',
             filter='ramp', shift=0.5),
        # the same with 16-bit storage
        dict(name='rec_2048_half', kind='rec', n=2048, nproj=1500, nz=8, dtype='float16',
             filter='ramp', shift=0.5),
        # a detector width with the factors 3 and 17
        dict(name='rec_2448', kind='rec', n=2448, nproj=1500, nz=8, dtype='float32',
             filter='shepp', shift=-3.25),
        # the widest detector
        dict(name='rec_4096', kind='rec', n=4096, nproj=3000, nz=8, dtype='float32',
             filter='parzen', shift=0.0),
        # filter and backprojection called one after the other: an odd number of slices and
        # angles, a width with a power of five
        dict(name='split_1000_bf16', kind='split', n=1000, nproj=901, nz=5, dtype='bfloat16',
             filter='hann', shift=1.5),
        # counts to sinograms with stripe removal at the benchmark's chunk
        dict(name='prep_fw_2048', kind='prep', n=2048, nproj=1500, nz=8, dtype='float32',
             stripe='fw'),
        # a resident scan of 32 slices in chunks of 8, with stripe removal
        dict(name='scan_1024', kind='scan', n=1024, nproj=721, nz=32, ncz=8, dtype='float32',
             filter='parzen', stripe='fw', shift=0.5),
        # sparse-view iterative reconstruction: 180 angles, 32 slices
        dict(name='grad_1024', kind='grad', n=1024, nproj=180, nz=32),
        # a block of full-frame projections
        dict(name='phase_2048', kind='phase', nproj=16, dy=2048, dz=2048),
        # requests of several sizes at once
        dict(name='batch_12', kind='batch', count=12, seed=2024, largest=1024),
    ]


def _width(rng, lo, hi):
    """An even detector width: one in two a usual size, otherwise anything the plans take
    (prime factors up to 127; above 2836 only a few odd shapes are accepted)."""
    usual = [w for w in (128, 256, 320, 400, 512, 612, 640, 768, 960, 1024, 1080, 1224, 1280,
                         1536, 1600, 1920, 2048, 2160, 2448, 2560, 3072, 3584, 4096)
             if lo <= w <= hi]
    if rng.random() < 0.5:
        return rng.choice(usual)
    while True:
        n = 2 * int(round(math.exp(rng.uniform(math.log(lo), math.log(min(hi, 2836)))) / 2))
        m = n
        for p in range(2, 128):
            while m % p == 0:
                m //= p
        if m == 1:
            return n


def draw(rng):
    largest = _weight(dict(kind='rec', n=4096, nproj=3000, nz=8))
    while True:
        kind = rng.choices(['rec', 'split', 'prep', 'scan', 'grad', 'phase', 'batch'],
                           [8, 2, 4, 2, 3, 2, 1])[0]
        dtype = rng.choices(['float32', 'float16', 'bfloat16'], [6, 2, 1])[0]
        fil = rng.choice(['parzen', 'ramp', 'shepp', 'hann', 'hamming', 'cosine'])
        shift = rng.choice([0.0, 0.5, round(rng.uniform(-8, 8), 2)])
        if kind in ('rec', 'split'):
            n = _width(rng, 128, 4096)
            c = dict(kind=kind, n=n, nproj=int(n * rng.uniform(0.3, 1.5)) + 1,
                     nz=rng.choice([1, 2, 4, 5, 8, 8, 16]), dtype=dtype, filter=fil, shift=shift)
        elif kind == 'prep':
            n = _width(rng, 128, 4096)
            c = dict(kind=kind, n=n, nproj=int(n * rng.uniform(0.3, 1.5)) + 1,
                     nz=rng.choice([1, 2, 4, 7, 8, 16]), dtype=dtype,
                     stripe=rng.choice(['fw', 'fw', 'none']))
        elif kind == 'scan':
            n = _width(rng, 256, 2048)
            ncz = rng.choice([2, 4, 8])
            c = dict(kind=kind, n=n, nproj=int(n * rng.uniform(0.3, 1.0)) + 1,
                     nz=ncz * rng.randint(2, 4), ncz=ncz, dtype=dtype, filter=fil,
                     stripe=rng.choice(['fw', 'none']), shift=shift)
        elif kind == 'grad':
            n = _width(rng, 128, 2048)
            c = dict(kind=kind, n=n, nproj=int(n * rng.uniform(0.1, 0.8)) + 1,
                     nz=rng.choice([1, 2, 3, 8, 16, 32]))
        elif kind == 'phase':
            c = dict(kind=kind, nproj=rng.randint(2, 24), dy=2 * rng.randint(64, 1024),
                     dz=2 * rng.randint(128, 1280))
        else:
            c = dict(kind=kind, count=rng.randint(3, 16), seed=rng.randrange(1 << 20),
                     largest=rng.choice([512, 768, 1024]))
        if kind in ('rec', 'split', 'prep', 'scan', 'grad') and c['nproj'] < 16:
            continue
        if _weight(c) <= largest:
            return c


def _requests(case):
    """The batch's requests: ``(n, nproj, nz)`` each."""
    rng = np.random.default_rng(case['seed'])
    sizes = [s for s in (256, 384, 512, 768, 1024) if s <= case['largest']]
    return [(int(rng.choice(sizes)), int(rng.integers(100, 700)), int(rng.integers(1, 9)))
            for _ in range(case['count'])]


def _weight(c):
    """A rough cost of a pass in bytes moved, to keep the drawn cases within the listed ones."""
    if c['kind'] == 'phase':
        return c['nproj'] * 16.0 * 4 * c['dy'] * c['dz'] * 4
    if c['kind'] == 'batch':
        return sum(_weight(dict(kind='rec', n=n, nproj=p, nz=z)) for n, p, z in _requests(c))
    grid = 10 * 16 * c['n'] ** 2
    one = c['nz'] * (c['nproj'] * c['n'] * 30 + (0 if c['kind'] == 'prep' else grid))
    return one * (3 if c['kind'] == 'grad' else 1)


def work(case):
    """Bytes: each input read once, each output written once.  Flops: the transforms at
    5 N log2 N, 8 for each tap of the 9 x 9 gridding footprint of a complex sample."""
    k = case['kind']
    if k == 'phase':
        px = case['nproj'] * case['dy'] * case['dz']
        full = case['nproj'] * 4 * case['dy'] * case['dz']
        return {'bytes': 8.0 * px, 'flops': 2 * 5.0 * full * math.log2(4 * case['dy'] * case['dz'])}
    if k == 'batch':
        parts = [work(dict(kind='rec', n=n, nproj=p, nz=z, dtype='float32'))
                 for n, p, z in _requests(case)]
        return {q: sum(p[q] for p in parts) for q in ('bytes', 'flops')}
    n, nproj, nz = case['n'], case['nproj'], case['nz']
    sino, img = nz * nproj * n, nz * n * n
    nzc = (nz + 1) // 2
    plane = nzc * 5.0 * (4 * n * n) * math.log2(4 * n * n)
    rows = nzc * nproj * 5.0 * n * math.log2(n)
    gridding = nzc * nproj * n * 81 * 4.0
    if k == 'grad':
        # projection and its transpose; the images in and out, the measured data, the residual
        return {'bytes': 4.0 * (2 * img + 2 * sino), 'flops': 2 * (plane + rows + gridding)}
    b = BYTES[case['dtype']]
    flt = nzc * nproj * 2 * 5.0 * 2 * n * math.log2(2 * n)
    fw = 0.0
    if case.get('stripe') == 'fw':
        # two directions, analysis and synthesis, 32 taps, all levels
        fw = sino * 32 * 2 * 4.0
    if k == 'prep':
        return {'bytes': sino * (2.0 + b) + (NDARK + NFLAT) * nz * n * 2.0,
                'flops': fw + 10.0 * sino}
    if k == 'scan':
        return {'bytes': 2.0 * sino + (NDARK + NFLAT) * nz * n * 2.0 + b * img,
                'flops': fw + 10.0 * sino + flt + rows + gridding + plane}
    return {'bytes': float(b) * (sino + img) + (b * sino if k == 'split' else 0.0),
            'flops': flt + rows + gridding + plane}


# ---- inputs --------------------------------------------------------------------------


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _theta(nproj):
    return (np.arange(nproj) * np.pi / nproj).astype(np.float32)


def _optical_depth(n, nproj, nz, seed):
    """Float32 sinograms (nz, nproj, n) of 10 random ellipses for each slice."""
    rng = np.random.default_rng(int(seed))
    r = n / 2
    s = torch.arange(n, device=DEV, dtype=torch.float32) - r
    th = torch.from_numpy(_theta(nproj)).to(DEV)
    out = torch.zeros((nz, nproj, n), device=DEV)
    for z in range(nz):
        for _ in range(10):
            a, b = rng.uniform(0.05, 0.4, 2) * r
            rad, ang = r * math.sqrt(rng.uniform(0, 0.8)), rng.uniform(0, 2 * math.pi)
            phi, rho = rng.uniform(0, math.pi), rng.uniform(0.1, 0.8) / r
            h2 = (a * torch.cos(th + phi)) ** 2 + (b * torch.sin(th + phi)) ** 2
            s0 = rad * torch.cos(th + ang)
            d2 = (h2[:, None] - (s[None, :] - s0[:, None]) ** 2).clamp_(min=0)
            out[z] += (2 * a * b * rho) * d2.sqrt_() / h2[:, None]
    return out


def _sinograms(n, nproj, nz, dtype, seed):
    """-log sinograms with the noise of 30000 counts a pixel, in the storage type."""
    p = _optical_depth(n, nproj, nz, seed)
    p += torch.randn(p.shape, generator=_gen(seed), device=DEV) * torch.exp(0.5 * p) / 173.0
    return p.to(DTYPES[dtype])


def _measured(n, nproj, nz, seed):
    """Sinograms at the scale of the forward projections of ``_images``."""
    return 5.0 * n / nproj * _sinograms(n, nproj, nz, 'float32', seed)


def _counts(n, nproj, nz, seed):
    """uint16 detector counts: projections (nproj, nz, n), darks and flats."""
    g = _gen(seed)
    u = lambda lo, hi: lo + (hi - lo) * torch.rand((nz, n), generator=g, device=DEV)
    gain, dark = 30000 * u(0.98, 1.02), u(95, 105)
    stripe = torch.where(u(0, 1) < 0.05, u(0.97, 1.03), torch.ones((nz, n), device=DEV))
    to16 = lambda x: (torch.poisson(x, generator=g).clamp_(0, 65535).to(torch.int32)
                      .to(torch.int16).view(torch.uint16))
    lam = (gain * stripe)[:, None] * torch.exp(-_optical_depth(n, nproj, nz, seed)) + dark[:, None]
    data = to16(lam.transpose(0, 1).contiguous())
    darks = to16(dark.expand(NDARK, nz, n).contiguous())
    flats = to16((gain + dark).expand(NFLAT, nz, n).contiguous())
    return data, darks, flats


def _images(n, nz, seed):
    """Smooth images inside the circle, as an iterate of a reconstruction holds them."""
    g = _gen(seed)
    coarse = torch.rand((nz, 1, 16, 16), generator=g, device=DEV)
    img = torch.nn.functional.interpolate(coarse, size=(n, n), mode='bilinear')[:, 0]
    return (img + 0.02 * torch.randn((nz, n, n), generator=g, device=DEV)).contiguous()


def _projections(case, seed):
    """Transmission images (nproj, dy, dz) with edge enhancement and counting noise."""
    dy, dz = case['dy'], case['dz']
    p = _optical_depth(dz, case['nproj'], dy // 64 + 1, seed)  # (rows / 64, nproj, dz)
    p = torch.nn.functional.interpolate(p.permute(1, 0, 2)[:, None], size=(dy, dz),
                                        mode='bilinear')[:, 0]
    x = torch.exp(-p)
    x += torch.randn(x.shape, generator=_gen(seed), device=DEV) * x.sqrt() / 173.0
    return x.contiguous()


def _scan_inputs(case, seed):
    """Chunk-major counts: (chunks, nproj | ndark | nflat, ncz, n)."""
    parts = [_counts(case['n'], case['nproj'], case['ncz'], 1000 * seed + k)
             for k in range(case['nz'] // case['ncz'])]
    # (torch.stack has no uint16 form on the GPU: stack the same bits as int16)
    return tuple(torch.stack([p[i].view(torch.int16) for p in parts]).view(torch.uint16)
                 for i in range(3))


# ---- the framework's calls -----------------------------------------------------------


def prepare(case, seed):
    k = case['kind']
    st = dict(case=case)
    if k == 'phase':
        st['raw'] = _projections(case, seed)
        st['data'] = torch.empty_like(st['raw'])
        return st
    if k == 'batch':
        from tomocupy_amd.batch import BatchRec
        reqs = [dict(n=n, nz=z, theta=_theta(p)) for n, p, z in _requests(case)]
        b = BatchRec(reqs, grid='batched')
        for i, ((n, p, z), d) in enumerate(zip(_requests(case), b.inputs())):
            d.copy_(_sinograms(n, p, z, 'float32', 1000 * seed + i))
        b.capture()
        st['batch'] = b
        return st
    n, nproj, nz = case['n'], case['nproj'], case['nz']
    theta = torch.from_numpy(_theta(nproj)).to(DEV)
    if k == 'grad':
        from tomocupy_amd.fourierrec import FourierRec
        st['rec'] = FourierRec(n, nproj, nz, theta, 'float32')
        st['x'] = _images(n, nz, seed).requires_grad_()
        st['data'] = _measured(n, nproj, nz, seed)
        return st
    dt = DTYPES[case['dtype']]
    if k == 'prep':
        from tomocupy_amd.proc_functions import ProcFunctions
        st['pf'] = ProcFunctions(nproj, nz, n, NDARK, NFLAT, case['dtype'],
                                 remove_stripe_method=case['stripe'], fw_sigma=FW_SIGMA,
                                 fw_filter='sym16', fw_level=FW_LEVEL)
        st['in'] = _counts(n, nproj, nz, seed)
        st['out'] = torch.empty((nz, nproj, n), dtype=dt, device=DEV)
        return st
    if k == 'scan':
        from tomocupy_amd.rec import GPURec
        st['gr'] = GPURec(n, nproj, nz, case['ncz'], theta, n / 2 + case['shift'], NDARK, NFLAT,
                          case['dtype'], fbp_filter=case['filter'],
                          remove_stripe_method=case['stripe'], fw_sigma=FW_SIGMA,
                          fw_filter='sym16', fw_level=FW_LEVEL)
        st['in'] = _scan_inputs(case, seed)
        st['out'] = torch.empty((nz, n, n), dtype=dt, device=DEV)
        return st
    from tomocupy_amd.backproj_functions import BackprojFunctions
    st['bf'] = BackprojFunctions(n, nproj, nz, theta, n / 2 + case['shift'], case['dtype'],
                                 case['filter'])
    st['data'] = _sinograms(n, nproj, nz, case['dtype'], seed)
    st['out'] = torch.empty((nz, n, n), dtype=dt, device=DEV)
    if k == 'split':
        st['filtered'] = torch.empty_like(st['data'])
    return st


def run(st):
    k = st['case']['kind']
    if k == 'rec':
        return st['bf'].fbp_filter_backprojection(st['out'], st['data'])
    if k == 'split':
        # (the filter works in place: the program keeps its sinograms)
        st['filtered'].copy_(st['data'])
        st['bf'].fbp_filter_center(st['filtered'])
        st['bf'].cl_rec.backprojection(st['out'], st['filtered'])
        return {'filtered': st['filtered'], 'images': st['out']}
    if k == 'prep':
        return st['pf'].proc_chunk(*st['in'], out=st['out'])
    if k == 'scan':
        # the driver works on its own stream, between what the program queued before and after
        cur, own = torch.cuda.current_stream(), st['gr'].stream2
        own.wait_stream(cur)
        st['gr'].recon_resident(*st['in'], st['out'])
        cur.wait_stream(own)
        return st['out']
    if k == 'grad':
        from tomocupy_amd.autograd import project
        y = project(st['x'], st['rec'])
        (g,) = torch.autograd.grad(y, st['x'], y.detach() - st['data'])
        return {'projection': y.detach(), 'gradient': g}
    if k == 'phase':
        from tomocupy_amd.retrieve_phase import paganin_filter
        # (the filter works in place: the program keeps its projections)
        st['data'].copy_(st['raw'])
        return paganin_filter(st['data'], **PAGANIN)
    st['batch'].run()
    return st['batch'].outputs()


# ---- the same in 64 bits -------------------------------------------------------------

_SYM16 = np.array([  # sym16 decomposition low-pass taps
    6.230006701220761e-06, -3.113556407621969e-06, -0.00010943147929529757,
    2.8078582128442894e-05, 0.0008523547108047095, -0.0001084456223089688,
    -0.0038809122526038786, 0.0007182119788317892, 0.012666731659857348,
    -0.0031265171722710075, -0.031051202843553064, 0.004869274404904607,
    0.032333091610663785, -0.06698304907021778, -0.034574228416972504, 0.39712293362064416,
    0.7565249878756971, 0.47534280601152273, -0.054040601387606135, -0.15959219218520598,
    0.03072113906330156, 0.07803785290341991, -0.003510275068374009, -0.024952758046290123,
    0.001359844742484172, 0.0069377611308027096, -0.00022211647621176323,
    -0.0013387206066921965, 3.656592483348223e-05, 0.00016545679579108483,
    -5.396483179315242e-06, -1.0797982104319795e-05])


def _analysis(x, dim):
    """Half-sample symmetric extension and stride-2 filtering: (low, high) along ``dim``."""
    L = len(_SYM16)
    x = x.movedim(dim, -1)
    N = x.shape[-1]
    No = (N + L - 1) // 2
    pad = (2 * (No - 1) - N + L) // 2
    i = (np.arange(2 * No + L - 2) - pad) % (2 * N)
    x = x[..., torch.from_numpy(np.where(i >= N, 2 * N - 1 - i, i)).to(x.device)]
    lo = torch.zeros(x.shape[:-1] + (No,), dtype=x.dtype, device=x.device)
    hi = torch.zeros_like(lo)
    for j in range(L):
        part = x[..., j:j + 2 * No - 1:2]
        lo += _SYM16[L - 1 - j] * part
        hi += (-1) ** (L - j) * _SYM16[j] * part
    return lo.movedim(-1, dim), hi.movedim(-1, dim)


def _synthesis(lo, hi, dim):
    L = len(_SYM16)
    lo, hi = lo.movedim(dim, -1), hi.movedim(dim, -1)
    N = lo.shape[-1]
    y = torch.zeros(lo.shape[:-1] + (2 * N + L - 2,), dtype=lo.dtype, device=lo.device)
    for j in range(L):
        y[..., j:j + 2 * N - 1:2] += _SYM16[L - 1 - j] * lo + (-1) ** (L - j) * _SYM16[j] * hi
    return y[..., L - 2:2 * N].movedim(-1, dim)


def _stripes64(x):
    """Fourier-wavelet stripe removal of transmissions (nz, nproj, n)."""
    nz, nproj, n = x.shape
    pad = nproj // 8
    st = pad // 2
    s = torch.zeros((nz, nproj + pad, n), dtype=x.dtype, device=x.device)
    s[:, st:st + nproj] = x
    bands = []
    for _ in range(FW_LEVEL):
        lo, hi = _analysis(s, -1)
        s, lh = _analysis(lo, -2)
        hl, hh = _analysis(hi, -2)
        my = hl.shape[-2]
        y = np.fft.ifftshift((np.arange(-my, my, 2) + 1) / 2)[:my // 2 + 1]
        damp = torch.from_numpy(-np.expm1(-y ** 2 / (2 * FW_SIGMA ** 2))).to(x.device)
        hl = torch.fft.irfft(torch.fft.rfft(hl, dim=-2) * damp[:, None], n=my, dim=-2)
        bands.append((lh, hl, hh))
    for lh, hl, hh in reversed(bands):
        s = s[..., :lh.shape[-2], :lh.shape[-1]]
        s = _synthesis(_synthesis(s, lh, -2), _synthesis(hl, hh, -2), -1)
    return s[:, st:st + nproj, :n]


def _prep64(data, dark, flat, stripe):
    f = lambda a: a.view(torch.int16).to(torch.int32).bitwise_and_(0xffff).to(torch.float64)
    dark0, flat0 = f(dark).mean(0), f(flat).mean(0) * float(np.float32(1 + 1e-5))
    x = ((f(data) - dark0) / (flat0 - dark0)).transpose(0, 1).contiguous()
    if stripe == 'fw':
        x = _stripes64(x)
    return -torch.log(torch.where(x <= 0, torch.ones_like(x), x))


def _quadrature(t, m=12):
    """Weights w with sum_j w_j f_j = integral of t f(t): degree-(m-1) polynomials through
    every m neighbouring samples, averaged over the windows that share an interval; the last 40
    weights are a line through zero."""
    N = len(t)
    s = np.linspace(1e-40, 1, m)
    inv = np.linalg.inv(s[None, :] ** np.arange(m)[:, None])
    moments = np.diff(s[None, :] ** np.arange(1, m + 2)[:, None] / np.arange(1, m + 2)[:, None])
    quad, lin = inv @ moments[1:], inv @ moments[:-1]
    share = 1.0 / np.minimum(np.minimum(np.arange(1, N), np.arange(N - 1, 0, -1)), m - 1)
    j = np.arange(N - m + 1)
    h = t[j + m - 1] - t[j]
    w = np.zeros(N)
    for i in range(m):
        c = np.zeros(len(j))
        for k in range(m - 1):
            c += share[j + k] * (h * h * quad[i, k] + h * t[j] * lin[i, k])
        w[i:i + len(j)] += c
    w[-40:] = w[-40] / (N - 40) * np.arange(N - 40, N)
    return w


def _filter64(name, ne):
    t = np.arange(ne // 2 + 1) / ne
    win = {'ramp': np.ones_like(t), 'shepp': np.sinc(t), 'cosine': np.cos(np.pi * t),
           'hamming': 0.54 + 0.46 * np.cos(2 * np.pi * t),
           'hann': 0.5 + 0.5 * np.cos(2 * np.pi * t), 'parzen': (1 - 2 * t) ** 3}[name]
    w = np.maximum(_quadrature(t) * win, 0.0)
    w[0] *= 2
    return w


def _fbp64(data, case):
    """Edge-replicated rows of length ne, filtered, shifted to the rotation axis, cropped."""
    n = data.shape[-1]
    ne = 4 * n if case['dtype'] != 'float16' else 2 ** math.ceil(math.log2(4 * n))
    pad = ne // 2 - n // 2
    f = np.arange(ne // 2 + 1) / ne
    w = _filter64(case['filter'], ne) * np.exp(2j * np.pi * case['shift'] * f)
    w = torch.from_numpy(w * ne).to(data.device)
    out = torch.empty_like(data)
    for z in range(data.shape[0]):
        x = data[z]
        x = torch.cat([x[:, :1].expand(-1, pad), x, x[:, -1:].expand(-1, ne - pad - n)], 1)
        out[z] = torch.fft.irfft(torch.fft.rfft(x) * w, n=ne)[:, pad:pad + n]
    return out


class _Usfft64:
    """The Gaussian-gridding transform between images and sinograms and its transpose."""

    def __init__(self, n, nproj, theta=None):
        self.n, self.nproj = n, nproj
        th = (_theta(nproj) if theta is None else theta).astype(np.float64)
        t = (np.arange(n) - n // 2) / n
        xy = np.stack([t * np.cos(th)[:, None], -t * np.sin(th)[:, None]])
        xy = 2 * n * np.where(xy >= 0.5, 0.5 - 1e-5, xy)
        self.cell = torch.from_numpy(np.floor(xy)).to(DEV).to(torch.int64)
        self.frac = torch.from_numpy(xy - np.floor(xy)).to(DEV)
        mu = math.log(1e3) / (2.0 * n * n)
        self.c1 = -math.pi ** 2 / (mu * 4.0 * n * n)
        self.scale = 4.0 / n * math.pi / (mu * 4.0 * n * n)
        d = np.arange(n) / n - 0.5
        phi = np.exp(mu * n * n * (d[:, None] ** 2 + d[None, :] ** 2)) / nproj * (1 - n % 4)
        u = (np.arange(n) - n // 2) / n
        phi *= 4 * (u[:, None] ** 2 + u[None, :] ** 2) < 1
        self.phi = torch.from_numpy(phi).to(DEV)
        sign = lambda m: (2.0 * (torch.arange(m, device=DEV) % 2) - 1).to(torch.float64)
        self.s1, s2 = sign(n), sign(2 * n)
        self.s2 = s2[:, None] * s2[None, :]

    def _taps(self):
        """For blocks of angles: flat cells and weights of the 81 taps of each sample."""
        n2 = 2 * self.n
        i = torch.arange(9, device=DEV)
        step = max(1, (1 << 24) // (81 * self.n))
        for p in range(0, self.nproj, step):
            at = slice(p, p + step)
            c = (self.cell[:, at, :, None] + self.n - 4 + i) % n2
            w = torch.exp(self.c1 * (i - 4 - self.frac[:, at, :, None]) ** 2)
            cells = c[1][..., :, None] * n2 + c[0][..., None, :]
            yield at, cells.reshape(-1), w[1][..., :, None] * w[0][..., None, :]

    def images(self, data):
        n, nz = self.n, data.shape[0]
        nzc = (nz + 1) // 2
        g = torch.zeros((nzc,) + data.shape[1:], dtype=torch.complex128, device=DEV)
        g.real.copy_(data[:nzc])
        g.imag[:nz - nzc].copy_(data[nzc:])
        G = self.scale * self.s1 * torch.fft.fft(self.s1 * g)
        out = torch.empty((nz, n, n), dtype=torch.float64, device=DEV)
        F = torch.zeros((nzc, 2, 4 * n * n), dtype=torch.float64, device=DEV)
        for at, cells, w in self._taps():
            for c in range(nzc):
                v = G[c, at][..., None, None]
                F[c, 0].scatter_add_(0, cells, (w * v.real).reshape(-1))
                F[c, 1].scatter_add_(0, cells, (w * v.imag).reshape(-1))
        for c in range(nzc):
            f = torch.complex(F[c, 0], F[c, 1]).view(2 * n, 2 * n) * self.s2
            f = torch.fft.ifft2(f, norm='forward') * self.s2
            f = f[n // 2 + 1:n // 2 + 1 + n, n // 2:n // 2 + n] * self.phi
            out[c] = f.real
            if nzc + c < nz:
                out[nzc + c] = f.imag
        return out

    def sinograms(self, obj):
        n, nz = self.n, obj.shape[0]
        nzc = (nz + 1) // 2
        G = torch.zeros((nzc, self.nproj, n), dtype=torch.complex128, device=DEV)
        planes = []
        for c in range(nzc):
            f = torch.zeros((2 * n, 2 * n), dtype=torch.complex128, device=DEV)
            im = obj[nzc + c] if nzc + c < nz else torch.zeros_like(obj[0])
            f[n // 2 + 1:n // 2 + 1 + n, n // 2:n // 2 + n] = torch.complex(obj[c], im) * self.phi
            planes.append((torch.fft.fft2(f * self.s2) * self.s2).reshape(-1))
        for at, cells, w in self._taps():
            for c in range(nzc):
                G[c, at] = (planes[c][cells].view(w.shape) * w).sum((-1, -2))
        g = self.s1 * torch.fft.ifft(self.s1 * G * self.scale, norm='forward')
        return torch.cat([g.real, g.imag[:nz - nzc]])


def _paganin64(x):
    wl = 2 * 3.14159265359 * 6.58211928e-19 * 299792458e+2 / PAGANIN['energy']
    ps, dist = PAGANIN['pixel_size'], PAGANIN['dist']
    _, dy, dz = x.shape

    def grid(dim):
        wide = math.ceil(3.14159265359 * wl * dist / ps ** 2)
        pad = int((2 ** math.ceil(math.log2(dim + wide)) - dim) * 0.5)
        m = dim + 2 * pad
        return pad, torch.from_numpy(np.arange(1 - m, m, 2) * (0.5 / ((m - 1) * ps))).to(x.device)

    (py, ry), (pz, rz) = grid(dy), grid(dz)
    h = 1 / (wl * dist * (ry[:, None] ** 2 + rz[None, :] ** 2) / (4 * 3.14159265359)
             + PAGANIN['alpha'])
    h = torch.fft.fftshift(h / h.max())
    iy = torch.arange(-py, dy + py, device=x.device).clamp_(0, dy - 1)
    iz = torch.arange(-pz, dz + pz, device=x.device).clamp_(0, dz - 1)
    out = torch.empty(x.shape, dtype=torch.float64, device=x.device)
    for m in range(x.shape[0]):
        p = x[m].to(torch.float64)[iy][:, iz]
        out[m] = torch.fft.ifft2(torch.fft.fft2(p) * h).real[py:py + dy, pz:pz + dz]
    return out


def exact(case, seed):
    k = case['kind']
    if k == 'phase':
        return _paganin64(_projections(case, seed))
    if k == 'batch':
        out = []
        for i, (n, p, z) in enumerate(_requests(case)):
            x = _sinograms(n, p, z, 'float32', 1000 * seed + i).to(torch.float64)
            x = _fbp64(x, dict(dtype='float32', filter='parzen', shift=0.0))
            out.append(_Usfft64(n, p).images(x))
        return out
    n, nproj, nz = case['n'], case['nproj'], case['nz']
    if k == 'prep':
        return _prep64(*_counts(n, nproj, nz, seed), case['stripe'])
    if k == 'grad':
        op = _Usfft64(n, nproj)
        y = op.sinograms(_images(n, nz, seed).to(torch.float64))
        data = _measured(n, nproj, nz, seed).to(torch.float64)
        return {'projection': y, 'gradient': op.images(y - data)}
    op = _Usfft64(n, nproj)
    if k == 'scan':
        out = []
        for chunk in zip(*_scan_inputs(case, seed)):
            out.append(op.images(_fbp64(_prep64(*chunk, case['stripe']), case)))
        return torch.cat(out)
    x = _fbp64(_sinograms(n, nproj, nz, case['dtype'], seed).to(torch.float64), case)
    if k == 'split':
        return {'filtered': x, 'images': op.images(x)}
    return op.images(x)
