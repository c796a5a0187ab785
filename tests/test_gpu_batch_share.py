"""Requests of a batch that together fill the chip, each of them small: the batch's
two modes agree to the bit, and with a plan of its own to rounding (1e-6, the bound
of the autotuner's options, which change only rounding too)."""
import numpy as np
import pytest
import torch

from tomocupy_amd import BackprojFunctions, synth

pytestmark = pytest.mark.gpu


def test_rows_count_together():
    from tomocupy_amd.batch import BatchRec
    sizes = [(512, 600, 8), (256, 200, 2), (512, 601, 7), (768, 510, 6), (512, 580, 7)]
    reqs = [dict(n=n, nz=nz, theta=synth.angles(p)) for n, p, nz in sizes]
    rng = np.random.default_rng(4)
    data = [torch.from_numpy(rng.standard_normal((nz, p, n)).astype(np.float32)).cuda()
            for n, p, nz in sizes]
    out = {}
    for mode in ('streams', 'batched'):
        b = BatchRec(reqs, fbp_filter='shepp', streams=2, grid=mode)
        for d, x in zip(b.inputs(), data):
            d.copy_(x)
        b.run_eager()
        torch.cuda.synchronize()
        out[mode] = [o.clone() for o in b.outputs()]
        b.free()
    for (n, p, nz), x, o, e in zip(sizes, data, out['streams'], out['batched']):
        assert torch.equal(o, e)
        bf = BackprojFunctions(n, p, nz, torch.from_numpy(synth.angles(p)).cuda(), n / 2,
                               'float32', 'shepp')
        ref = torch.empty_like(o)
        bf.fbp_filter_backprojection(ref, x)
        err = float((o - ref).norm() / ref.norm())
        print((n, p, nz), 'rel-L2 %.3g' % err)
        assert err <= 1e-6
        bf.free()
