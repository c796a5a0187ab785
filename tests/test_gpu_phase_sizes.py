"""Phase retrieval over its padded lengths (run-time plans below 512, each
compiled length, half a row of spectrum narrower than a block of columns)
against the FP64 oracle.

Tolerance: two 2-D transforms of at most eight passes each way, a pass adding
about 1e-7 relative to the image's rms, and a factor of three roundings: below
1e-6, asserted at 2e-6."""
import numpy as np
import pytest
import torch

from oracle import phase_fp64 as ph
from tomocupy_amd import retrieve_phase as rp

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('dy,dz,dist,method', [
    (2, 6, 0.01, 'paganin'), (6, 20, 0.01, 'Gpaganin'), (30, 2, 0.01, 'paganin'),
    (50, 118, 5.0, 'paganin'), (200, 202, 5.0, 'Gpaganin'), (300, 6, 0.01, 'paganin'),
    (500, 500, 5.0, 'paganin'), (20, 900, 5.0, 'paganin'), (1000, 300, 5.0, 'Gpaganin'),
    (1500, 2000, 5.0, 'paganin'), (3000, 130, 5.0, 'paganin'), (100, 4090, 5.0, 'paganin'),
    (5000, 60, 5.0, 'paganin')])
def test_padded_lengths(dy, dz, dist, method):
    kw = dict(pixel_size=1e-4, dist=dist, energy=20.0, db=1000.0, W=2e-4, alpha=1e-3)
    rng = np.random.default_rng(dy * dz)
    data = np.exp(-rng.random((5, dy, dz))).astype(np.float32)
    ref = ph.retrieve_phase(data.astype(np.float64), method, **kw)
    g = torch.from_numpy(data).cuda()
    plan = rp.PhasePlan(dy, dz, method, **kw, batch=2)
    plan.apply(g)
    err = np.linalg.norm(g.cpu().numpy() - ref) / np.linalg.norm(ref)
    print('%d x %d padded %d x %d %s %.3g' % (dy, dz, plan.Ny, plan.Nx, method, err))
    assert err <= 2e-6
