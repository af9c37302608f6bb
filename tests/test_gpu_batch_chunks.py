"""A batch large enough for the longer bounds chunks (more than 2,048 of 1,024
slots): every instance as its own engine, bit for bit, over border-cell
updates and full scans, with instances that are no whole number of chunks.
"""
import numpy as np
import pytest

from gpu_util import make_engine, perturbed, say
from hipsph import scenarios
from hipsph.batch import BatchEngine, params_for
from hipsph.device import soa_from_particles

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('border', [True, False])
def test_large_batch_matches_engines(border):
    scs = [scenarios.dam_break(1.0, 2.0, d, name=f'chunks{k}') for k, d in enumerate([0.0012, 0.0015, 0.02, 0.05])]
    pAs = [perturbed(sc.pA, 41 + k) for k, sc in enumerate(scs)]
    n = [len(p) for p in pAs]
    say('batch chunks', border, n)
    assert sum(n) > 2048 * 1024
    b = BatchEngine([params_for(sc, 0.02, precision='fp32c') for sc in scs], device='cuda:0')
    b.set_border_bounds(border)
    b.upload([soa_from_particles(p) for p in pAs])
    b.step(5)
    b.download()
    off = 0
    for sc, pA in zip(scs, pAs):
        m = sc.method()
        m.alpha = 0.02
        e = make_engine(pA, m, precision='fp32c')
        e.step(5)
        want = e.download(to_numpy=False)
        e.close()
        for k in ('x', 'y', 'vx', 'vy', 'rho', 'ax', 'ay', 'drho', 'p'):
            np.testing.assert_array_equal(b.io[k][off:off + len(pA)].cpu().numpy(), want[k].cpu().numpy(), err_msg=k)
        off += len(pA)
    b.close()
