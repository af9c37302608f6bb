"""More instances than a launch grid's y axis holds (65,535): every instance
of a batch of 65,600 small ones as an engine of its own, bit for bit.
"""
import numpy as np
import pytest

from gpu_util import make_engine, say
from hipsph import scenarios
from hipsph.batch import BatchEngine, params_for
from hipsph.device import soa_from_particles

pytestmark = pytest.mark.gpu

FIELDS = ('x', 'y', 'vx', 'vy', 'rho', 'ax', 'ay', 'drho')


def _kinds():
    """Three small states, each a corner of a dam break of its own spacing."""
    out = []
    for k, dx in enumerate((0.05, 0.04, 0.03)):
        sc = scenarios.dam_break(0.4, 0.5, dx, tank_w=1.0, tank_h=0.8, name=f'many{k}')
        f = np.nonzero(sc.pA['label'] == 0)[0][:9 + k]
        w = np.nonzero(sc.pA['label'] != 0)[0][:3]
        pA = sc.pA[np.concatenate((f, w))].copy()
        pA['vx'][:9] = 0.1 * (k + 1)
        out.append((sc, pA))
    return out


def test_more_instances_than_a_grid_axis():
    K, cap = 65600, 252
    kinds = _kinds()
    say('batch of', K)
    params, soa = [], []
    for sc, pA in kinds:
        p = params_for(sc, 0.02, cell_capacity=cap)
        p.n = len(pA)
        params.append(p)
        soa.append(soa_from_particles(pA))
    which = np.arange(K) % 3
    b = BatchEngine([params[w] for w in which], device='cuda:0')
    b.upload([soa[w] for w in which])
    b.step(4)
    st = b.status()
    got = b.download()
    b.close()
    for w, (sc, pA) in enumerate(kinds):
        m = sc.method()
        m.alpha = 0.02
        e = make_engine(pA, m, cell_capacity=cap)
        e.step(4)
        want, clock = e.download(), e.status()
        e.close()
        for f in FIELDS:
            all_ = np.stack([got[k][f] for k in range(w, K, 3)])
            np.testing.assert_array_equal(all_, np.broadcast_to(want[f], all_.shape), err_msg=f'kind {w} {f}')
        assert all(st[k]['steps'] == 4 and st[k]['flags'] == clock['flags'] and st[k]['t'] == clock['t']
                   for k in range(w, K, 3))
