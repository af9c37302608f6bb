"""Batch instances on both sides of the sizes up to which every tile and chunk
has partials of its own (512 tiles of 256 slots; 128 chunks of 1,024, or of 4,096
in batches of more than 2,097,152): every instance as an engine of its own, bit
for bit, over border-cell updates and full scans, where the fused pass and
where the corrector leaves the dt partials, again after a second upload of
calmer states (the first's partials are gone), and past the end of one instance.
"""
import numpy as np
import pytest

from gpu_util import make_engine, perturbed, say
from hipsph import scenarios
from hipsph.batch import BatchEngine, params_for
from hipsph.device import soa_from_particles

pytestmark = pytest.mark.gpu

FIELDS = ('x', 'y', 'vx', 'vy', 'rho', 'ax', 'ay', 'drho')


def _cut(n, seed, vscale):
    """The first n particles of a dam break."""
    sc = scenarios.dam_break(1.0, 2.0, float(np.sqrt(1.96 / n)), name='large')
    pA = perturbed(sc.pA, seed, vscale=vscale)
    assert len(pA) >= n
    return sc, pA[:n].copy()


SIZES = {'small chunks': [131072, 131073, 5000, 400000, 65537],
         'large chunks': [800000, 524288, 524289, 300000]}


@pytest.mark.parametrize('integrator', ['pec', 'euler'])
@pytest.mark.parametrize('border', [True, False])
@pytest.mark.parametrize('sizes', list(SIZES))
def test_instances_match_engines(sizes, border, integrator):
    n = SIZES[sizes]
    assert (sum(n) > 2048 * 1024) == (sizes == 'large chunks')
    say('large instances', sizes, border, integrator)
    b = None
    for seed, vscale in ((71, 3.0), (72, 0.05)):
        cut = [_cut(k, seed + j, vscale) for j, k in enumerate(n)]
        soa = [soa_from_particles(pA) for _, pA in cut]
        if b is None:
            params = [params_for(sc, 0.02, precision='fp32c', integrator=integrator) for sc, _ in cut]
            for k, p in enumerate(params):
                p.n = n[k]
            params[2].duration = 1e-12  # over after the first step
            b = BatchEngine(params, device='cuda:0')
            b.set_border_bounds(border)
        b.upload(soa)
        b.step(5)
        st = b.status()
        got = b.download()
        for k, (sc, pA) in enumerate(cut):
            m = sc.method()
            m.alpha = 0.02
            e = make_engine(pA, m, precision='fp32c', integrator=integrator, duration=params[k].duration)
            e.step(5)
            want, clock = e.download(), e.status()
            e.close()
            assert st[k]['steps'] == clock['steps'] and st[k]['dt'] == clock['dt'] and st[k]['t'] == clock['t'], k
            for f in FIELDS:
                np.testing.assert_array_equal(got[k][f], want[f], err_msg=f'instance {k} {f}')
        assert st[2]['steps'] == 1 and st[0]['steps'] == 5
    b.close()


@pytest.mark.parametrize('precision', ['fp64', 'fp32c'])
def test_one_large_among_many(precision):
    """The scan's workgroups by the tables: 60 small instances beside two large ones."""
    n = [200000] + [700] * 60 + [140000]
    say('one large among many', precision)
    cut = {k: _cut(k, 75, 0.3) for k in set(n)}
    params = {}
    for k, (sc, pA) in cut.items():
        params[k] = params_for(sc, 0.02, precision=precision, cell_capacity=0 if k > 700 else 4000)
        params[k].n = k
    b = BatchEngine([params[k] for k in n], device='cuda:0')
    b.upload([soa_from_particles(cut[k][1]) for k in n])
    b.step(4)
    got = b.download()
    b.close()
    for k, (sc, pA) in cut.items():
        m = sc.method()
        m.alpha = 0.02
        e = make_engine(pA, m, precision=precision)
        e.step(4)
        want = e.download()
        e.close()
        for j in np.nonzero(np.array(n) == k)[0]:
            for f in FIELDS:
                np.testing.assert_array_equal(got[j][f], want[f], err_msg=f'instance {j} {f}')
