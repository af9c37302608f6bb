"""A batch whose instances end at different times, against single engines.

Instances that reach their duration, or halt, stay where they are while the
others go on: their particles keep their places (nothing sorts them) and their
states come back as they were when they stopped, bit for bit the state of an
engine of their own. Sizes from a thousand to 12,000 particles, in uneven order.
"""
import numpy as np
import pytest

from gpu_util import FIELDS, make_engine, perturbed, say
from hipsph import scenarios
from hipsph.batch import BatchEngine, params_for
from hipsph.device import soa_from_particles

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('precision', ['fp64', 'fp32c'])
@pytest.mark.parametrize('uniform', [True, False])
def test_instances_that_stop(uniform, precision):
    scs = [scenarios.dam_break(w, h, dx, tank_w=1.5, tank_h=1.2, name=f'stop_{k}')
           for k, (w, h, dx) in enumerate([(0.4, 0.3, 0.02), (1.0, 1.0, 0.0095), (0.5, 0.4, 0.015), (0.7, 0.9, 0.03)])]
    pAs = [perturbed(s.pA, 50 + k) for k, s in enumerate(scs)]
    if not uniform:
        pAs[1]['m'][::2] *= 1.01
    steps = [40, 9, 0, 23]
    params, want = [], []
    for s, pA, n in zip(scs, pAs, steps):
        m = s.method()
        e = make_engine(pA, m, precision=precision)
        e.step(40)
        t = np.cumsum(e.dt_history(40)[:, 0])
        e.close()
        # the step that would start at or after the duration does not run
        duration = 0.0 if n == 0 else (t[n - 1] + t[n - 2]) / 2 if n < 40 else np.inf
        e = make_engine(pA, m, precision=precision, duration=duration)
        e.step(40)
        assert e.status()['steps'] == n
        want.append(e.download())
        e.close()
        params.append(params_for(s, precision=precision, duration=duration))
    say('batch with finished instances', uniform, precision, [s.n for s in scs])
    b = BatchEngine(params)
    b.upload([soa_from_particles(pA) for pA in pAs])
    b.step(40)
    got, st = b.download(), b.status()
    assert [s['steps'] for s in st] == steps
    b.close()
    for k in range(len(scs)):
        for f in FIELDS:
            if precision == 'fp64' or uniform:
                np.testing.assert_array_equal(got[k][f], want[k][f], err_msg=f'{k} {f}')
            else:  # a mixed batch runs the general float pass, an engine of one mass the uniform one
                scale = np.max(np.abs(want[k][f])) or 1.0
                assert np.max(np.abs(got[k][f] - want[k][f])) <= 2e-4 * scale, (k, f)
