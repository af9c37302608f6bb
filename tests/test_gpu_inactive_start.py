"""PEC's start-of-step values x0 ... rho0 through steps and predictors that do
not run (the clock is past the duration): a corrector after them starts from
the values that were there before (PEC.correct, src/Integrators/PEC.py:61-89),
which are the uploaded state, in memory (a scatter wrote them) or not.
"""
import numpy as np
import pytest

from gpu_util import make_engine, perturbed, say
from hipsph import scenarios

pytestmark = pytest.mark.gpu

IDLE = {'step': lambda e: e.step(1), 'steps': lambda e: e.step(2), 'update': lambda e: (e.dt(), e.nn_update()),
        'split step': lambda e: (e.step_begin(), e.step_end()), 'predict': lambda e: (e.dt(), e.predict())}


@pytest.mark.parametrize('n_fluid', [500, 120000])  # both forms of the reorder
@pytest.mark.parametrize('scatter', [False, True])
@pytest.mark.parametrize('idle', list(IDLE))
def test_corrector_after_a_step_that_does_not_run(idle, scatter, n_fluid):
    sc = scenarios.dam_break(0.5, 1.0, float(np.sqrt(0.5 / n_fluid)), tank_w=1.0, tank_h=1.2, name='idle')
    pA, m = perturbed(sc.pA, 51), sc.method()
    f = pA['label'] == 0
    pA['ax'][f], pA['ay'][f], pA['drho'][f] = 3.0, -2.0, 40.0
    say('idle', idle, scatter, len(pA))
    e = make_engine(pA, m, fixed_dt=1e-3, damping=0.1, duration=1.0)
    x0 = {k: pA[k].copy() for k in ('x', 'y', 'vx', 'vy', 'rho')}
    now = {k: v.copy() for k, v in x0.items()}
    if scatter:
        ids = np.nonzero(f)[0][:50]
        for k in ('x', 'vx'):
            now[k][ids] += 0.01
        e.scatter(ids, {k: now[k][ids] for k in ('x', 'vx')})
    e.set_clock(2.0)
    IDLE[idle](e)
    d = e.download()
    for k in x0:
        np.testing.assert_array_equal(d[k], now[k], err_msg=f'idle {k}')
    e.set_clock(0.0)
    e.dt()
    e.correct()
    d = e.download()
    e.close()
    dt, e1 = 1e-3, 1 + 0.5 * 0.1
    for a, v, r in (('x', 'vx', 'ax'), ('y', 'vy', 'ay')):  # moved by the velocity the state holds now
        np.testing.assert_array_equal(d[a][f], 2 * (x0[a][f] + 0.5 * dt * now[v][f]) - x0[a][f], err_msg=a)
        np.testing.assert_array_equal(d[v][f], 2 * ((x0[v][f] + 0.5 * dt * pA[r][f]) / e1) - x0[v][f], err_msg=v)
    rho = 2 * (x0['rho'][f] + 0.5 * dt * pA['drho'][f]) - x0['rho'][f]
    np.testing.assert_array_equal(d['rho'][f], rho, err_msg='rho')
