"""State in and out of the engine where parts of it are not in memory.

After an upload the start-of-step values x0 ... rho0 are the state itself and
are written only when something needs them, and fields that hold one value (m,
h, an XSPH velocity nobody gave) are not read from the device's buffers on the
way out. Each against what the stored values would give, FP64:
  * a corrector straight after an upload, with and without a neighbour update
    and a host scatter between (PEC.correct from x0 = the uploaded state,
    src/Integrators/PEC.py:61-89);
  * states without any fluid, with wall masses of their own, and with an XSPH
    velocity given.
"""
import numpy as np
import pytest

from gpu_util import make_engine, perturbed, say
from hipsph import scenarios

pytestmark = pytest.mark.gpu


def _state(seed=41):
    sc = scenarios.dam_break(0.4, 0.5, 0.02, tank_w=1.0, tank_h=0.8, name='io')
    return perturbed(sc.pA, seed), sc.method()


@pytest.mark.parametrize('integrator', ['pec', 'euler'])
@pytest.mark.parametrize('between', ['', 'update', 'scatter', 'scatter+update', 'update+scatter'])
def test_corrector_after_upload(between, integrator):
    pA, m = _state()
    f = pA['label'] == 0
    pA['ax'][f], pA['ay'][f], pA['drho'][f] = 3.0, -2.0, 40.0
    say('corrector after upload', between, integrator)
    e = make_engine(pA, m, integrator=integrator, fixed_dt=1e-3, damping=0.1)
    e.dt()
    x = {k: pA[k].copy() for k in ('x', 'y', 'vx', 'vy', 'rho')}
    moved = {k: v.copy() for k, v in x.items()}
    for what in between.split('+'):
        if what == 'update':
            e.nn_update()
        elif what == 'scatter':
            ids = np.nonzero(f)[0][:50]
            for k in ('x', 'vx'):
                moved[k][ids] += 0.01
            e.scatter(ids, {k: moved[k][ids] for k in ('x', 'vx')})
    e.correct()
    d = e.download()
    e.close()
    dt, e1 = 1e-3, 1 + 0.5 * 0.1
    for a, v, r in (('x', 'vx', 'ax'), ('y', 'vy', 'ay')):
        acc = pA[r][f]
        if integrator == 'pec':  # from the uploaded start, moved by the velocity the state holds now
            want_x = 2 * (x[a][f] + 0.5 * dt * moved[v][f]) - x[a][f]
            want_v = 2 * ((x[v][f] + 0.5 * dt * acc) / e1) - x[v][f]
        else:
            want_x = moved[a][f] + dt * moved[v][f] + 0.5 * dt * dt * acc
            want_v = moved[v][f] + dt * acc
        np.testing.assert_array_equal(d[a][f], want_x, err_msg=a)
        np.testing.assert_array_equal(d[v][f], want_v, err_msg=v)


@pytest.mark.parametrize('case', ['plain', 'no_fluid', 'wall_mass', 'xsph_given', 'mixed_h'])
def test_download_gives_the_upload_back(case):
    pA, m = _state()
    f = pA['label'] == 0
    if case == 'no_fluid':
        pA = pA[~f].copy()
    elif case == 'wall_mass':
        pA['m'][~f] = 7.0
    elif case == 'xsph_given':
        pA['xsphx'], pA['xsphy'] = np.arange(len(pA)), -np.arange(len(pA))
    elif case == 'mixed_h':
        pA['h'][::3] *= 1.1
    say('upload and download', case)
    e = make_engine(pA, m)
    e.nn_update()
    d = e.download()
    e.close()
    for k in ('x', 'y', 'vx', 'vy', 'rho', 'ax', 'ay', 'drho', 'm', 'h', 'label'):
        np.testing.assert_array_equal(d[k], pA[k], err_msg=k)
    w = pA['label'] != 0  # without XSPH the fluid's reads as 0 once it has been sorted
    for k in ('xsphx', 'xsphy'):
        np.testing.assert_array_equal(d[k][w], pA[k][w], err_msg=k)
        assert np.all(d[k][~w] == 0.0)
