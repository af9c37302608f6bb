"""FP64 pair terms whose operands lie at the ends of the exponent range, in the
lane-group pass and (more particles) the thread-per-target pass, bit for bit
against the general pass, and against the CPU oracle where the rates are finite
(it also adds pairs outside the support, whose zero gradient times an infinite
viscosity is no number): positions moved off the lattice, so that every operand
has a mantissa of its own, and velocities scaled so that the viscosity's
numerators h v.r and quotients reach the subnormal numbers, or overflow. The
density is the reference one, so no pressure hides the viscosity. Then the
lengths up to which Wendland's quotients are formed in this way.
"""
import numpy as np
import pytest

from gpu_util import make_engine, oracle_loop, perturbed, say
from hipsph import scenarios

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('n_fluid', [1500, 70000])
@pytest.mark.parametrize('kernel', ['cubic', 'wendland'])
@pytest.mark.parametrize('power', [0, -300, -480, -930, -970, -1000, -1030, -1060, 300, 480, 930, 1000])
def test_scaled_velocities(power, kernel, n_fluid):
    sc = scenarios.dam_break(1.0, 1.0, float(np.sqrt(1.0 / n_fluid)), tank_w=2.0, tank_h=1.2, name='ends')
    pA = perturbed(sc.pA, 91, rscale=0.0)
    f = pA['label'] == 0
    rng = np.random.default_rng(92)
    for k in ('x', 'y'):
        pA[k][f] += rng.uniform(-0.1, 0.1, f.sum()) * sc.dx
    for k in ('vx', 'vy'):
        pA[k][f] = np.ldexp(pA[k][f], power)
    m = sc.method()
    m.beta = 0.3
    pA['rho'][f] = m.rho0
    assert m.Pb == 0.0
    say('scaled velocities', power, kernel, len(pA))
    e = make_engine(pA, m, kernel=kernel)
    assert e.pair_form() == 'fp64-uniform'
    e.nn_update()
    e.compute()
    got = e.download()
    e.compute_counts()  # by the general pass
    want = e.download()
    e.close()
    for k in ('drho', 'ax', 'ay'):
        np.testing.assert_array_equal(got[k], want[k], err_msg=k)
    if power <= 480:
        want, _ = oracle_loop(pA, m, kernel)
        for k in ('drho', 'ax', 'ay'):
            np.testing.assert_array_equal(got[k], want[k], err_msg=k)


@pytest.mark.parametrize('power,form', [(-200, 'fp64-uniform'), (180, 'fp64-uniform'), (200, 'fp64')])
def test_wendland_lengths(power, form):
    sc = scenarios.dam_break(1.0, 1.0, float(np.sqrt(1.0 / 1500)), tank_w=2.0, tank_h=1.2, name='lengths')
    pA = perturbed(sc.pA, 93)
    m = sc.method()
    for f in ('x', 'y', 'h'):
        pA[f] = np.ldexp(pA[f], power)
    m.r0 = float(np.ldexp(m.r0, power))
    say('scaled lengths', power, len(pA))
    want, _ = oracle_loop(pA, m, 'wendland')
    e = make_engine(pA, m, kernel='wendland')
    assert e.pair_form() == form
    e.nn_update()
    e.compute()
    got = e.download()
    e.close()
    for k in ('drho', 'ax', 'ay'):
        np.testing.assert_array_equal(got[k], want[k], err_msg=k)
