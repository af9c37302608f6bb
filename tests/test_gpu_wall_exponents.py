"""The wall force's exponents: whole numbers of 0 to 16 take passes without a
pow(), anything else the passes with it.

The Lennard-Jones force D ((r0 / r)^p1 - (r0 / r)^p2) / r^2
(src/Equations/BoundaryForce.py:31-41) of fluid pressed into the walls, in the
uniform and the general pass, with one and with several lanes per target and
in a batch, against the CPU oracle; whole exponents in FP64 bit for bit, the
others to 1e-12 (pow is another library's).
"""
import numpy as np
import pytest

from gpu_util import make_engine, oracle_loop, perturbed, rel_err, say
from hipsph import scenarios
from hipsph.batch import BatchEngine, params_for
from hipsph.device import soa_from_particles

pytestmark = pytest.mark.gpu

EXPONENTS = [(4, 2), (12, 6), (16, 1), (17, 2), (4.5, 2.5), (4, 2.5)]


def _state(n_fluid, uniform):
    sc = scenarios.dam_break(1.0, 1.0, float(np.sqrt(1.0 / n_fluid)), tank_w=2.0, tank_h=1.2, name='walls')
    pA = perturbed(sc.pA, 61)
    f = pA['label'] == 0
    pA['x'][f] -= 0.4 * sc.dx  # into the left wall
    pA['y'][f] -= 0.3 * sc.dx
    if not uniform:
        pA['m'][::2] *= 1.01
    return sc, pA


@pytest.mark.parametrize('n_fluid', [4000, 110000])
@pytest.mark.parametrize('uniform', [True, False])
@pytest.mark.parametrize('p1,p2', EXPONENTS)
def test_exponents_against_oracle(p1, p2, uniform, n_fluid):
    sc, pA = _state(n_fluid, uniform)
    m = sc.method()
    m.p1, m.p2 = p1, p2
    say('wall exponents', p1, p2, uniform, len(pA))
    want, _ = oracle_loop(pA, m)
    f = pA['label'] == 0
    for precision in ('fp64', 'fp32c'):
        e = make_engine(pA, m, precision=precision)
        e.nn_update()
        e.compute()
        got = e.download()
        e.close()
        for k in ('drho', 'ax', 'ay'):
            if precision == 'fp32c':
                assert rel_err(got[k], want[k], f) < 2e-5, k
            elif float(p1).is_integer() and float(p2).is_integer() and max(p1, p2) <= 16:
                np.testing.assert_array_equal(got[k], want[k], err_msg=k)
            else:
                assert rel_err(got[k], want[k], f) < 1e-12, k


@pytest.mark.parametrize('precision', ['fp64', 'fp32c'])
def test_batch_of_mixed_exponents(precision):
    """One instance with a broken exponent puts the batch on the passes with pow()."""
    sc, pA = _state(3000, True)
    out = []
    for exps in ([(4, 2), (12, 6)], [(4, 2), (12, 6), (4.5, 2)]):
        params = [params_for(sc, precision=precision) for _ in exps]
        for p, (p1, p2) in zip(params, exps):
            p.p1, p.p2 = p1, p2
        say('batch exponents', precision, exps)
        b = BatchEngine(params)
        b.upload([soa_from_particles(pA) for _ in exps])
        b.step(5)
        out.append(b.download())
        b.close()
    for k in range(2):
        for f in ('x', 'vx', 'rho', 'ax', 'ay', 'drho'):
            np.testing.assert_array_equal(out[0][k][f], out[1][k][f], err_msg=f'{k} {f}')
