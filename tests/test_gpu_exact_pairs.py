"""FP64 pair terms at the ends of the range their roots and quotients are
formed in without scaling (1e-100 < h < 1e100), and beyond it, where the
general pass takes over: lengths scaled by powers of two, bit for bit against
the CPU oracle, in the lane-group pass and (more particles) the thread-per-target pass.
"""
import numpy as np
import pytest

from gpu_util import make_engine, oracle_loop, perturbed, say
from hipsph import scenarios

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('n_fluid', [1500, 70000])
@pytest.mark.parametrize('power', [0, 40, -40, 200, -200, -340])
def test_scaled_lengths(power, n_fluid):
    sc = scenarios.dam_break(1.0, 1.0, float(np.sqrt(1.0 / n_fluid)), tank_w=2.0, tank_h=1.2, name='scaled')
    pA = perturbed(sc.pA, 81)
    m = sc.method()
    s = 2.0 ** power
    for f in ('x', 'y', 'h'):
        pA[f] = pA[f] * s
    m.r0 = m.r0 * s
    say('scaled lengths', power, len(pA))
    want, _ = oracle_loop(pA, m)
    e = make_engine(pA, m)
    assert e.pair_form() == ('fp64-uniform' if power > -330 else 'fp64')
    e.nn_update()
    e.compute()
    got = e.download()
    e.close()
    for k in ('drho', 'ax', 'ay'):
        np.testing.assert_array_equal(got[k], want[k], err_msg=k)
