"""The staged walk of the uniform FP64 pair passes: the oracle's bits and the
unstaged walk's, for workgroups within the stage and beyond it (wider
smoothing lengths: more records per row range), the split passes, and particles
in random order (ranges of all slots).
"""
import numpy as np
import pytest

from gpu_util import make_engine, oracle_loop, perturbed, say
from hipsph import scenarios

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('kernel', ['cubic', 'wendland'])
@pytest.mark.parametrize('wide', [1.0, 2.0, 3.5])
def test_staged_walk(wide, kernel):
    sc = scenarios.dam_break(1.0, 1.0, float(np.sqrt(1.0 / 62000)), tank_w=2.0, tank_h=1.2, name='staged64')
    pA = perturbed(sc.pA, 91)
    pA['h'] = pA['h'] * wide
    pA = pA[np.random.default_rng(92).permutation(len(pA))]
    m = sc.method()
    say('staged fp64', kernel, wide, len(pA))
    want, _ = oracle_loop(pA, m, kernel=kernel)
    out = []
    for staging in (True, False):
        e = make_engine(pA, m, kernel=kernel)
        e.set_pair_staging(staging)
        assert e.pair_form() == 'fp64-uniform'
        e.nn_update()
        e.compute()
        got = e.download()
        for k in ('drho', 'ax', 'ay'):
            np.testing.assert_array_equal(got[k], want[k], err_msg=k)
        e.continuity()
        e.momentum()
        split = e.download()
        e.step(3)
        out.append((got, split, e.download()))
        e.close()
    for a, b in zip(*out):
        for k in a:
            np.testing.assert_array_equal(a[k], b[k], err_msg=k)
    for k in ('drho', 'ax', 'ay'):
        np.testing.assert_array_equal(out[0][0][k], out[0][1][k], err_msg='split ' + k)
