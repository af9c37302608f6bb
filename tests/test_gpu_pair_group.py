"""The pair passes with several lanes per target, at each lane count.

Below a size that depends on the form, 16, 8 or 4 lanes share a target
(16 up to 16,384 particles, 8 up to 32,768, 4 above); their sums keep the
order of the one-thread passes, so the results are the same bits:
  * FP64, uniform (one h, one fluid mass) and general (two masses): the rates
    of one loop bit-identical to the CPU oracle (the Gaussian, whose exp is
    another library's, within 1e-12);
  * FP32C: the general pass bit-identical to its one-thread form (the pass
    that reports neighbour counts); the uniform pass within 2e-6 of it (the
    general pass sums in float with TwoSum, the uniform one in double);
  * h = 3 dx: about 110 contributors per target, more than a list holds;
  * above the limits, the float pass staged in LDS against the same pass
    reading global memory, with workgroups too large for the stage.
"""
import numpy as np
import pytest

from gpu_util import make_engine, oracle_loop, perturbed, rel_err, say
from hipsph import scenarios

pytestmark = pytest.mark.gpu

RATES = ('drho', 'ax', 'ay')


def _state(n_fluid, uniform, seed):
    sc = scenarios.dam_break(1.0, 2.0, float(np.sqrt(2.0 / n_fluid)), name='group')
    pA = perturbed(sc.pA, seed)
    if not uniform:
        pA['m'][:: 2] *= 1.01
    return pA, sc.method()


@pytest.mark.parametrize('n_fluid', [7000, 20000, 36000])
@pytest.mark.parametrize('uniform', [True, False])
@pytest.mark.parametrize('kernel', ['cubic', 'gaussian', 'wendland'])
def test_group_pass_fp64(kernel, uniform, n_fluid):
    pA, m = _state(n_fluid, uniform, 31)
    say('group fp64', kernel, uniform, len(pA))
    want, _ = oracle_loop(pA, m, kernel)
    e = make_engine(pA, m, kernel=kernel)
    e.nn_update()
    assert e.pair_form() == ('fp64-uniform' if uniform else 'fp64')
    e.compute()
    got = e.download()
    e.nn_update()
    e.continuity()
    e.momentum()
    split = e.download()
    e.close()
    f = pA['label'] == 0
    for k in RATES:
        np.testing.assert_array_equal(split[k], got[k], err_msg=k)
        if kernel == 'gaussian':
            assert rel_err(got[k], want[k], f) < 1e-12, k
        else:
            np.testing.assert_array_equal(got[k], want[k], err_msg=k)


@pytest.mark.parametrize('n_fluid', [7000, 20000, 36000])
@pytest.mark.parametrize('uniform', [True, False])
@pytest.mark.parametrize('kernel', ['cubic', 'gaussian', 'wendland'])
def test_group_pass_fp32c(kernel, uniform, n_fluid):
    pA, m = _state(n_fluid, uniform, 32)
    say('group fp32c', kernel, uniform, len(pA))
    e = make_engine(pA, m, kernel=kernel, precision='fp32c')
    e.nn_update()
    e.compute()
    got = e.download()
    e.compute_counts()
    one = e.download()
    e.close()
    f = pA['label'] == 0
    for k in RATES:
        if uniform:
            assert rel_err(got[k], one[k], f) < 2e-6, k
        else:
            np.testing.assert_array_equal(got[k], one[k], err_msg=k)


@pytest.mark.parametrize('precision', ['fp64', 'fp32c'])
def test_group_lists_that_fill(precision):
    sc = scenarios.stress_lattice(nside=160, hfac=3.0)
    pA = sc.pA.copy()
    if precision == 'fp32c':
        pA['m'][::2] *= 1.01  # the general pass, bit-identical to its one-thread form
    say('group lists', precision, len(pA))
    e = make_engine(pA, sc.method(), precision=precision)
    e.nn_update()
    e.compute()
    got = e.download()
    e.compute_counts()
    one = e.download()
    e.close()
    f = pA['label'] == 0
    for k in RATES:
        np.testing.assert_array_equal(got[k][f], one[k][f], err_msg=k)


def test_staged_walk_above_the_group_sizes():
    sc = scenarios.stress_lattice(nside=340, hfac=3.0)
    out = []
    for staging in (True, False):
        say('staged walk', len(sc.pA), staging)
        e = make_engine(sc.pA, sc.method(), precision='fp32c')
        assert e.pair_form() == 'fp32c-uniform'
        e.set_pair_staging(staging)
        e.step(10)
        out.append(e.download())
        e.close()
    for k in RATES + ('x', 'y', 'vx', 'vy', 'rho'):
        np.testing.assert_array_equal(out[0][k], out[1][k], err_msg=k)
