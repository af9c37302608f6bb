"""The FP64 Gaussian where the smoothing length is not positive: the
reference's gradient is zero unless r h > 1e-12 (src/Kernels/Gaussian.py:39-60),
so such pairs add nothing.
"""
import numpy as np
import pytest

from gpu_util import make_engine, oracle_loop, perturbed, say
from hipsph import scenarios

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('p1', [4.0, 4.5])  # lane groups, a thread per target
@pytest.mark.parametrize('which', ['all', 'some'])
def test_negative_lengths(which, p1):
    sc = scenarios.dam_break(1.0, 1.0, 0.05, tank_w=2.0, tank_h=1.2, name='negative')
    pA = perturbed(sc.pA, 93)
    pA['h'][::1 if which == 'all' else 50] *= -1.0
    m = sc.method()
    m.p1 = p1
    say('negative lengths', which, p1, len(pA))
    want, _ = oracle_loop(pA, m, 'gaussian')
    e = make_engine(pA, m, kernel='gaussian')
    e.nn_update()
    e.compute()
    got = e.download()
    e.close()
    for k in ('drho', 'ax', 'ay'):
        scale = np.max(np.abs(want[k]))
        np.testing.assert_allclose(got[k], want[k], rtol=0.0, atol=1e-12 * max(scale, 1.0), err_msg=k)
