"""The pressure probe with a wavefront and with a thread per point: the same
bits for the same points on both sides of the limit (65,536 points), for each
kernel, in cells of fewer and of more than a wavefront's candidates, and for
points outside the grid.
"""
import numpy as np
import pytest

from gpu_util import make_engine, perturbed, say
from hipsph import scenarios

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('crowded', [False, True])
@pytest.mark.parametrize('kernel', ['cubic', 'wendland', 'gaussian'])
def test_forms_give_the_same_bits(kernel, crowded):
    sc = scenarios.dam_break(0.5, 0.5, 0.02, tank_w=1.0, tank_h=0.8, name='probe_forms')
    pA = perturbed(sc.pA, 71)
    if crowded:
        pA['h'][pA['label'] == 0] *= 3.0
        pA['h'][pA['label'] != 0] *= 3.0
    e = make_engine(pA, sc.method(), kernel=kernel)
    e.nn_update()
    rng = np.random.default_rng(72)
    n = 65537
    x, y = rng.uniform(-0.2, 1.2, n), rng.uniform(-0.2, 1.0, n)
    x[:3], y[:3] = (1e12, -1e12, 0.25), (0.1, 0.1, np.nan)
    h = rng.uniform(0.5, 1.5, n) * pA['h'][0]
    say('probe forms', kernel, crowded)
    many = e.probe_pressure(x, y, h)
    few = e.probe_pressure(x[:-1], y[:-1], h[:-1])
    one = e.probe_pressure(x[-1:], y[-1:], h[-1:])
    e.close()
    for a, b, c in zip(many, few, one):
        np.testing.assert_array_equal(a[:-1], b)
        np.testing.assert_array_equal(a[-1:], c)
    assert np.isfinite(many[0]).any()
