"""The neighbour update's cell order at its edges, FP64, against the CPU oracle.

The double pair pass sums in the order of the cell lists, so its rates are
bit-identical to the oracle's only if every cell's particles are in the order
of their index: particles given in random order (every cell filled by many
runs), cells of hundreds of particles (longer than a wavefront), a sparse
domain of many more cells than particles, and particle counts on both sides
of the one-kernel scan's limit (65,536).
"""
import numpy as np
import pytest

from gpu_util import make_engine, oracle_loop, perturbed, say
from hipsph import scenarios

pytestmark = pytest.mark.gpu


def _dam(n_fluid):
    return scenarios.dam_break(1.0, 2.0, float(np.sqrt(2.0 / n_fluid)), name='order')


def _dense():
    """One wall particle without h: cells of 1 m, about 400 particles each."""
    sc = scenarios.dam_break(1.5, 1.5, 0.05, tank_w=2.0, tank_h=2.0, name='dense')
    sc.pA['h'][-1] = 0.0
    return sc


def _sparse():
    """The walls' last column far away: hundreds of thousands of empty cells."""
    sc = scenarios.dam_break(0.4, 0.5, 0.02, tank_w=1.0, tank_h=0.8, name='sparse')
    sc.pA['x'][-40:] += 500.0
    return sc


@pytest.mark.parametrize('case', ['dam_5k', 'dense', 'sparse', 'below', 'above'])
def test_cell_order_fp64_bitexact(case):
    sc = {'dam_5k': lambda: _dam(5000), 'dense': _dense, 'sparse': _sparse, 'below': lambda: _dam(57000),
          'above': lambda: _dam(62000)}[case]()
    pA = perturbed(sc.pA, 21)
    pA = pA[np.random.default_rng(22).permutation(len(pA))]
    say('cell order', case, 'n', len(pA))
    if case in ('below', 'above'):
        assert (len(pA) <= 65536) == (case == 'below')
    m = sc.method()
    want, _ = oracle_loop(pA, m)
    e = make_engine(pA, m, cell_capacity=1 << 18)  # the sparse grid has 190,000 cells
    for _ in range(2):  # from the given order, then from the cell order
        e.nn_update()
        e.compute()
        got = e.download()
        for k in ('drho', 'ax', 'ay'):
            np.testing.assert_array_equal(got[k], want[k], err_msg=f'{case} {k}')
    e.close()
