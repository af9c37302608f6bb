"""Bins of more particles than the neighbour update lists, FP64, bit for bit
against the CPU oracle, in every form of the update: grids of so many cells that
the fewest indices are listed of each (16), grids of few cells (256), both
sides of the limits between the forms (57,344 and 114,688 particles), and
capacities above 2^20 cells, where the scan, the places and the reorder are
kernels of their own.
"""
import numpy as np
import pytest

from gpu_util import make_engine, oracle_loop, perturbed, say
from hipsph import scenarios

pytestmark = pytest.mark.gpu


def _check(pA, m, capacity, seed):
    pA = pA[np.random.default_rng(seed).permutation(len(pA))]
    say('crowded bins', len(pA), capacity)
    want, _ = oracle_loop(pA, m)
    e = make_engine(pA, m, cell_capacity=capacity)
    for k in range(2):  # from the given order, then from the cell order
        e.nn_update()
        e.compute()
        got = e.download()
        for f in ('drho', 'ax', 'ay'):
            np.testing.assert_array_equal(got[f], want[f], err_msg=f'update {k} {f}')
    e.close()


@pytest.mark.parametrize('dx', [0.3, 0.2, 0.1, 0.05])
@pytest.mark.parametrize('far,capacity', [(False, 0), (False, (1 << 20) + 1), (True, 210000), (True, 1 << 20),
                                          (True, (1 << 20) + 1)])
def test_cells_of_one_metre(dx, far, capacity):
    """A wall particle without h: cells of 1 m, of about 11 to 400 particles;
    far: another one 1,000 m to the right and 200 m up, 203,000 cells."""
    sc = scenarios.dam_break(1.5, 1.5, dx, tank_w=2.0, tank_h=2.0, name='crowded')
    pA = perturbed(sc.pA, 61)
    pA['h'][-1] = 0.0
    if far:
        pA['x'][-2] += 1000.0
        pA['y'][-2] += 200.0
    _check(pA, sc.method(), capacity, 62)


@pytest.mark.parametrize('far', [False, True])
@pytest.mark.parametrize('n', [57344, 57345, 114688, 114689])
def test_one_crowded_cell(n, far):
    """One cell of 400 particles in a dam break; far: a wall particle so far
    away that the grid has about 4 cells per particle."""
    sc = scenarios.dam_break(1.0, 2.0, float(np.sqrt(2.0 / n)), name='wide')
    pA = perturbed(sc.pA, 63)
    pA = pA[np.sort(np.random.default_rng(64).permutation(len(pA))[:n])]
    f = np.nonzero(pA['label'] == 0)[0][:400]
    pA['x'][f] = 0.31 + 1e-5 * np.arange(400)  # 400 particles in one cell
    pA['y'][f] = 0.47 + 1e-5 * (np.arange(400) % 20)
    if far:
        cs = 2.0 * pA['h'].min()
        pA['x'][np.nonzero(pA['label'] != 0)[0][-1]] += 4 * n / np.ceil(np.ptp(pA['y']) / cs) * cs
    _check(pA, sc.method(), 0, 65)
