"""The neighbour update of small states (offsets, places and reorder in one
kernel) at its edges, FP64, against the CPU oracle bit for bit: particle
counts on both sides of its two forms' limits, one particle more than whole
workgroups, cells of more particles than k_keys lists, in index order and not,
and cell capacities that leave the kernel out or list the fewest members.
"""
import numpy as np
import pytest

from gpu_util import make_engine, oracle_loop, perturbed, say
from hipsph import scenarios

pytestmark = pytest.mark.gpu

FIELDS = ('drho', 'ax', 'ay')


def _check(pA, m, **kw):
    want, _ = oracle_loop(pA, m)
    e = make_engine(pA, m, **kw)
    for k in range(2):  # from the given order, then from the cell order
        e.nn_update()
        e.compute()
        got = e.download()
        for f in FIELDS:
            np.testing.assert_array_equal(got[f], want[f], err_msg=f'update {k} {f}')
    e.close()


@pytest.mark.parametrize('n', [257, 57344, 57345, 114688, 114689])
def test_particle_counts(n):
    sc = scenarios.dam_break(1.0, 2.0, float(np.sqrt(2.0 / n)), name='counts')
    pA = perturbed(sc.pA, 31)
    assert len(pA) >= n
    pA = pA[np.sort(np.random.default_rng(32).permutation(len(pA))[:n])]
    pA = pA[np.random.default_rng(33).permutation(n)]
    say('reorder scan', n)
    _check(pA, sc.method())


@pytest.mark.parametrize('dx,capacity', [(0.1, 0), (0.05, 0), (0.1, 1 << 20), (0.015, 1 << 20)])
def test_crowded_cells(dx, capacity):
    """One wall particle without h: cells of 1 m, of about 100, 400 or 4,400
    particles; 256 are listed per bin, 32 with the largest capacity."""
    sc = scenarios.dam_break(1.5, 1.5, dx, tank_w=2.0, tank_h=2.0, name='crowded')
    pA = perturbed(sc.pA, 34)
    pA['h'][-1] = 0.0
    pA = pA[np.random.default_rng(35).permutation(len(pA))]
    say('crowded', dx, capacity, len(pA))
    _check(pA, sc.method(), cell_capacity=capacity)


def test_capacity_beyond_the_kernel():
    sc = scenarios.dam_break(0.5, 0.5, 0.02, tank_w=1.0, tank_h=0.8, name='beyond')
    pA = perturbed(sc.pA, 36)
    _check(pA[np.random.default_rng(37).permutation(len(pA))], sc.method(), cell_capacity=(1 << 20) + 1)
