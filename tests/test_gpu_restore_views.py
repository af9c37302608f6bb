"""Engine.restore reads contiguous device tensors in place; what is stored
otherwise than it reads (a lazily negated view) is copied first."""
import numpy as np
import pytest
import torch

from gpu_util import make_engine, perturbed, say
from hipsph import scenarios

pytestmark = pytest.mark.gpu


def test_restore_of_a_negated_view():
    sc = scenarios.dam_break(0.4, 0.5, 0.02, tank_w=1.0, tank_h=0.8, name='views')
    pA = perturbed(sc.pA, 71)
    e = make_engine(pA, sc.method())
    st = e.download(to_numpy=False)
    st['vx'] = torch._neg_view(st['vx'])
    assert st['vx'].is_contiguous()
    say('negated view', len(pA))
    e.restore(st, 0.0)
    got = e.download()
    e.close()
    np.testing.assert_array_equal(got['vx'], -pA['vx'])
    np.testing.assert_array_equal(got['vy'], pA['vy'])
