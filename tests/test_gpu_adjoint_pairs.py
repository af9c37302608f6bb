"""The reversed pair pass over its forms: each kernel, whole and fractional
wall exponents (the pass is built for both), and smoothing lengths whose
particles list fewer and more pairs than one fill of the pass's list holds.

The oracle is the central difference of the device's own forward, as in
test_gpu_adjoint.py, to its 1e-4 relative; the steps are chosen so that the
differences' truncation and rounding lie below that.
"""
import numpy as np
import pytest
import torch

from gpu_util import say
from hipsph import scenarios
from hipsph.adjoint import SPHRun

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('wide', [1.0, 1.7])
@pytest.mark.parametrize('exponents', ['whole', 'fractional'])
@pytest.mark.parametrize('kernel', ['cubic', 'wendland', 'gaussian'])
def test_reversed_pair_pass(kernel, exponents, wide):
    sc = scenarios.dam_break(0.3, 0.3, 0.02, tank_w=0.6, tank_h=0.5, name='adj_pairs')
    m = sc.method()
    if exponents == 'fractional':
        m.p1, m.p2 = 4.5, 2.25
    pA = sc.pA.copy()
    pA['h'] = pA['h'] * wide
    rng = np.random.default_rng(11)
    fluid = pA['label'] == 0
    nf = int(fluid.sum())
    # off the lattice: no two pairs share a distance, none sits on a kink
    pA['x'][fluid] += rng.uniform(-2e-3, 2e-3, nf)
    pA['y'][fluid] += rng.uniform(-2e-3, 2e-3, nf)
    v0 = torch.as_tensor(rng.normal(0, 0.3, (nf, 2)), device='cuda')
    run = SPHRun(pA, m, nsteps=3, checkpoint_every=2, kernel=kernel, fixed_dt=0.1 * sc.h / m.co)
    w = torch.as_tensor(rng.normal(0, 1, (nf, 2)), device='cuda')
    run.forward(m.alpha, m.co, v0)
    ga, gc, gv = run.backward(w)
    gv = gv.clone()

    def loss(a=m.alpha, c=m.co, v=v0):
        return float(torch.sum(w * run.forward(a, c, v, keep=False)))

    eps = 1e-6
    d = torch.as_tensor(rng.normal(0, 1, (nf, 2)), device='cuda')
    fd_v = (loss(v=v0 + eps * d) - loss(v=v0 - eps * d)) / (2 * eps)
    # alpha and c0 act on 3 short steps: larger steps keep the differences
    # above the loss's rounding (~1e-15). The loss is linear in alpha within one
    # step, so alpha's may be 1e-2: 1e-15 / (2 * 1e-2 * 0.01) = 5e-12 of ~1e-6.
    ea, e = 1e-2, 1e-4
    fd_a = (loss(a=m.alpha * (1 + ea)) - loss(a=m.alpha * (1 - ea))) / (2 * ea * m.alpha)
    fd_c = (loss(c=m.co * (1 + e)) - loss(c=m.co * (1 - e))) / (2 * e * m.co)
    say(kernel, exponents, wide, 'alpha', float(ga), fd_a, 'c0', float(gc), fd_c, 'v0', float((gv * d).sum()), fd_v)
    run.close()
    assert abs(float((gv * d).sum()) - fd_v) < 1e-4 * abs(fd_v)
    assert abs(float(ga) - fd_a) < 1e-4 * abs(fd_a)
    assert abs(float(gc) - fd_c) < 1e-4 * abs(fd_c)
