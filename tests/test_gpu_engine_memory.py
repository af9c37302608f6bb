"""Device memory of small engines: a program may keep many of them."""
import pytest
import torch

from gpu_util import make_engine, say
from hipsph import scenarios

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('n_fluid', [500, 5000])
def test_small_engines_stay_small(n_fluid):
    """64 bytes per cell for the bins' members beside about 12 of the cell
    table, at 8 cells per particle and 65,536 more; 600 bytes per particle of
    state and 1.5 MB of dt history; 2 MB for the allocator's granularity."""
    sc = scenarios.dam_break(0.5, 1.0, (0.5 / n_fluid) ** 0.5, tank_w=1.0, tank_h=1.2, name='memory')
    n, count = len(sc.pA), 12
    make_engine(sc.pA, sc.method()).close()  # what the first engine of a process loads
    torch.cuda.synchronize()
    free0 = torch.cuda.mem_get_info()[0]
    keep = [make_engine(sc.pA, sc.method()) for _ in range(count)]
    torch.cuda.synchronize()
    per = (free0 - torch.cuda.mem_get_info()[0]) / count
    for e in keep:
        e.close()
    say('engine of', n, 'particles:', per / 2 ** 20, 'MiB')
    assert per < 80 * (8 * n + 65536) + 600 * n + 3.5e6
