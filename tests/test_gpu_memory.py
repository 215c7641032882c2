"""Device memory that calls keep: buffers are allocated for the largest
request and reused.  hipMemGetInfo reports what the device has left, to the
allocator's granularity of some MiB, so the sizes are chosen far above it.
"""
import numpy as np
import pytest
import torch

from plum_amd import engine as E
from plum_amd import systems

pytestmark = pytest.mark.gpu
MIB = 1 << 20


def _used():
    torch.cuda.synchronize()
    free, total = torch.cuda.mem_get_info()
    return total - free


def test_growth_buffers_of_alternating_shapes():
    """Growths of two shapes in turn, each larger than the other in one way:
    the buffers hold both after the first of each (at 1,024 trials and 512 steps
    a set is 26 MiB)."""
    sd = systems.config("gc_small")
    Lb = sd["box"][0]
    eng = E.Engine(sd)
    rng = np.random.default_rng(7)

    def grow(K, L):
        v = rng.normal(size=(L, K, 3))
        v /= np.linalg.norm(v, axis=-1)[..., None]
        return eng.cbmc_grow(2, L, K, 0, -1.0, first=rng.uniform(0, Lb, (2, 3)), disp=v,
                             ions=rng.uniform(0, Lb, (L, K, 3)), sel=rng.uniform(0, 1, L), type_ion=1, q_ion=1.0)

    shapes = [(1024, 4), (8, 512), (1024, 512)]
    for s in shapes:
        grow(*s)
    before = _used()
    for _ in range(6):
        for s in shapes:
            grow(*s)
    assert _used() - before < 16 * MIB, (_used() - before) / MIB
    eng.close()
