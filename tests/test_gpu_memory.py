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


def test_training_workspace():
    """The FP32 forward allocates the rows and activations (3.3 KB a row, 652
    MiB), not the partials of a gradient (1.3 KB a row more if every chunk of 128
    rows had its own, 253 MiB); a gradient of as many rows then adds at most the
    21 MB of 128 chunks."""
    sd = systems.config("tiny")
    xyz, q, ty, ms = systems.build_bulk(1, 200, 0, 40.0, 3)
    sd.update(xyz=xyz, q=q * 0.0, type=ty, mol_start=ms, box=[40.0] * 3, alpha=0.05)
    eng = E.Engine(sd)
    eng.surrogate_enable(train_every=0, train_samples=1, ring=1, r_d=2.5, seed=3)
    samples, m = 512, eng.max_mol_len()
    rows = 2 * m * samples
    x = np.zeros((rows, 64), np.float32)
    before = _used()
    eng.surrogate_forward(x, bf16=False)
    mid = _used()
    assert mid - before < rows * (64 + 6 * 128 + 2) * 4 + 64 * MIB, (mid - before) / MIB
    eng.surrogate_gradient(x.reshape(samples, 2 * m, 64), np.zeros(samples), np.full(samples, m, np.int32))
    assert _used() - mid < 48 * MIB, (_used() - mid) / MIB
    eng.close()
