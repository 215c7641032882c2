"""Edges of the engine's kernels against the CPU oracle: sizes at which a
tile, a remainder or an image range can go wrong.  Device-loop decisions are
replayed as in test_gpu_record.py; its tolerance (1e-10 of max(|dE|, 0.01
kT)) is used unless a test derives its own.
"""
import numpy as np
import pytest

from oracle import oracle as O
from plum_amd import engine as E
from plum_amd import systems
from test_gpu_record import record_run, replay

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("L,alpha,cells", [(8.0, 0.39, 1), (7.0, 0.12, 2), (6.5, 0.05, 3)])
def test_pair_images_when_the_cutoff_passes_the_box(L, alpha, cells):
    """Explicit pair sums (moved-moved and cross terms) where 2 rc > L, up to
    three image shells: only the offsets within rc are visited."""
    sd = systems.config("tiny")
    xyz, q, ty, ms = systems.build_bulk(2, 5, 10, L, 11)
    sd.update(xyz=xyz, q=q, type=ty, mol_start=ms, box=[L, L, L], alpha=alpha)
    eng, _, recs, _ = record_run(sd, 300, 16, seed=5)
    assert max(eng.info().real_cell) == cells
    replay(sd, recs, 1e-10)
    # beads exactly half an edge apart: either image is the minimum one
    a, b = ms[0], ms[1]
    x = eng.positions()[a:b]
    new = x.copy()
    new[1:] = x[:1] + np.array([0.5 * L, 0.0, 0.0]) + 0.9 * np.arange(1, b - a)[:, None] * [0.0, 0.0, 1.0]
    new[1] = x[0] + [0.5 * L, 0.5 * L, 0.0]
    orc = O.Oracle(dict(sd, xyz=eng.positions()))
    idx = np.arange(a, b, dtype=np.int32)
    orc.set_trial(0, idx, new)
    t_ref, d_ref = orc.delta(0)
    t, d = eng.delta(0, idx, new)
    eng.finalize(False)
    for k in E.TERMS:
        assert abs(d[k] - d_ref[k]) <= 1e-10 * max(abs(d_ref[k]), 1e-2), (k, d[k], d_ref[k])
