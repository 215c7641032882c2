"""Which image of a bead a query takes: the from-scratch energy, the pressure
sample and the device loop against the oracle where the choice shows.

Tolerances: 1e-10 of max(|term|, 0.01 kT) as in test_gpu_record.py; the
pressure sample 1e-14 of the summed energies as in test_gpu_pressure.py, the
LJ sentinels of coincident pairs (1e8 each, equal on both sides of the
stretch) left out of the sum.
"""
import numpy as np
import pytest

from oracle import oracle as O
from plum_amd import engine as E
from plum_amd import systems
from test_gpu_record import record_run, replay

pytestmark = pytest.mark.gpu


def _full_matches(eng, orc, rel=1e-10):
    got, ref = eng.energy_full(), orc.energy_full()
    for k in E.TERMS:
        assert abs(got[k] - ref[k]) <= rel * max(abs(ref[k]), 1e-2), (k, got[k], ref[k])
    return ref


def _vp_matches(eng, orc, scale):
    got, ref = eng.vp_sample(), orc.vp_sample(0)
    for k in ("el", "lj", "wall", "bond", "dU"):
        assert abs(got[k] - ref[k]) <= 1e-14 * scale, (k, got[k], ref[k], scale)


@pytest.mark.parametrize("cell_div", [1, 2])
@pytest.mark.parametrize("precision", [E.PLUM_FP64, E.PLUM_FP32_PAIR])
def test_coincident_beads(cell_div, precision):
    """Ions put exactly on chain beads, the chains around the box origin: such
    a pair is at distance 0 to the bit whatever the cells and images it is met
    in, so it has the LJ sentinel 1e8 and no real-space term, in the totals, in
    the stretch of a pressure sample and in the dE of the moves that separate
    it."""
    L = 12.0
    sd = systems.config("tiny")
    xyz, q, ty, ms = systems.build_bulk(4, 10, 44, L, 17)
    rng = np.random.default_rng(2)
    for c in range(4):
        a, b = ms[c], ms[c + 1]
        xyz[a:b] += rng.uniform(-0.4, 0.4, 3) - xyz[a + c]   # bead c of chain c next to the origin
    pairs = [(int(ms[c]) + k, int(ms[4 + 10 * c + k])) for c in range(4) for k in range(10)]
    for chain_bead, ion in pairs:
        xyz[ion] = xyz[chain_bead]
    sd.update(xyz=xyz, q=q, type=ty, mol_start=ms, box=[L, L, L], alpha=0.2,
              move_prob=[0.4, 0.2, 0.2, 0.1, 0.1])
    orc = O.Oracle(sd)
    eng = E.Engine(sd, precision=precision, cell_div=cell_div)
    ref = _full_matches(eng, orc)
    assert ref["lj"] >= 40e8
    _full_matches(eng, orc)
    _vp_matches(eng, orc, sum(abs(v) for k, v in ref.items() if k != "lj") + ref["lj"] % 1e8)
    eng.close()
    if precision == E.PLUM_FP64:
        _, st, recs, _ = record_run(sd, 200, 16, seed=3)
        assert sum(r["dE"]["lj"] < -0.9e8 for r in recs) >= 5
        # a move within a chain cancels up to ten sentinels, 1e8 each rounded
        # to 1.5e-8 in both sums: 3e-7 at most, 1e-10 of a floor of 1e4
        replay(sd, recs, 1e-10, floor=1e4)
