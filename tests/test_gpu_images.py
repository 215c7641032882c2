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
from plum_amd import host, systems
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


def _slab(L, alpha, length, seed, dipole):
    """Chains and ions between two walls, beads of some chains at both."""
    sd = systems.config("slab_small")
    box = [12.0, 12.0, L]
    xyz, q, ty, ms = host.synth_system(6, length, 6 * length, 0, box, seed, npbc=2, z_range=(0.7, L - 0.7))
    # chain 0 straight up, from wall to wall
    a, b = int(ms[0]), int(ms[1])
    xyz[a:b] = [0.3, 0.4, 0.0] + np.linspace(0.7, L - 0.7, b - a)[:, None] * [0.0, 0.0, 1.0]
    sd.update(xyz=xyz, q=q, type=ty, mol_start=ms, box=box, alpha=alpha, dipole=dipole, grafted=0,
              move_prob=[0.2, 0.2, 0.2, 0.2, 0.2])
    return sd


@pytest.mark.parametrize("L,length,dipole", [(8.0, 9, 0), (8.0, 20, 0), (10.0, 11, 0), (8.0, 9, 1)])
@pytest.mark.parametrize("cell_div", [1, 2])
def test_slab_thinner_than_the_cutoff(L, length, dipole, cell_div):
    """Two periodic dimensions and no padding: one cell, and one cluster of a
    chain's beads, spans more than half of the height.  LJ takes z as it is
    (no image of z), the real-space sum has the period of the height."""
    sd = _slab(L, (5.0 / 12.0) ** 2, length, 4, dipole)
    orc = O.Oracle(sd)
    eng = E.Engine(sd, cell_div=cell_div)
    assert eng.info().real_cutoff > L / 2
    ref = _full_matches(eng, orc)
    _vp_matches(eng, orc, sum(abs(v) for v in ref.values()))
    eng.close()
    eng, _, recs, _ = record_run(sd, 150, 16, seed=6)
    # a trial that leaves the slab is rejected by its wall term, its LJ (at a z
    # that the cell list wraps) is not the reference's
    out = [r for r in recs if r["dE"]["wall"] >= 0.9e8]
    assert not any(r["accepted"] for r in out) and len(out) <= len(recs) // 2
    for r in out:
        r["evaluated"] = False
    assert replay(sd, recs, 1e-10)[3] >= 50
    _full_matches(eng, O.Oracle(dict(sd, xyz=eng.positions())))


@pytest.mark.parametrize("box,npbc", [([6.0, 6.0, 6.0], 3), ([12.0, 12.0, 12.0], 3), ([9.0, 13.0, 18.0], 3),
                                      ([9.0, 9.0, 9.0], 2)])
def test_box_edge_equal_to_the_cutoff(box, npbc):
    """The derived cutoff is a whole number, and so are many boxes: a bead's own
    images then lie at the cutoff exactly, inside it (r <= r_c) in the energy,
    and the ones along z outside it in the stretched box."""
    sd = systems.config("slab_small" if npbc == 2 else "tiny")
    xyz, q, ty, ms = host.synth_system(4, 5, 20, 0, box, 3, npbc=npbc,
                                       z_range=(0.8, box[2] - 0.8) if npbc == 2 else None)
    sd.update(xyz=xyz, q=q, type=ty, mol_start=ms, box=box, alpha=systems.alpha_for_cutoff(box[0]), dipole=0,
              grafted=0)
    eng, orc = E.Engine(sd), O.Oracle(sd)
    assert eng.info().real_cutoff == box[0]
    ref = _full_matches(eng, orc)
    _vp_matches(eng, orc, sum(abs(v) for v in ref.values()))
