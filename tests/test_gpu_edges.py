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


@pytest.mark.parametrize("chain_len", [3, 8, 9, 17])
@pytest.mark.parametrize("split_div,cell_div", [(16, 4), (384, 1), (4000, 2)])
def test_query_shares_and_partial_clusters(chain_len, split_div, cell_div):
    """Real-space queries of one to eight blocks, clusters with one, seven and
    eight beads, cell lists from a few to over 256 cells per share; a fifth of
    the beads uncharged, so that pairs without an Ewald term occur too."""
    L = 15.0
    sd = systems.config("tiny")
    xyz, q, ty, ms = systems.build_bulk(6, chain_len, 6 * chain_len, L, 3 + chain_len)
    q = np.where(np.arange(len(q)) % 5 == 2, 0.0, q)
    sd.update(xyz=xyz, q=q, type=ty, mol_start=ms, box=[L, L, L], alpha=0.25)
    eng = E.Engine(sd, cell_div=cell_div)
    eng.set_tuning(split_div=split_div, cell_div=cell_div)
    eng.mc_record(200)
    eng.mc_run(120, sd["move_prob"], move_size=1.0, seed=chain_len)
    recs, _ = eng.mc_records(200)
    assert len(recs) >= 100
    replay(sd, recs, 1e-10)


@pytest.mark.parametrize("box,alpha,chain_len", [
    ([14.0, 14.0, 14.0], 0.02, 2),     # a handful of rows: one tile, mostly padding
    ([14.0, 14.0, 14.0], 0.9, 5),      # |l_z| on both sides of a tile edge
    ([9.0, 21.0, 14.0], 1.3, 3),       # unequal extents, two l_z groups in some rows only
    ([20.0, 8.0, 9.0], 0.5, 33),       # moved counts past a multiple of the four-step
])
def test_kspace_tiles(box, alpha, chain_len):
    """dS(k) of the speculative loop by tiles of 16 rows and 16 l_z."""
    sd = systems.config("tiny")
    xyz, q, ty, ms = systems.build_bulk(3, chain_len, 3 * chain_len, None, 21, box=box)
    sd.update(xyz=xyz, q=q, type=ty, mol_start=ms, box=box, alpha=alpha)
    eng, _, recs, _ = record_run(sd, 80, 16, seed=8)
    print("k extents", list(eng.info().repl_cell), "vectors", eng.info().n_k_half)
    replay(sd, recs, 1e-10)
    run, full = eng.totals(), eng.energy_full()
    assert abs(run["kspace"] - full["kspace"]) <= 1e-10 * max(1.0, abs(full["kspace"]))


def _full_matches(eng, orc, rel=1e-10):
    got, ref = eng.energy_full(), orc.energy_full()
    for k in E.TERMS:
        assert abs(got[k] - ref[k]) <= rel * max(abs(ref[k]), 1e-2), (k, got[k], ref[k])


@pytest.mark.parametrize("n_chains,chain_len,salt,L,alpha,cell_div", [
    (1, 2, 0, 12.0, 0.2, 1),        # four beads, most cells empty
    (2, 3, 1, 6.0, 0.05, 2),        # three image shells, one pair of ions
    (7, 9, 11, 16.0, 0.3, 3),       # odd counts
    (3, 100, 40, 14.0, 0.1, 1),     # one cell of 680 beads
])
def test_from_scratch_energy_and_cell_order(n_chains, chain_len, salt, L, alpha, cell_div):
    """The device-built cell list and the from-scratch sums (cluster queries,
    S(k) tiles, springs by waves), fresh, after moves that leave tombstones,
    and after a resync."""
    sd = systems.config("tiny")
    from plum_amd import host
    xyz, q, ty, ms = host.synth_system(n_chains, chain_len, n_chains * chain_len, salt, [L, L, L], 5)
    q = np.where(np.arange(len(q)) % 7 == 3, 0.0, q)
    sd.update(xyz=xyz, q=q, type=ty, mol_start=ms, box=[L, L, L], alpha=alpha)
    eng = E.Engine(sd, cell_div=cell_div)
    _full_matches(eng, O.Oracle(sd))
    rng = np.random.default_rng(1)
    for k in range(6):
        idx = np.arange(ms[k % n_chains], ms[k % n_chains + 1], dtype=np.int32)
        eng.delta(k % n_chains, idx, eng.positions()[idx] + rng.uniform(-2, 2, 3))
        eng.finalize(True)
    orc = O.Oracle(dict(sd, xyz=eng.positions()))
    _full_matches(eng, orc)
    run = eng.totals()
    drift = eng.resync()
    after = eng.totals()
    for k in E.TERMS:
        assert abs(run[k] - after[k] - drift[k]) <= 1e-12 * max(1.0, abs(run[k]))
    _full_matches(eng, orc)


def test_from_scratch_kspace_of_long_phase_rows():
    """A box 200 times as long as wide: a bead's phase table has 839 entries, four
    of which do not fit the LDS stage of the S(k) tiles, so S(k) is summed a
    thread per vector; and the trial move's k space with such rows."""
    sd = systems.config("tiny")
    box = [6.0, 6.0, 1300.0]
    xyz, q, ty, ms = systems.build_bulk(4, 5, 20, None, 3, box=box)
    sd.update(xyz=xyz, q=q, type=ty, mol_start=ms, box=box, alpha=0.4)
    eng, orc = E.Engine(sd), O.Oracle(sd)
    assert sum(eng.info().repl_cell) + 3 > 768
    _full_matches(eng, orc)
    idx = np.arange(ms[0], ms[1], dtype=np.int32)
    orc.set_trial(0, idx, xyz[idx] + 0.3)
    t_ref, d_ref = orc.delta(0)
    _, d = eng.delta(0, idx, xyz[idx] + 0.3)
    eng.finalize(True)
    for k in E.TERMS:
        assert abs(d[k] - d_ref[k]) <= 1e-10 * max(abs(d_ref[k]), 1e-2), (k, d[k], d_ref[k])
    eng.mc_run(64, sd["move_prob"], move_size=1.0, seed=3)
    run = eng.totals()
    _full_matches(eng, O.Oracle(dict(sd, xyz=eng.positions())))
    assert abs(run["kspace"] - eng.energy_full()["kspace"]) <= 1e-10 * abs(run["kspace"])


@pytest.mark.parametrize("L,cell_div,chains", [(100.0, 2, 5), (60.0, 2, 55), (100.0, 1, 5), (100.0, 2, 55)])
def test_mostly_empty_cells(L, cell_div, chains):
    """Neutral chains in a box of up to 512,000 cells, several hundred to a block
    of the from-scratch sums and several to a wave of the compaction: energy
    and pressure sample (over the pairs up to 2,048 beads, by cells beyond)
    against the oracle, fresh and after moves (tombstones, two compactions)."""
    from plum_amd import host
    sd = systems.config("tiny")
    xyz, q, ty, ms = host.synth_system(chains, 40, 0, 0, [L, L, L], 5, bead_q=0.0)
    xyz[80:120] = xyz[:40] + [0.4, 0.4, 0.4]     # two chains in the same cells
    sd.update(xyz=xyz, q=q, type=ty, mol_start=ms, box=[L, L, L], use_ewald=0)
    eng = E.Engine(sd, cell_div=cell_div)
    for moves in (0, 900):
        if moves:
            eng.mc_run(moves, sd["move_prob"], move_size=1.0, seed=3)
        orc = O.Oracle(dict(sd, xyz=eng.positions()))
        _full_matches(eng, orc)
        got, ref = eng.vp_sample(), orc.vp_sample(0)
        scale = sum(abs(v) for v in orc.energy_full().values())
        for k in ("lj", "bond", "dU"):
            assert abs(got[k] - ref[k]) <= 1e-14 * scale, (k, got[k], ref[k], scale)
        run, full = eng.totals(), eng.energy_full()
        assert abs(run["lj"] - full["lj"]) <= 1e-10 * scale


@pytest.mark.parametrize("npbc,phantom,use_bond", [(3, 0, 1), (2, 6, 1), (3, 4, 0)])
@pytest.mark.parametrize("length", [10, 130])   # 60 and 780 beads
def test_volume_perturbation_without_charges(npbc, phantom, use_bond, length):
    """The LJ part of a pressure sample over the bead pairs: with images, surface
    sites (which take no part), rigid molecules, beads far outside the box."""
    from plum_amd import host
    box = [20.0, 20.0, 14.0]
    sd = systems.config("slab_small" if npbc == 2 else "tiny")
    xyz, q, ty, ms = host.synth_system(6, length, 0, 0, box, 5, bead_q=0.0, npbc=npbc, min_sep=0.7,
                                       z_range=(0.8, box[2] - 0.8) if npbc == 2 else None)
    if npbc == 3:
        xyz = xyz + np.array([0.0, 0.0, 2.3 * box[2]])
    sites = np.c_[np.linspace(1, 19, phantom), np.linspace(1, 19, phantom), np.full(phantom, 7.0)]
    ms = np.r_[np.arange(phantom), ms + phantom].astype(np.int32)
    sd.update(xyz=np.r_[sites, xyz], q=np.r_[np.zeros(phantom), q], type=np.r_[np.zeros(phantom), ty].astype(np.int32),
              mol_start=ms, box=box, use_ewald=0, use_bond=use_bond, dipole=0, grafted=0, phantom=phantom)
    eng, orc = E.Engine(sd), O.Oracle(sd)
    got, ref = eng.vp_sample(phantom), orc.vp_sample(phantom)
    # 1e-14 of the energies, ten times that for coordinates 2.3 edges out (as
    # in test_volume_perturbation_sizes)
    scale = 1e-13 * sum(abs(v) for v in orc.energy_full().values())
    assert abs(ref["lj"]) > 1e3 * scale
    for k in ("lj", "wall", "bond", "dU"):
        assert abs(got[k] - ref[k]) <= scale, (k, got[k], ref[k], scale)


def test_spring_energy_has_one_set_of_bits():
    """The molecule springs of the from-scratch pass equal the trial path's
    bit for bit: a move that changes nothing has a spring dE of exactly 0."""
    sd = systems.config("tiny")
    from plum_amd import host
    xyz, q, ty, ms = host.synth_system(2, 700, 0, 0, [40.0, 40.0, 40.0], 9, bead_q=0.0)
    sd.update(xyz=xyz, q=q, type=ty, mol_start=ms, box=[40.0, 40.0, 40.0], alpha=0.05)
    eng = E.Engine(sd)
    for mol in (0, 1):
        idx = np.arange(ms[mol], ms[mol + 1], dtype=np.int32)
        _, d = eng.delta(mol, idx, xyz[idx])
        eng.finalize(False)
        assert d["bond"] == 0.0


@pytest.mark.parametrize("n_chains,chain_len,L,alpha", [(1, 2, 9.0, 0.2), (3, 7, 7.0, 0.06), (5, 11, 13.0, 0.5)])
def test_volume_perturbation_sizes(n_chains, chain_len, L, alpha):
    """The pressure sample by cluster queries and short bead chunks, from four
    beads up, with up to two image shells, the chains outside the box so that
    the listed images differ from the coordinates.  Bound of
    test_gpu_pressure.py (1e-14 of the summed energies), ten times wider: the
    oracle's stretched coordinates, up to 3.3 edges, round that much more."""
    sd = systems.config("tiny")
    xyz, q, ty, ms = systems.build_bulk(n_chains, chain_len, n_chains * chain_len, L, 31)
    xyz = xyz + np.array([0.0, 0.0, 2.3 * L])      # wrapped images differ from the coordinates
    sd.update(xyz=xyz, q=q, type=ty, mol_start=ms, box=[L, L, L], alpha=alpha)
    eng = E.Engine(sd)
    got = eng.vp_sample()
    orc = O.Oracle(sd)
    ref = orc.vp_sample(0)
    scale = sum(abs(v) for v in orc.energy_full().values())
    for k in ("el", "lj", "bond", "dU"):
        assert abs(got[k] - ref[k]) <= 1e-13 * scale, (k, got[k], ref[k], scale)


@pytest.mark.parametrize("samples,chain_len", [(1, 2), (3, 5), (2, 33), (17, 8)])
def test_gradient_tiles(samples, chain_len):
    """Loss and gradient with rows short of, at and past the 64-row and
    128-row tiles, against the float64 reference; FP32 products and sums of up
    to 272 rows and 128 inputs carry about sqrt(272 * 128) * 6e-8 of the
    gradient's norm at most (bound 1e-4, that of test_gpu_surrogate.py)."""
    sd = systems.config("tiny")
    xyz, q, ty, ms = systems.build_bulk(2, chain_len, 2 * chain_len, 12.0, 41)
    sd.update(xyz=xyz, q=q, type=ty, mol_start=ms, box=[12.0, 12.0, 12.0], alpha=0.2)
    eng = E.Engine(sd)
    eng.surrogate_enable(train_every=0, train_samples=1, ring=1, r_d=2.5, seed=3)
    rng = np.random.default_rng(samples)
    m = chain_len
    x = np.abs(rng.normal(0, 0.3, (samples, 2 * m, 64))).astype(np.float32)
    n = rng.integers(1, m + 1, samples).astype(np.int32)
    t = rng.normal(0, 15.0, samples)
    w = eng.surrogate_weights()
    loss, grad = eng.surrogate_gradient(x.reshape(-1, 64), t, n)
    ref_loss, ref = _reference_gradient(w, x, t, n)
    assert abs(loss - ref_loss) <= 1e-5 * abs(ref_loss)
    assert np.linalg.norm(grad - ref) <= 1e-4 * np.linalg.norm(ref)
    f = eng.surrogate_forward(x.reshape(-1, 64), bf16=False)
    assert np.max(np.abs(f - _reference_forward(w, x.reshape(-1, 64))[-1])) <= 1e-5 * max(1.0, np.max(np.abs(f)))


def test_gradient_in_several_passes():
    """155 chunks of 128 rows, a second pass of the weight gradients over 27 of
    them, the last one short."""
    test_gradient_tiles(300, 33)


def _layers(w):
    o = np.cumsum([0, 64 * 128, 128, 128 * 128, 128, 128 * 128, 128, 128, 1])
    w = np.asarray(w, dtype=np.float64)
    p = [w[o[i]:o[i + 1]] for i in range(8)]
    return [p[0].reshape(64, 128), p[1], p[2].reshape(128, 128), p[3], p[4].reshape(128, 128), p[5], p[6], p[7]]


def _reference_forward(w, x):
    p = _layers(w)
    h1 = np.tanh(x @ p[0] + p[1])
    h2 = np.tanh(h1 @ p[2] + p[3])
    h3 = np.tanh(h2 @ p[4] + p[5])
    return h1, h2, h3, h3 @ p[6] + p[7][0]


def _reference_gradient(w, x, t, n, clip=20.0):
    s, m2, _ = x.shape
    m = m2 // 2
    p = _layers(w)
    X = x.reshape(-1, 64).astype(np.float64)
    h1, h2, h3, f = _reference_forward(w, X)
    f = f.reshape(s, 2, m)
    used = np.arange(m)[None] < n[:, None]
    res = ((f[:, 1] - f[:, 0]) * used).sum(1) - np.clip(t, -clip, clip)
    g = np.zeros((s, 2, m))
    g[:, 0], g[:, 1] = -2 * res[:, None] * used / s, 2 * res[:, None] * used / s
    g = g.reshape(-1)
    d3 = np.outer(g, p[6]) * (1 - h3 ** 2)
    d2 = (d3 @ p[4].T) * (1 - h2 ** 2)
    d1 = (d2 @ p[2].T) * (1 - h1 ** 2)
    parts = [X.T @ d1, d1.sum(0), h1.T @ d2, d2.sum(0), h2.T @ d3, d3.sum(0), h3.T @ g, [g.sum()]]
    return np.mean(res ** 2), np.concatenate([np.ravel(v) for v in parts])


@pytest.mark.parametrize("K,L,mode,charged", [(1, 1, 0, True), (1, 5, 0, True), (3, 4, 1, True), (17, 6, 0, False),
                                              (33, 3, 2, True), (300, 2, 0, True)])
@pytest.mark.parametrize("precision", [E.PLUM_FP64, E.PLUM_FP32_PAIR])
def test_growth_steps(K, L, mode, charged, precision, alpha=None):
    """A whole growth (the choice of a bead repeated in every block, or past 32
    trials or 1,024 blocks made by one block) against the single-step trial energies of plum_cbmc_trials with the same
    draws: weight to 1e-10 (FP32 pairs: 1e-5, the exponent of the summed 1e-6
    errors), chosen beads exactly."""
    sd = systems.config("gc_small")
    if alpha:
        sd["alpha"] = alpha
    Lb = sd["box"][0]
    rng = np.random.default_rng(K + L)
    eng = E.Engine(sd, precision=precision)
    first = np.array([[0.3, 0.4, 0.2], [7.0, 6.0, 5.0]])
    d = first[:, None] - sd["xyz"][None]
    d -= Lb * np.round(d / Lb)
    while (d ** 2).sum(-1).min() < 0.81:
        first = rng.uniform(0, Lb, (2, 3))
        d = first[:, None] - sd["xyz"][None]
        d -= Lb * np.round(d / Lb)
    v = rng.normal(size=(L, K, 3))
    disp = v / np.linalg.norm(v, axis=-1)[..., None]
    ions = rng.uniform(0, Lb, (L, K, 3))
    sel = rng.uniform(0, 1, L)
    ms = sd["mol_start"]
    kw = dict(type_ion=1, q_ion=1.0) if charged else {}
    actual = exclude = None
    if mode == 1:
        exclude = (int(ms[0]), int(ms[7]) - 1)
        actual = np.concatenate([sd["xyz"][:L], sd["xyz"][6:6 + L]])
    for rep in range(2):   # the second growth replays the captured launches
        w, stop, chain = eng.cbmc_grow(mode, L, K, 0, -1.0, first=first, disp=disp, ions=ions, sel=sel, actual=actual,
                                       charged=charged, exclude=exclude, **kw)
    beads, gi, W, end = np.zeros((0, 3)), np.zeros((0, 3)), 1.0, -1
    for s in range(L):
        if s == 0:
            b, i = (actual[:1], actual[L:L + 1]) if mode == 1 else (first[:1], first[1:])
        else:
            b, i = beads[-1] + disp[s], ions[s].copy()
            if mode == 1:
                b[0], i[0] = actual[s], actual[L + s]
        e = eng.cbmc_trials(b, 0, -1.0, grown=beads, ions=i if charged else None, type_ion=1, q_ion=1.0,
                            grown_ions=gi if charged else None, exclude=exclude)
        p = np.exp(-e)
        W *= p.sum() / len(p)
        if W == 0:   # every trial overlaps: the growth ends here
            end = s
            break
        pick = 0
        if s and mode != 1:
            pick = min(int(np.searchsorted(np.cumsum(p), sel[s] * p.sum())), len(p) - 1)
        beads, gi = np.vstack([beads, b[pick]]), np.vstack([gi, i[pick]])
    assert stop == end
    assert abs(w - W) <= (1e-10 if precision == E.PLUM_FP64 else 1e-5) * W
    assert np.array_equal(chain[:len(beads)], beads)
    if charged:
        assert np.array_equal(chain[L:L + len(gi)], gi)


@pytest.mark.parametrize("K,L,mode,alpha", [(32, 4, 0, None), (33, 4, 1, None), (32, 4, 0, 3.2), (30, 3, 1, 3.2),
                                            (1024, 2, 0, None)])
def test_growth_on_both_sides_of_the_choice_rule(K, L, mode, alpha):
    """The last number of trials whose choice every block repeats, the first
    whose choice one block makes, the same below 32 trials with so many k
    vectors that the step passes 1,024 blocks, and the largest number."""
    if alpha:
        eng = E.Engine(dict(systems.config("gc_small"), alpha=alpha))
        assert K * (3 + eng.info().n_k_half // 256) > 1024
        eng.close()
    test_growth_steps(K, L, mode, True, E.PLUM_FP64, alpha)


def test_growth_after_a_regrid():
    """The captured growth belongs to one cell list: after a re-grid it is
    captured again, and gives the weight it gave before."""
    sd = systems.config("gc_small")
    rng = np.random.default_rng(4)
    Lb = sd["box"][0]
    kw = dict(first=np.array([[0.3, 0.4, 0.2], [7.0, 6.0, 5.0]]), disp=np.full((3, 4, 3), 0.58),
              ions=rng.uniform(0, Lb, (3, 4, 3)), sel=np.full(3, 0.5), type_ion=1, q_ion=1.0)
    eng = E.Engine(sd)
    a = eng.cbmc_grow(2, 3, 4, 0, -1.0, **kw)
    eng.set_tuning(cell_div=3)
    eng.mc_run(40, sd["move_prob"], seed=3)
    x = eng.positions()
    b = eng.cbmc_grow(2, 3, 4, 0, -1.0, **kw)
    c = E.Engine(dict(sd, xyz=x)).cbmc_grow(2, 3, 4, 0, -1.0, **kw)
    assert abs(b[0] - c[0]) <= 1e-9 * abs(c[0]) and np.array_equal(b[2], c[2])


@pytest.mark.parametrize("n", [0, 1, 7, 8, 9, 17, 70])
def test_host_moves_of_every_size(n):
    """The caller's move read from pinned memory, eight beads a block: any
    subset of a molecule's beads, three moves in a row, the second one
    rejected, each against the oracle at the coordinates before it."""
    sd = systems.config("tiny")
    xyz, q, ty, ms = systems.build_bulk(2, 70, 6, 14.0, 3)
    sd.update(xyz=xyz, q=q, type=ty, mol_start=ms, box=[14.0] * 3)
    eng = E.Engine(sd)
    rng = np.random.default_rng(n)
    for step in range(3):
        x = eng.positions()
        idx = np.sort(rng.choice(np.arange(ms[0], ms[1]), n, replace=False)).astype(np.int32)
        new = x[idx] + rng.normal(0, 0.02, (n, 3))
        orc = O.Oracle(dict(sd, xyz=x))
        orc.set_trial(0, idx, new)
        t_ref, d_ref = orc.delta(0)
        t, d = eng.delta(0, idx, new)
        for k in E.TERMS:
            assert abs(d[k] - d_ref[k]) <= 1e-10 * max(abs(d_ref[k]), 1e-2), (step, k, d[k], d_ref[k])
        eng.finalize(step != 1)
        x1 = x.copy()
        if step != 1:
            x1[idx] = new
        assert np.array_equal(eng.positions(), x1)


@pytest.mark.parametrize("pmax", [1, 2, 3, 15, 16])
@pytest.mark.parametrize("alpha", [0.02, 0.9])   # fewer k vectors than waves; several steps a wave
def test_cross_sums_of_a_batch(pmax, alpha):
    """Cross terms of one to sixteen slots: the k-space Gram matrix with rows
    and k vectors past the end, the near pairs a wave each."""
    sd = systems.config("tiny")
    xyz, q, ty, ms = systems.build_bulk(4, 40, 20, 14.0, 6)
    sd.update(xyz=xyz, q=q, type=ty, mol_start=ms, box=[14.0] * 3, alpha=alpha, move_prob=[0.6, 0.1, 0.1, 0.1, 0.1])
    eng, st, recs, _ = record_run(sd, 200, pmax, seed=pmax)
    run, full = eng.totals(), eng.energy_full()
    # dE_k is what is left of sums whose terms add up to about the k-space and
    # self energies E (a hundred kT and more at alpha 0.9), each with phases of
    # l <= 20 rounded factors: up to 20 x 2.2e-16 E each way, 1e-14 E together,
    # which the scaled tolerance allows at a floor of 1e-4 E
    scale = max(abs(full["kspace"]), abs(full["self"]))
    replay(sd, recs, 1e-10, floor=max(1e-2, 1e-4 * scale))
    assert abs(run["kspace"] - full["kspace"]) <= 1e-10 * max(1.0, abs(full["kspace"]))


def test_training_ring_rows_past_a_sample():
    """Rows of the training ring past a sample's beads are never written and do
    not reach the gradient: the ring starts as NaN, most samples move fewer beads
    than the longest molecule has, and loss and weights stay finite."""
    sd = systems.config("slab_small")
    eng = E.Engine(sd)
    eng.surrogate_enable(screen=16, fill=8, train_every=0, train_samples=64, ring=512, seed=8)
    eng.mc_run(600, sd["move_prob"], move_size=sd["move_size"], seed=5, phantom=sd.get("phantom", 0),
               grafted=sd.get("grafted", 0), bond_len=1.0)
    a, b = eng.surrogate_train(1), eng.surrogate_train(50)
    assert np.isfinite(a) and np.isfinite(b)
    assert np.all(np.isfinite(eng.surrogate_weights()))
