"""Faults that were found in the kernels and mended, each with the case that showed it, through the C ABI.

Tolerances as where the kernels' sizes are tested: trajectories bit for bit; a whole-system energy within 1e-5 of
the sum of the particles' |E| + 2e-4 kT, a particle's energy within 1e-5 |E| + 2e-4 kT of the FP64 oracle.
"""
import numpy as np
import pytest

import sc_amd
from sc_amd import workloads as W
import pyoracle as po

pytestmark = pytest.mark.gpu
ROT_HALF = 20.0 / 180 * np.pi / 4


def say(*a):
    print(*a, flush=True)


def psc_state(g, n, eta, seed, box=None):
    """n PSC at random without overlap; the oracle's topology and the device's own state"""
    top = W.top_init([W.TYPES["psc"]], [n])
    types = np.ones(n, np.int32)
    box = np.full(3, (n * W.particle_volume(1.0, 3.0) / eta) ** (1.0 / 3.0)) if box is None else np.asarray(box, float)
    g.load_topology(top)
    pos, d, q = g.generate_rsa(types, box, seed)
    g.set_config(box, pos, d, q, types)
    b, p, dd, qq = g.get_config()
    return po.Topo(top), po.State(b, p, dd, qq, types)


@pytest.mark.parametrize("eta,r", [(0.01, 1), (0.02, 1), (0.02, 2), (0.04, 1)])
def test_chain_sweep_of_sparse_stencils(eta, r):
    """A stage copied in two passes, from stencils of fewer particles than the block has lanes: waves without a
    particle of their own must not write over the cell's centre that the others still read (the compaction counts
    lay in the same LDS words).  The one-trial-at-a-time trajectory bit for bit."""
    say("case: chain sweep, eta %.2f, r %d" % (eta, r))
    box, pos, d, q, t = W.chain_lattice(300, eta, 11)
    out = []
    for nw in (0, 1):
        with sc_amd.GpuSystem(0) as g:
            g.load_topology(W.chain_topology(300))
            g.set_config(box, pos, d, q, t)
            g.set_block_waves(nw)
            s = g.sweep(20, 1.1, 0.3, ROT_HALF, r=r, seed=23, counter=0)
            out.append((s, g.get_config()))
    (s1, c1), (s2, c2) = out
    say("accepted %d / %d" % (s1["trans_acc"] + s1["rot_acc"], s1["trans_try"] + s1["rot_try"]))
    assert s1["trans_acc"] + s1["rot_acc"] > 0
    for k in ("trans_acc", "trans_try", "rot_acc", "rot_try", "left_cell", "bond_rejected"):
        assert s1[k] == s2[k], k
    for a, b in zip(c1, c2):
        np.testing.assert_array_equal(a, b)


@pytest.mark.parametrize("n,eta", [(150, 0.05), (1000, 0.20), (3000, 0.20)])
def test_whole_system_energy_of_two_pass_stages(n, eta):
    """the same words under the whole-system energy: stencils of one to a few waves of particles"""
    say("case: whole-system energy, %d PSC at eta %.2f" % (n, eta))
    with sc_amd.GpuSystem(0) as g:
        tp, st = psc_state(g, n, eta, n)
        e, want = g.allToAll(), po.energy_all(tp, st, use_cells=True)
        size = np.abs(po.energy_one_each(tp, st, np.arange(n))).sum()
        say("gpu %.8f oracle %.8f" % (e, want))
        assert abs(e - want) <= 1e-5 * size + 2e-4


@pytest.mark.parametrize("before", ["pair list", "pair list below the cells' width", "alignment order", "trial box"])
def test_particle_energies_after_another_grid(before):
    """Energies of single particles search the cell list that is there: not one with narrower cells, as a pair list
    of a short range and a larger trial box leave it."""
    say("case: particle energies after a", before)
    n = 3000
    with sc_amd.GpuSystem(0) as g:
        tp, st = psc_state(g, n, 0.2, 21)
        if before == "pair list":
            g.neighbor_pairs(2.5)
        elif before == "pair list below the cells' width":
            g.neighbor_pairs(0.5)
        elif before == "alignment order":
            g.alignment_order()
        else:
            g.allToAllTrial(2.0 * st.box)
        one = g.oneToAll(7)
        trial = g.oneToAllTrial(7, st.pos[7], st.dir[7], st.pd0[7])
        mol = g.mol2others(7, 1)
        e, want = g.energy_per_particle(), po.energy_one_each(tp, st, np.arange(n))
        say("max error %.2e; particle 7: %.8f, oracle %.8f" % (np.abs(e - want).max(), one, want[7]))
        assert np.all(np.abs(e - want) <= 1e-5 * np.abs(want) + 2e-4)
        for v in (one, trial, mol):
            assert abs(v - want[7]) <= 1e-5 * abs(want[7]) + 2e-4


def crowded_ball(g):
    """320 small spheres in a ball, a sphere beside it that has them all within reach (as many as a trial's list
    holds), and one more at the end of that sphere's reach"""
    k = np.stack(np.meshgrid(*[np.arange(7)] * 3, indexing="ij"), -1).reshape(-1, 3)[:320]
    pos = np.concatenate([(k - 3) * 0.35, [[3.0, 0.0, 0.0], [8.003, 0.0, 0.0]]]) + 8.0
    n = len(pos)
    g.load_topology(W.top_init(["S 1 SPA 1.0 0.3 4.5 0.5"], [n]))
    g.set_config(np.full(3, 24.0), pos / 24.0, np.tile([0.0, 0.0, 1.0], (n, 1)), np.tile([1.0, 0.0, 0.0], (n, 1)),
                 np.ones(n, np.int32))


def test_full_list_of_a_trial_behind_an_accepted_one():
    """A speculative trial whose list is full because of where an earlier accepted trial of its round stood is
    evaluated again, not reported: at these seeds the far sphere leaves the reach before the near one's trial."""
    for seed in (94, 149, 176, 461):
        say("case: the last candidate has left, seed %d" % seed)
        out = []
        for nw in (0, 1):
            with sc_amd.GpuSystem(0) as g:
                crowded_ball(g)
                g.set_block_waves(nw)
                s = g.sweep(1, 1000.0, 0.05, 0.1, r=1, seed=seed, counter=0)
                out.append((s["trans_acc"], s["trans_try"], g.get_config()))
        assert out[0][:2] == out[1][:2] and out[0][0] > 0
        for a, b in zip(out[0][2], out[1][2]):
            np.testing.assert_array_equal(a, b)
    for seed in (0, 1):
        say("case: the list is full in sequence too, seed %d" % seed)
        with sc_amd.GpuSystem(0) as g:
            crowded_ball(g)
            with pytest.raises(sc_amd.SCError, match="320 particles"):
                g.sweep(1, 1000.0, 0.05, 0.1, r=1, seed=seed, counter=0)


def with_nan_axis(g, line, n, box, seed, k=5):
    """n particles at random, the axis of particle k no number; (positions, axes, patch directions)"""
    rng = np.random.default_rng(seed)
    top, types = W.top_init([line], [n]), np.ones(n, np.int32)
    g.load_topology(top)
    pos, d, q = g.generate_rsa(types, np.full(3, box), seed)
    bad = d.copy()
    bad[k] = np.nan
    g.set_config(np.full(3, box), pos, bad, q, types)
    return pos, d, q


def test_axis_that_is_no_number():
    """A rod with a NaN axis has NaN energies with what lies within the cutoff; a sphere's axis does not matter."""
    say("case: rods")
    rod = W.TYPES["psc"]
    with sc_amd.GpuSystem(0) as g:
        pos, d, q = with_nan_axis(g, rod, 600, 22.0, 3)
        assert np.isnan(g.allToAll()) and np.isnan(g.oneToAll(5))
        g.set_config(np.full(3, 22.0), pos, d, q, np.ones(600, np.int32))
        assert np.isfinite(g.allToAll()) and np.isnan(g.oneToAllTrial(9, pos[9], np.full(3, np.nan), q[9]))
    say("case: spheres")
    with sc_amd.GpuSystem(0) as g:
        pos, d, q = with_nan_axis(g, "S 1 SPA 1.0 1.0 1.0 0.2", 600, 10.0, 4)
        e, each = g.allToAll(), g.energy_per_particle()
        g.set_config(np.full(3, 10.0), pos, d, q, np.ones(600, np.int32))
        assert each[5] != 0.0
        np.testing.assert_array_equal(each, g.energy_per_particle())
        assert e == g.allToAll()


def test_sweep_with_an_axis_that_is_no_number():
    """A rod of NaN axis with others in its cutoff never moves (its energy differences are NaN); a sphere's moves
    are those of the one-trial-at-a-time trajectory."""
    say("case: sweep of rods")
    with sc_amd.GpuSystem(0) as g:
        with_nan_axis(g, W.TYPES["psc"], 600, 22.0, 6)
        u = g.fixed_positions()
        s = g.sweep(10, 1.0, 0.2, ROT_HALF, r=1, seed=2, counter=0)
        assert s["trans_acc"] > 0
        np.testing.assert_array_equal(g.fixed_positions()[5], u[5])
    say("case: sweep of spheres")
    out = []
    for nw in (0, 1):
        with sc_amd.GpuSystem(0) as g:
            with_nan_axis(g, "S 1 SPA 1.0 1.0 1.0 0.2", 600, 10.0, 6)
            g.set_block_waves(nw)
            s = g.sweep(10, 1.0, 0.2, ROT_HALF, r=1, seed=2, counter=0)
            out.append((s, g.fixed_positions()))
    assert out[0][0]["trans_acc"] == out[1][0]["trans_acc"] > 0
    np.testing.assert_array_equal(out[0][1], out[1][1])


def crowded_cell(g):
    """1,280 rods of two types within 28 sigma of a box of 240"""
    types = np.repeat([1, 2], 640).astype(np.int32)
    g.load_topology(W.top_init([W.TYPES["psc"], W.TYPES["cpsc"]], [640, 640]))
    pos, d, q = g.generate_rsa(types, np.full(3, 28.0), 8)
    g.set_config(np.full(3, 240.0), pos * 28.0 / 240.0 + 0.3, d, q, types)
    g.set_max_active_cells(1)


def test_sweep_of_a_crowded_cell():
    """as many rods in one cell as a stage of records alone holds: the rows and the source list beside them are no
    reason to refuse it"""
    say("case: 1280 rods in one cell")
    with sc_amd.GpuSystem(0) as g:
        crowded_cell(g)
        e0 = 0.5 * g.energy_per_particle().sum()
        s = g.sweep(10, 1.0, 0.3, ROT_HALF, r=1, seed=3, counter=0)
        e1 = 0.5 * g.energy_per_particle().sum()
        say("accepted %d / %d" % (s["trans_acc"] + s["rot_acc"], s["trans_try"] + s["rot_try"]))
        assert s["trans_try"] + s["rot_try"] == 12800 and s["trans_acc"] + s["rot_acc"] > 0
        assert abs(e1 - e0 - s["energy_change"]) <= 1e-8 * max(abs(e0), abs(e1), 1.0)


def test_chain_sweep_of_a_crowded_cell():
    """402 chains in one cell: the table of their partners does not fit beside the stage, and the
    one-trial-at-a-time trajectory comes out all the same."""
    say("case: 402 chains in one cell")
    small, pos, d, q, t = W.chain_lattice(402, 0.2, 5)
    out = []
    for nw in (0, 1):
        with sc_amd.GpuSystem(0) as g:
            g.load_topology(W.chain_topology(402))
            g.set_config(np.full(3, 120.0), pos * small / 120.0 + 0.35, d, q, t)
            g.set_max_active_cells(1)
            g.set_block_waves(nw)
            s = g.sweep(10, 1.1, 0.3, ROT_HALF, r=1, seed=29, counter=0)
            out.append((s, g.get_config()))
    (s1, c1), (s2, c2) = out
    say("accepted %d / %d" % (s1["trans_acc"] + s1["rot_acc"], s1["trans_try"] + s1["rot_try"]))
    assert s1["trans_acc"] + s1["rot_acc"] > 0
    for k in ("trans_acc", "trans_try", "rot_acc", "rot_try", "left_cell", "bond_rejected"):
        assert s1[k] == s2[k], k
    for a, b in zip(c1, c2):
        np.testing.assert_array_equal(a, b)


@pytest.mark.parametrize("key,cap", [("psc", 0), ("psc", 4), ("tchpsc", 0), ("tchpsc", 4)])
def test_sweep_without_rows(key, cap):
    """Patch terms of neighbours whose vectors the stage does not hold, derived a chunk of entries at a time (16 of one
    patch, 8 of two): the one-trial-at-a-time trajectory bit for bit in a dense system, entries beyond one chunk."""
    say("case: sweep of %s without rows, home cache %d" % (key, cap))
    n, ty, length = 800, {"psc": 1, "tchpsc": 3}[key], {"psc": 3.0, "tchpsc": 4.0}[key]
    start = np.full(3, (n * W.particle_volume(1.0, length) / 0.13) ** (1.0 / 3.0))
    box = start * (0.13 / 0.38) ** (1.0 / 3.0)
    out = []
    for nw in (0, 1):
        with sc_amd.GpuSystem(0) as g:
            g.load_topology(W.top_init([W.TYPES[key]], [n]))
            pos, d, q = g.generate_rsa(np.full(n, ty, np.int32), start, 12)
            g.set_config(start, pos, d, q, np.full(n, ty, np.int32))
            for k in range(1, 9):
                g.update_box(start * (box / start) ** (k / 8.0))
                g.sweep(5, 0.3, 0.3, ROT_HALF, r=1, seed=4, counter=10 * k)
            g.set_block_waves(nw)
            g.set_home_cache(cap)
            s = g.sweep(10, 0.3, 0.2, ROT_HALF, r=1, seed=7, counter=1000)
            out.append((s, g.get_config()))
    (s1, c1), (s2, c2) = out
    say("accepted %d / %d" % (s1["trans_acc"] + s1["rot_acc"], s1["trans_try"] + s1["rot_try"]))
    assert s1["trans_acc"] + s1["rot_acc"] > 0
    for k in ("trans_acc", "trans_try", "rot_acc", "rot_try", "left_cell"):
        assert s1[k] == s2[k], k
    for a, b in zip(c1, c2):
        np.testing.assert_array_equal(a, b)


@pytest.mark.parametrize("nchains", [30, 250])
def test_chain_moves_proposed_beside_a_move(nchains):
    """Few molecules per coarse cell and 27 visits: the molecule proposed beside a move is often the one that moves,
    and is proposed again.  Staged passes, moves of both kinds accepted, no cell left out; every accepted energy
    change was taken from the state that the move found (a stale proposal breaks the sum)."""
    say("case: proposals beside moves, %d chains" % nchains)
    with sc_amd.GpuSystem(0) as g:
        box, pos, d, q, t = W.chain_lattice(nchains, 0.2 if nchains > 100 else 0.01, 4)
        g.load_topology(W.chain_topology(nchains))
        g.set_config(box, pos, d, q, t)
        g.set_trial_mode(1)
        g.set_chain_moves(0.3, 0.5, 0.2)
        g.set_chain_visit_factor(27)
        e0 = g.allToAll()
        s = g.sweep(20, 1.0, 0.3, ROT_HALF, r=1, seed=9, counter=0)
        e1 = g.allToAll()
        say({k: v for k, v in s.items() if k.startswith("chain")})
        assert g.chain_pass_info()[1] and s["chain_cells_skipped"] == 0
        assert s["chain_disp_acc"] > 0 and s["chain_rot_acc"] > 0
        assert abs(e1 - e0 - s["energy_change"]) <= 1e-8 * max(abs(e0), abs(e1), 1.0)


SPECIES = {"psc": (W.TYPES["psc"], 1, 3.0), "cpsc": (W.TYPES["cpsc"], 2, 3.0), "tchpsc": (W.TYPES["tchpsc"], 3, 4.0),
           "tcpsc": ("D 4 TCPSC 1.0 1.0 1.0 0.2 80.0 5.0 3.0 0.0 120.0 70.0 5.0", 4, 3.0),
           "spa": ("S 6 SPA 1.0 1.0 1.0 0.2", 6, 0.0)}


@pytest.mark.parametrize("keys", [("psc",), ("cpsc",), ("tchpsc",), ("tcpsc",), ("tchpsc", "spa"), ("psc", "cpsc", "tchpsc")])
def test_one_value_of_a_pair_in_queries_and_lists(keys):
    """A pair has one FP32 value wherever it is priced: a particle's energy is the sum of its pairs' energies, the
    whole system's the sum of all, but for the order of FP64 sums.  (The queries normalised their neighbours' axes
    with a correctly rounded root where the other kernels have the hardware's: 1e-7 to 1e-6 kT off.)"""
    say("case: pair values of", *keys)
    m = 1800 // len(keys)
    types = np.concatenate([np.full(m, SPECIES[k][1], np.int32) for k in keys])
    vol = sum(m * W.particle_volume(1.0, SPECIES[k][2]) for k in keys)
    start = np.full(3, (vol / 0.12) ** (1.0 / 3.0))
    with sc_amd.GpuSystem(0) as g:
        g.load_topology(W.top_init([SPECIES[k][0] for k in keys], [m] * len(keys)))
        pos, d, q = g.generate_rsa(types, start, 3)
        g.set_config(start, pos, d, q, types)
        for k in range(1, 7):
            g.update_box(start * (0.12 / 0.28) ** (k / 18.0))
            g.sweep(4, 1.0, 0.3, ROT_HALF, r=1, seed=4, counter=10 * k)
        p = g.neighbor_pairs(g.maxcut)
        e = g.p2p(p[:, 1], p[:, 0])
        each = np.zeros(len(types))
        np.add.at(each, p[:, 0], e)
        np.add.at(each, p[:, 1], e)
        got = g.energy_per_particle()
        say("largest difference %.2e kT" % np.abs(got - each).max())
        size = np.zeros(len(types))
        np.add.at(size, p[:, 0], np.abs(e))
        np.add.at(size, p[:, 1], np.abs(e))
        assert np.all(np.abs(got - each) <= 1e-12 * (1.0 + size))
        assert abs(g.oneToAll(5) - each[5]) <= 1e-12 * (1.0 + size[5])
        assert abs(g.allToAll() - e.sum()) <= 1e-12 * (1.0 + np.abs(e).sum())


def test_network_screen_of_the_sweeps_variants():
    """The speculative sweep with the network screen is the one-trial-at-a-time sweep: every trial past the first
    screen goes to the network, so a feature an ulp off in one of them would show as another decision."""
    say("case: network screen, 32,768 TCHPSC, speculative and four waves a trial")
    n = 32768
    types = np.full(n, 3, np.int32)
    start = np.full(3, (n * W.particle_volume(1.0, 4.0) / 0.13) ** (1.0 / 3.0))
    rng = np.random.default_rng(5)
    w = None
    out = []
    for nw in (0, 4):
        with sc_amd.GpuSystem(0) as g:
            g.load_topology(W.top_init([W.TYPES["tchpsc"]], [n]))
            pos, d, q = g.generate_rsa(types, start, 6)
            g.set_config(start, pos, d, q, types)
            for k in range(1, 7):
                g.update_box(start * (0.13 / 0.25) ** (k / 18.0))
                g.sweep(4, 1.0, 0.3, ROT_HALF, r=1, seed=4, counter=10 * k)
            g.mlp_init(3, seed=2)
            if w is None:
                w = g.mlp_get_weights()
                w[-65:-1] = 3.0 * rng.normal(size=64)
            g.mlp_set_weights(w)
            g.set_surrogate(1)
            g.set_network_min_entries(0)
            g.set_trial_mode(1)
            g.set_visit_factor(8)
            g.set_block_waves(nw)
            s = g.sweep(400, 1.0, 0.3, ROT_HALF, r=1, seed=8, counter=1000)
            out.append((s, g.fixed_positions()))
    (s1, u1), (s2, u2) = out
    say("screened %d, passed %d and %d" % (s1["stage2_try"], s1["stage2_acc"], s2["stage2_acc"]))
    assert s1["stage2_try"] > 10 ** 6
    for k in ("stage1_acc", "stage2_try", "stage2_acc", "trans_acc", "rot_acc"):
        assert s1[k] == s2[k], k
    np.testing.assert_array_equal(u1, u2)
