"""Sizes at which a kernel's split, capacity or remainder changes, through the
C ABI, against the FP64 oracle (or the other variant of the same kernel).

Tolerances:
  * energies: a pair term's FP32 error is that of its separation vector (2e-7
    sigma) times the term's slope (up to ~100 kT per sigma outside overlaps),
    with ten such terms per particle: 1e-5 |E| + 2e-4 kT per particle energy,
    1e-5 of the sum of the particles' |E| + 2e-4 kT for the whole system;
  * FP64 pair energies 1e-9 relative, as everywhere;
  * network outputs 1e-5, gradients 2e-4 of the block's largest, as everywhere;
  * cell lists, pair lists and trajectories bit for bit; energies that differ
    in the order of FP64 sums only: 1e-9; energy bookkeeping 1e-8 |E|;
  * S2: the axes are FP32 unit vectors, 1e-6.
"""
import os

import numpy as np
import pytest

import sc_amd
from sc_amd import workloads as W
import mlp_oracle as mo
import pyoracle as po

pytestmark = pytest.mark.gpu
ROT_HALF = 20.0 / 180 * np.pi / 4
GOLD = os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden")


def say(*a):
    print(*a, flush=True)


def axes(n, rng):
    d = rng.normal(size=(n, 3))
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    q = np.cross(d, rng.normal(size=(n, 3)))
    return d, q / np.linalg.norm(q, axis=1, keepdims=True)


def mixture(g, n, box, seed):
    """n particles, PSC and CPSC alternating, at random without overlap; the device's own state"""
    top = W.top_init([W.TYPES["psc"], W.TYPES["cpsc"]], [n - n // 2, n // 2])
    types = np.array([1] * (n - n // 2) + [2] * (n // 2), np.int32)
    g.load_topology(top)
    pos, d, q = g.generate_rsa(types, np.asarray(box, float), seed)
    g.set_config(box, pos, d, q, types)
    b, p, dd, qq = g.get_config()
    return po.Topo(top), po.State(b, p, dd, qq, types)


def edge(n, eta):
    return (n * W.particle_volume(1.0, 3.0) / eta) ** (1.0 / 3.0)


@pytest.mark.parametrize("n", [2, 63, 64, 65, 1023, 1024, 1025])
def test_particle_energies(n):
    """one wave or four per query; the queries of a call beyond the pinned ones"""
    say("case: per-particle energies, n %d" % n)
    with sc_amd.GpuSystem(0) as g:
        tp, st = mixture(g, n, np.full(3, max(14.0, edge(n, 0.15))), n)
        e, want = g.energy_per_particle(), po.energy_one_each(tp, st, np.arange(n))
        say("max error %.2e of |E| up to %.2f" % (np.abs(e - want).max(), np.abs(want).max()))
        assert np.all(np.abs(e - want) <= 1e-5 * np.abs(want) + 2e-4)
        assert abs(g.oneToAll(n - 1) - e[n - 1]) <= 1e-9 * max(1.0, abs(e[n - 1]))


@pytest.mark.parametrize("shape", [(1.5, 1.5, 1.5), (2.2, 2.2, 2.2), (2.6, 2.6, 2.6), (3.4, 3.4, 3.4),
                                   (1.5, 2.6, 5.1), (5.1, 5.1, 5.1)])
def test_whole_system_energy(shape):
    """boxes of one cell per axis to more than the stencil: pairs by half the stencil or by ID"""
    say("case: whole-system energy, box %s maxcut" % (shape,))
    with sc_amd.GpuSystem(0) as g:
        g.load_topology(W.top_init([W.TYPES["psc"], W.TYPES["cpsc"]], [1, 1]))
        box = g.maxcut * np.array(shape)
        n = int(0.12 * box.prod() / W.particle_volume(1.0, 3.0))
        tp, st = mixture(g, n, box, 17)
        size = np.abs(po.energy_one_each(tp, st, np.arange(n))).sum()
        for s in (1.0, 1.004):
            e = g.allToAll() if s == 1.0 else g.allToAllTrial(box * s)
            want = po.energy_all(tp, po.State(box * s, st.pos, st.dir, st.pd0, st.types), use_cells=False)
            say("n %d, box x%.3f: gpu %.8f oracle %.8f" % (n, s, e, want))
            assert abs(e - want) <= 1e-5 * size + 2e-4


@pytest.mark.parametrize("nx,spread", [(6, 3.0), (16, 4.0), (22, 1.02)])
def test_whole_system_energy_of_a_cluster(nx, spread):
    """aligned rods packed in a corner of their box, and a box full of them (beyond the estimated stage: evaluated
    again with the full one); a cluster of 1024 in a box of four times its edges is beyond every stage and refused"""
    k = np.stack(np.meshgrid(np.arange(nx), np.arange(nx), np.arange(max(2, nx // 4)), indexing="ij"), -1).reshape(-1, 3)
    pos = k * np.array([1.1, 1.1, 4.2]) + 0.5
    n, rng = len(k), np.random.default_rng(nx)
    box = spread * (pos.max(0) + np.array([0.6, 0.6, 3.7]))
    say("case: whole-system energy, cluster of %d rods in a box of %s" % (n, np.round(box, 1)))
    d = rng.normal(0.0, 0.01, (n, 3)) + [0.0, 0.0, 1.0]   # (the oracle has no value for exactly parallel pairs)
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    q = np.cross(d, rng.normal(size=(n, 3)))
    q /= np.linalg.norm(q, axis=1, keepdims=True)
    types = np.ones(n, np.int32)
    top = W.top_init([W.TYPES["psc"]], [n])
    with sc_amd.GpuSystem(0) as g:
        g.load_topology(top)
        g.set_config(box, pos / box, d, q, types)
        b, p, dd, qq = g.get_config()
        tp, st = po.Topo(top), po.State(b, p, dd, qq, types)
        if nx == 16:
            with pytest.raises(sc_amd.SCError, match="stage capacity"):
                g.allToAll()
            return
        one = po.energy_one_each(tp, st, np.arange(n))
        e, want = g.allToAll(), po.energy_all(tp, st, use_cells=True)
        say("gpu %.8f oracle %.8f" % (e, want))
        assert abs(e - want) <= 1e-5 * np.abs(one).sum() + 2e-4
        eg = g.energy_per_particle()
        assert np.all(np.abs(eg - one) <= 1e-5 * np.abs(one) + 2e-4)


def test_replica_energies_equal_those_of_the_replicas():
    say("case: energies of a batch of uneven replicas")
    sizes, top = [60, 65, 700, 1500], W.top_init([W.TYPES["psc"]], [2325])
    with sc_amd.GpuSystem(0) as g, sc_amd.GpuSystem(0) as s:
        g.load_topology(top)
        parts, boxes = [], []
        for k, n in enumerate(sizes):
            boxes.append([edge(n, 0.15)] * 3)
            parts.append(g.generate_rsa(np.ones(n, np.int32), np.array(boxes[-1]), 5 + k))
        g.set_config(np.array(boxes[0]), *(np.concatenate([p[i] for p in parts]) for i in range(3)),
                     np.ones(2325, np.int32))
        g.batch_set(np.array(sizes, np.int32), np.array(boxes))
        e = g.batch_energies()
        s.load_topology(top)
        for k, n in enumerate(sizes):
            s.set_config(np.array(boxes[k]), *parts[k], np.ones(n, np.int32))
            want = s.allToAll()
            say("replica %d: batch %.12f alone %.12f" % (k, e[k], want))
            assert abs(e[k] - want) <= 1e-9 * max(1.0, abs(want))


@pytest.mark.parametrize("n,cells", [(1, (2, 2, 2)), (4095, (20, 20, 20)), (4096, (16, 16, 32)), (4097, (16, 16, 32)),
                                     (4096, (20, 20, 22)), (5000, (2, 2, 2)), (5000, (26, 26, 26)), (20000, (32, 32, 32))])
def test_cell_list(n, cells):
    """one block or several launches (4096 particles, 8192 cells); the scan's chunks of 8192 cells"""
    say("case: cell list, %d particles, cells %s" % (n, cells))
    with sc_amd.GpuSystem(0) as g:
        g.load_topology(W.top_init([W.TYPES["psc"]], [n]))
        box = g.maxcut * (np.array(cells) + 0.3)
        rng = np.random.default_rng(n)
        d, q = axes(n, rng)
        g.set_config(box, rng.random((n, 3)), d, q, np.ones(n, np.int32))
        u = g.fixed_positions()
        cell_of, start, srt, nc = g.build_cells(r=1, shift=(777, 12345678, 99))
        c2, s2, o2 = po.cell_list(u, nc, (777, 12345678, 99))
        assert nc == cells
        np.testing.assert_array_equal(cell_of, c2)
        np.testing.assert_array_equal(start, s2)
        np.testing.assert_array_equal(srt, o2)


@pytest.mark.parametrize("n,rc", [(2, 0.87), (33, 0.87), (513, 0.87), (514, 0.87), (1100, 0.3), (1100, 0.12)])
def test_pair_list(n, rc):
    """rows of up to 512 partners and longer ones; rc of the box edge (0.87: every pair)"""
    say("case: pair list, %d particles, rc %.2f of the edge" % (n, rc))
    with sc_amd.GpuSystem(0) as g:
        g.load_topology(W.top_init([W.TYPES["psc"]], [n]))
        rng = np.random.default_rng(n)
        d, q = axes(n, rng)
        box = np.full(3, 20.0)
        g.set_config(box, rng.random((n, 3)), d, q, np.ones(n, np.int32))
        a, b = g.neighbor_pairs(rc * 20.0), po.neighbor_pairs(g.fixed_positions(), box, rc * 20.0)
        say("%d pairs, longest row %d" % (len(b), np.bincount(b[:, 0]).max() if len(b) else 0))
        if rc == 0.87:
            assert len(b) == n * (n - 1) // 2
        np.testing.assert_array_equal(a, b)


@pytest.mark.parametrize("m", [1, 255, 256, 257, 1000])
def test_pair_energies(m):
    """blocks of 256 pairs with every species in them, FP64 device mode"""
    say("case: %d pair energies" % m)
    z = np.load(os.path.join(GOLD, "pair_golden.npz"))
    st0 = po.State.from_real(z["mixed_box"], z["mixed_pos"], z["mixed_dir"], z["mixed_pd0"], z["mixed_types"])
    with sc_amd.GpuSystem(0) as g:
        g.load_topology(str(z["mixed_top"]))
        g.set_config(st0.box, st0.pos, st0.dir, st0.pd0, st0.types)
        b, p, dd, qq = g.get_config()
        tp, st = po.Topo(str(z["mixed_top"])), po.State(b, p, dd, qq, st0.types)
        k = np.random.default_rng(m).choice(len(z["mixed_i"]), m, replace=False)
        i, j = z["mixed_i"][k], z["mixed_j"][k]
        e, want = g.p2p(i, j, fp64=True), po.pair_energies(tp, st, i, j)
        rel = np.abs(e - want) / np.maximum(1.0, np.abs(want))
        say("max relative %.2e" % rel.max())
        assert np.mean(rel > 1e-9) <= 2e-3   # degenerate-branch pairs


@pytest.mark.parametrize("n", [1, 257, 16385])
def test_nematic_order(n):
    """one block, and more particles than the grid has threads"""
    say("case: S2 of %d axes" % n)
    with sc_amd.GpuSystem(0) as g:
        g.load_topology(W.top_init([W.TYPES["psc"]], [n]))
        rng = np.random.default_rng(n)
        d, q = axes(n, rng)
        g.set_config(np.full(3, 100.0), rng.random((n, 3)), d, q, np.ones(n, np.int32))
        s2 = g.nematic_order()[0]
        say("%.9f" % s2)
        assert s2 == pytest.approx(po.nematic_s2(g.get_config()[2]), abs=1e-6)


@pytest.mark.parametrize("rows", [1, 31, 32, 33, 16385])
def test_network_outputs(rows):
    """tiles of 32 rows and more rows than the grid has tiles"""
    say("case: FP32 network on %d rows" % rows)
    with sc_amd.GpuSystem(0) as g:
        g.load_topology(W.top_init([W.TYPES["tchpsc"]], [10]))
        g.mlp_init(3, seed=11)
        x = np.random.default_rng(rows).normal(size=(rows, mo.NF)).astype(np.float32)
        out, ref = g.mlp_forward(x, bf16=False), mo.forward(g.mlp_get_weights().astype(np.float64), x)
        say("max error %.2e" % np.abs(out - ref).max())
        assert np.abs(out - ref).max() <= 1e-5 * max(1.0, np.abs(ref).max())


@pytest.mark.parametrize("batch", [1, 31, 33, 255, 257])
def test_network_gradients(batch):
    """remainders of the blocks' tiles"""
    say("case: network gradients of %d rows" % batch)
    with sc_amd.GpuSystem(0) as g:
        g.load_topology(W.top_init([W.TYPES["tchpsc"]], [10]))
        g.mlp_init(3, seed=12)
        rng = np.random.default_rng(batch)
        x, y = rng.normal(size=(batch, mo.NF)).astype(np.float32), rng.normal(size=batch).astype(np.float32)
        grad, loss = g.mlp_gradients(x, y)
        lo, want = mo.loss_and_grad(g.mlp_get_weights().astype(np.float64), x, y)
        assert loss == pytest.approx(lo, rel=1e-5)
        cuts = [mo.OFF_W1, mo.OFF_B1, mo.OFF_W2, mo.OFF_B2, mo.OFF_W3, mo.OFF_B3, mo.OFF_W4, mo.OFF_B4, mo.NPARAM]
        for a, b in zip(cuts, cuts[1:]):
            assert np.abs(grad[a:b] - want[a:b]).max() <= 2e-4 * np.abs(want[a:b]).max() + 1e-9


@pytest.mark.parametrize("eta,r,visit,cap", [(0.02, 1, 1, None), (0.10, 1, 8, None), (0.10, 1, 8, 0), (0.10, 1, 8, 4),
                                             (0.25, 1, 8, None), (0.25, 2, 9, None), (0.25, 2, 1, 4)])
def test_sweep_of_a_mixture(eta, r, visit, cap):
    """Stages copied in one pass or two, rows of derived vectors for every staged particle, for the home cell's
    or for none: the one-trial-at-a-time trajectory bit for bit.  PSC, CPSC and TCHPSC: every kind of pair."""
    say("case: sweep of a mixture, eta %.2f, r %d, visit %d, home cache %s" % (eta, r, visit, cap))
    types = np.repeat([1, 2, 3], 400).astype(np.int32)
    vol = sum(400 * W.particle_volume(1.0, l) for l in (3.0, 3.0, 4.0))
    start = np.full(3, (vol / min(eta, 0.13)) ** (1.0 / 3.0))
    box = np.full(3, (vol / eta) ** (1.0 / 3.0))
    top = W.top_init([W.TYPES[k] for k in ("psc", "cpsc", "tchpsc")], [400] * 3)
    out = []
    for nw in (0, 1):
        with sc_amd.GpuSystem(0) as g:
            g.load_topology(top)
            pos, d, q = g.generate_rsa(types, start, 3)
            g.set_config(start, pos, d, q, types)
            for k in range(1, 9):   # shrunk in steps (the first sweeps resolve what overlaps)
                g.update_box(start * (box / start) ** (k / 8.0))
                g.sweep(5, 1.0, 0.3, ROT_HALF, r=1, seed=4, counter=10 * k)
            if cap is not None:
                g.set_home_cache(cap)
            g.set_trial_mode(1)
            g.set_visit_factor(visit)
            g.set_block_waves(nw)
            e0 = g.allToAll()
            s = g.sweep(10, 1.0, 0.3, ROT_HALF, r=r, seed=7, counter=1000)
            e1 = g.allToAll()
            assert abs(e1 - e0 - s["energy_change"]) <= 1e-8 * max(abs(e0), abs(e1), 1.0)
            out.append((s, g.get_config()))
    (s1, c1), (s2, c2) = out
    say("accepted %d / %d" % (s1["trans_acc"] + s1["rot_acc"], s1["trans_try"] + s1["rot_try"]))
    assert s1["trans_acc"] + s1["rot_acc"] > 0
    for k in ("trans_acc", "trans_try", "rot_acc", "rot_try", "left_cell"):
        assert s1[k] == s2[k], k
    for a, b in zip(c1, c2):
        np.testing.assert_array_equal(a, b)


@pytest.mark.parametrize("nchains", [30, 400])
def test_chain_moves_of_few_molecules(nchains):
    """few molecules per coarse cell and 27 visits: the molecule proposed beside a move is often the one that moved"""
    say("case: chain moves, %d chains" % nchains)
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
        say("E %.6f -> %.6f, sum dE %.6f; %s" % (e0, e1, s["energy_change"],
                                                 {k: v for k, v in s.items() if k.startswith("chain")}))
        assert abs(e1 - e0 - s["energy_change"]) <= 1e-8 * max(abs(e0), abs(e1), 1.0)
