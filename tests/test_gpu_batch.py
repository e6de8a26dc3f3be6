"""Batched replicas: results equal each replica run alone; graph replays equal eager steps."""
import numpy as np
import pytest

import decks
import tild
import tild_gen

pytestmark = pytest.mark.gpu


def _decks(tmp):
    out = []
    out.append(decks.melt3d(tmp / "a", n_chains=40, N=10, box=(6.0, 6.0, 6.0), grid=(12, 12, 12)))
    out.append(decks.melt3d(tmp / "b", n_chains=30, N=20, box=(7.5, 7.5, 9.0), grid=(15, 15, 18),
                            integrator="GJF", delt=0.01, styles=decks.MIXED))
    out.append(decks.melt2d(tmp / "c"))
    out.append(decks.charged(tmp / "d"))
    out.append(decks.melt3d(tmp / "e", n_chains=20, N=10, box=(6.0, 5.0, 7.0), grid=(12, 10, 14), pmeorder=2))
    return out


@pytest.mark.parametrize("graph", [False, True])
def test_batch_equals_alone(graph, tmp_path):
    systems = [(tild.System(t, d), d) for t, d in _decks(tmp_path)]
    alone = []
    for i, (s, _) in enumerate(systems):
        e = tild.Engine(s, device=0, seed=100 + i)
        e.step(67)
        alone.append((e.positions(), e.density(0), e.properties()))
        e.close()
    b = tild.Batch(device=0)
    ids = [b.add(s, 100 + i) for i, (s, _) in enumerate(systems)]
    b.step(3, graph=graph)
    b.step(64, graph=graph)   # with graph: one replay of the 60-step graph, then 4 eager steps
    for i, r in enumerate(ids):
        assert b.replica_step(r) == 67
        assert np.array_equal(b.positions(r), alone[i][0]), i
        assert np.array_equal(b.density(r, 0), alone[i][1]), i
        p = b.properties(r)
        assert p["Upe"] == alone[i][2]["Upe"], i
    print(f"{len(ids)} uneven replicas (graph={graph}): positions, densities, energies bit-identical to runs alone")
    b.close()


def test_graph_replays_match_eager_with_interleaved_work(tmp_path):
    systems = [(tild.System(t, d), d) for t, d in _decks(tmp_path)[:3]]
    ref = tild.Batch(device=0)
    gb = tild.Batch(device=0)
    rids = [ref.add(s, 7 + i) for i, (s, _) in enumerate(systems)]
    gids = [gb.add(s, 7 + i) for i, (s, _) in enumerate(systems)]
    # runs of 60 or more steps replay the 60-step graph, the rest run eagerly
    for rep, n in enumerate([2, 130, 2, 61]):
        ref.step(n, graph=False)
        gb.step(n, graph=True)
        # eager work and synchronisation between replays
        for r in gids:
            gb.properties(r)
        for a, c in zip(rids, gids):
            assert np.array_equal(ref.positions(a), gb.positions(c)), (rep, a)
    ref.close()
    gb.close()


def test_batch_subsets_and_removal(tmp_path):
    systems = [(tild.System(t, d), d) for t, d in _decks(tmp_path)[:3]]
    b = tild.Batch(device=0)
    ids = [b.add(s, 3) for s, _ in systems]
    b.step(2, replicas=[ids[0], ids[2]])
    assert [b.replica_step(r) for r in ids] == [2, 0, 2]
    b.remove(ids[1])
    b.step(1)
    assert b.replica_step(ids[0]) == 3 and b.replica_step(ids[2]) == 3
    r3 = b.add(systems[1][0], 3)
    b.step(1)
    assert b.replica_step(r3) == 1
    b.close()


@pytest.mark.parametrize("which", ["tiled", "mixed"])
def test_batched_spatial_reorder_is_invisible(which, tmp_path):
    # replicas due for their spatial reorder at the same step are reordered together
    # (one launch per kernel for the set) when all use the tiled spread, one by one
    # otherwise; either way positions are bit-identical to never reordering and the
    # FP64 energies equal to rounding (they sum the beads in another slot order)
    alld = _decks(tmp_path)
    chosen = [alld[0], alld[1], alld[3]] if which == "tiled" else alld
    systems = [tild.System(t, d) for t, d in chosen]
    out = []
    for every in (3, -1):
        # the tiled set is forced onto the tiled spread, so the set-wide reorder runs
        b = tild.Batch(device=0, reorder_every=every, spread_mode=2 if which == "tiled" else 0)
        ids = [b.add(s, 40 + i) for i, s in enumerate(systems)]
        b.step(4, graph=True)
        b.step(9, graph=True)
        b.step(2, graph=False)
        out.append([(b.positions(r), b.properties(r)) for r in ids])
        b.close()
    for i, ((xa, pa), (xb, pb)) in enumerate(zip(*out)):
        assert np.array_equal(xa, xb), (which, i)
        assert abs(pa["Upe"] - pb["Upe"]) <= 1e-12 * abs(pb["Upe"]), (which, i)
    print(f"[{which}] {len(systems)} replicas reordered every 3 steps: positions bit-identical to never reordering")


def test_square_planes_keep_their_bits_in_a_mixed_set(tmp_path):
    # with a rectangular or an odd-sided replica in the set, the forward plane pass is a
    # kernel that holds every form; square planes run the same transform in it
    grids = [(n, n, 10) for n in (24, 30, 32, 40, 48, 50, 64, 80, 128)] + [(36, 30, 10), (25, 27, 10)]
    systems = []
    for k, g in enumerate(grids):
        t, d = decks.melt3d(tmp_path / str(k), grid=g, box=tuple(0.5 * n for n in g), n_chains=5 * g[0], delt=0.02)
        systems.append(tild.System(t, d))
    b = tild.Batch(device=0)
    ids = [b.add(s, 20 + k) for k, s in enumerate(systems)]
    b.step(8)
    for k, s in enumerate(systems):
        e = tild.Engine(s, device=0, seed=20 + k)
        e.step(8)
        assert np.array_equal(b.positions(ids[k]), e.positions()), grids[k]
        e.close()
    b.close()


def test_y_inverse_keeps_its_bits_in_a_mixed_set(tmp_path):
    # planes without an inverse plane pass: with a y plan of grouped stages in the set the y
    # inverse is a kernel that holds every plan
    grids = [(20, n, 9) for n in (24, 25, 30, 32, 40, 48, 50, 64, 80, 128, 160)] + [(20, 36, 9), (20, 125, 9)]
    systems = []
    for k, g in enumerate(grids):
        t, d = decks.melt3d(tmp_path / str(k), grid=g, box=tuple(0.5 * n for n in g), n_chains=4 * g[1], delt=0.02)
        systems.append(tild.System(t, d))
    b = tild.Batch(device=0)
    ids = [b.add(s, 20 + k) for k, s in enumerate(systems)]
    b.step(8)
    for k, s in enumerate(systems):
        e = tild.Engine(s, device=0, seed=20 + k)
        assert e.geometry()["grad_reg"] == 1
        e.step(8)
        assert np.array_equal(b.positions(ids[k]), e.positions()), grids[k]
        e.close()
    b.close()


def test_x_c2r_keeps_its_bits_in_a_mixed_set(tmp_path):
    # films and planes without an inverse plane pass: with an x plan of grouped stages in the
    # set the x C2R is a kernel that holds every plan
    grids = [(n, 36) for n in (21, 24, 25, 30, 32, 40, 48, 50, 64, 80, 100, 128, 160)] + [(100, 128, 9), (64, 256, 9)]
    grids += [(96, 40), (225, 40), (120, 128, 9)]
    systems = []
    for k, g in enumerate(grids):
        mk = decks.melt3d if len(g) == 3 else decks.melt2d
        t, d = mk(tmp_path / str(k), grid=g, box=tuple(0.5 * n for n in g), n_chains=3 * g[0], delt=0.02)
        systems.append(tild.System(t, d))
    b = tild.Batch(device=0)
    ids = [b.add(s, 20 + k) for k, s in enumerate(systems)]
    b.step(8)
    for k, s in enumerate(systems):
        e = tild.Engine(s, device=0, seed=20 + k)
        e.step(8)
        assert np.array_equal(b.positions(ids[k]), e.positions()), grids[k]
        e.close()
    b.close()


@pytest.mark.parametrize("other", ["long_axis", "three_types"])
def test_last_axis_keeps_its_bits_in_a_mixed_set(other, tmp_path):
    # short axes of one or two types run the fused last-axis pass in the kernel of the longer
    # axes, or of the larger type counts, that share their set
    def deck(d, grid, ntypes, charged):
        box = tuple(0.5 * n for n in grid) + ((1.0,) if len(grid) == 2 else ())
        d.mkdir()
        pos, types, mols, bonds = tild_gen.diblock(np.random.default_rng(grid[-1]), 150, 10, 0.5, box, len(grid))
        types = 1 + np.arange(len(types)) % ntypes
        styles = [("gaussian", i, j, 0.5 + 0.2 * i * j, 0.5) for i in range(1, ntypes + 1) for j in range(i, ntypes + 1)]
        q = np.where(mols % 2 == 0, 1.0, -1.0) if charged else None
        tild_gen.write_data(d / "input.data", pos, types, mols, bonds, box, ntypes, len(grid), charges=q)
        return tild.System(tild_gen.deck("input.data", len(grid), grid, styles, "EM", 0.02, 3,
                                         **(dict(charges=(1.0, 0.7)) if charged else {})), d)

    cases = [((20, 18, n), 1 + k % 2, k % 3 == 0) for k, n in enumerate((24, 25, 27, 30, 32, 36, 40, 45, 48, 50, 64, 80, 96))]
    cases += [((18, n), 1 + k % 2, k % 3 == 1) for k, n in enumerate((24, 30, 48, 50, 64, 72, 80, 100))]
    cases += {"long_axis": [((20, 18, 128), 2, False), ((18, 160), 1, True)],
              "three_types": [((20, 18, 40), 3, False), ((18, 64), 4, True)]}[other]
    systems = [deck(tmp_path / str(k), *c) for k, c in enumerate(cases)]
    b = tild.Batch(device=0)
    ids = [b.add(s, 20 + k) for k, s in enumerate(systems)]
    b.step(8)
    for k, s in enumerate(systems):
        e = tild.Engine(s, device=0, seed=20 + k)
        assert e.geometry()["last_reg"] == 1
        e.step(8)
        assert np.array_equal(b.positions(ids[k]), e.positions()), cases[k]
        e.close()
    b.close()


@pytest.mark.parametrize("grids", [
    [(24, 32, 40), (20, 32, 40)], [(40, 80, 24), (20, 40, 24)], [(36, 36, 36), (20, 20, 20)], [(27, 27, 27), (20, 20, 20)],
    [(45, 36, 20), (20, 40, 24)], [(25, 30, 20), (15, 25, 30)], [(48, 80, 9), (20, 50, 9), (25, 25, 9)],
    [(128, 64, 9), (64, 128, 9), (20, 20, 9)], [(100, 128, 9), (125, 160, 9), (20, 25, 9)], [(64, 64), (96, 96), (20, 20)],
    [(160, 40), (225, 40), (24, 30, 20), (250, 20)], [(24, 24, 24), (24, 32, 20), (20, 32, 20)],
], ids=lambda g: "_".join("x".join(map(str, k)) for k in g))
def test_sides_with_and_without_a_compiled_plan_share_a_set(grids, tmp_path):
    # in small sets the register forms join the staged launches of the replicas that have no
    # other; each replica keeps the bits it has alone
    systems = []
    for k, g in enumerate(grids):
        mk = decks.melt3d if len(g) == 3 else decks.melt2d
        t, d = mk(tmp_path / str(k), grid=g, box=tuple(0.5 * n for n in g), n_chains=200, delt=0.02)
        systems.append(tild.System(t, d))
    b = tild.Batch(device=0)
    ids = [b.add(s, 20 + k) for k, s in enumerate(systems)]
    b.step(8, graph=False)
    b.step(70, graph=True)
    for k, s in enumerate(systems):
        e = tild.Engine(s, device=0, seed=20 + k)
        e.step(78)
        assert np.array_equal(b.positions(ids[k]), e.positions()), grids[k]
        assert all(np.array_equal(b.density(ids[k], t), e.density(t)) for t in range(s.ntypes))
        e.close()
    b.close()
