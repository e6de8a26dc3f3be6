"""Assignment orders 0 and 2-4: the tiled deposit's unrolled position records and the
gather's z slabs, against the FP64 oracle and against the global-atomic spread."""
import numpy as np
import pytest

import decks
import gpu_util as U
import oracle_ctypes as O
import tild

pytestmark = pytest.mark.gpu

GRIDS = {"3d": (20, 16, 24), "3d_odd": (25, 27, 30), "2d": (40, 48)}


@pytest.mark.parametrize("grid", list(GRIDS))
@pytest.mark.parametrize("order", [0, 2, 3, 4])
def test_order(order, grid, tmp_path):
    g = GRIDS[grid]
    box = tuple(0.5 * n for n in g)
    mk = decks.melt3d if len(g) == 3 else decks.melt2d
    text, d = mk(tmp_path, grid=g, box=box, n_chains=150, pmeorder=order)
    s = tild.System(text, d)
    tiled, atomic = tild.Engine(s, device=0, seed=3), tild.Engine(s, device=0, seed=3, spread_mode=1)
    o = O.System(text, d, seed=3)
    x = s.positions()
    x[:6] = [np.zeros(s.dim), np.array(box), 0.5 * np.ones(s.dim), np.array(box) - 0.25, 1e-6 * np.ones(s.dim),
             np.array(box) - 0.5]   # on the faces, on nodes and between them
    for e in (tiled, atomic):
        e.set_positions(x)
    o.set_positions(x.astype(np.float64))
    f, fa, fo = tiled.forces(), atomic.forces(), o.forces()
    for t in range(s.ntypes):   # both spreads round each weight to the same integer
        assert np.array_equal(tiled.density(t), atomic.density(t)), t
        ro = o.density(t)
        assert np.abs(tiled.density(t) - ro).max() < 2e-6 * np.abs(ro).max()
    ef = U.rel_norm(f, fo)
    print(f"order {order} {g}: |df|/|f| {ef:.2e}")
    # the engine's force tolerance against the oracle; order 0's force jumps where a bead
    # changes its node, which FP32 and FP64 decide alike (bins are FP32 in both)
    assert ef < 1e-5
    tiled.step(5)
    atomic.step(5)
    assert np.abs(U.min_image(tiled.positions().astype(np.float64) - atomic.positions(), np.array(box))).max() < 1e-4
    for e in (tiled, atomic):
        e.close()


def test_mixed_orders_in_a_batch(tmp_path):
    # replicas of several orders share the launches: each keeps the bits it has alone
    sys_ = []
    for order in (0, 1, 2, 3, 4):
        text, d = decks.melt3d(tmp_path / f"o{order}", grid=(16, 20, 24), box=(8.0, 10.0, 12.0), n_chains=100,
                               pmeorder=order)
        sys_.append(tild.System(text, d))
    b = tild.Batch(device=0)
    ids = [b.add(s, 5 + k) for k, s in enumerate(sys_)]
    b.step(7)
    for k, s in enumerate(sys_):
        e = tild.Engine(s, device=0, seed=5 + k)
        e.step(7)
        assert np.array_equal(b.positions(ids[k]), e.positions()), k
        e.close()
    b.close()


@pytest.mark.parametrize("dim", [2, 3])
@pytest.mark.parametrize("order", [0, 2, 3, 4])
def test_positions_without_a_place_deposit_alike(order, dim, tmp_path):
    # a coordinate that is not a number, infinite, or so large that its FP32 offset from the
    # node has no meaning still has a node (every index is wrapped) and weights, and both
    # spreads round those to the same integers, as for any other bead
    g = (20, 16, 24)[:dim]
    mk = decks.melt3d if dim == 3 else decks.melt2d
    text, d = mk(tmp_path, grid=g, box=tuple(0.5 * n for n in g), n_chains=150, pmeorder=order)
    s = tild.System(text, d)
    tiled, atomic = tild.Engine(s, device=0, seed=3, spread_mode=2), tild.Engine(s, device=0, seed=3, spread_mode=1)
    for bad in (np.nan, np.inf, -np.inf, 1e9, -3e7):
        for axis in range(dim):
            x = s.positions()
            x[5, axis] = bad
            rho = []
            for e in (tiled, atomic):
                e.set_positions(x)
                e.forces()
                rho.append([e.density(t) for t in range(s.ntypes)])
            for a, b in zip(*rho):
                assert np.array_equal(a, b, equal_nan=True), (bad, axis)
    tiled.close()
    atomic.close()
