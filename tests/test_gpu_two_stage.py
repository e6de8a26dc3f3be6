"""Every compiled plan of the register-resident FFT passes against the FP64 oracle: as
the last axis (fused z pass, one and two types and a charge field), as the film's last
axis, and as the sides of a square plane (plane passes); and the plans of grouped stages
against the LDS-staged passes, bit for bit."""
import numpy as np
import pytest

import decks
import gpu_util as U
import oracle_ctypes as O
import tild
import tild_gen

pytestmark = pytest.mark.gpu

# points of the compiled plans
LENGTHS = [21, 24, 25, 27, 28, 30, 32, 35, 36, 40, 45, 48, 50, 54, 60, 63, 64, 72, 75, 80, 90, 96, 100, 108, 120, 125,
           128, 144, 150, 160, 180, 192, 200, 216, 225, 240]


def _check(text, d, want_last=1):
    s = tild.System(text, d)
    e = tild.Engine(s, device=0, seed=7)
    o = O.System(text, d, seed=7)
    g = e.geometry()
    assert g["last_reg"] == want_last, g
    ef = U.rel_norm(e.forces(), o.forces())
    p, po = e.properties(), o.properties()
    eu = abs(p["Upe"] - po["Upe"]) / abs(po["Upe"])
    print(f"{s.grid_shape}: |df|/|f| {ef:.2e}, Upe {eu:.2e}")
    e.close()
    # the engine's force and energy tolerance against the oracle
    assert ef < 1e-5 and eu < 1e-5
    return g


@pytest.mark.parametrize("n", LENGTHS)
def test_last_axis(n, tmp_path):
    _check(*decks.melt3d(tmp_path / "3d", grid=(9, 8, n), box=(4.5, 4.0, 0.5 * n), n_chains=n))
    _check(*decks.melt2d(tmp_path / "2d", grid=(18, n), box=(9.0, 0.5 * n), n_chains=n))


@pytest.mark.parametrize("n", [27, 45, 96, 180, 225])
def test_last_axis_charged(n, tmp_path):
    # one type and a charge field: polycations and polyanions of the same type
    d = tmp_path
    rng = np.random.default_rng(n)
    box = (4.5, 4.0, 0.5 * n)
    pos, types, mols, bonds = tild_gen.diblock(rng, n, 10, 0.5, box, 3)
    types = np.ones_like(types)
    tild_gen.write_data(d / "input.data", pos, types, mols, bonds, box, 1, 3, charges=np.where(mols % 2 == 0, 1.0, -1.0))
    text = tild_gen.deck("input.data", 3, (9, 8, n), [("gaussian", 1, 1, 0.5, 0.5)], "EM", 0.005, 3, charges=(1.0, 0.7))
    _check(text, d)


# lengths whose passes stand for the LDS-staged ones with the same roundings: forward plane
# pass or y pass (odd sides), inverse plane pass of one and two fields with 512 and 1,024
# threads or y inverse and x pass, fused z pass of each order of the groups
@pytest.mark.parametrize("ntypes", [1, 2])
@pytest.mark.parametrize("grid", [(21, 21, 21), (27, 27, 54), (45, 45, 60), (54, 54, 9), (72, 72, 27), (75, 75, 9), (90, 90, 9),
                                  (96, 96, 28), (108, 108, 9), (45, 36, 60), (36, 45, 96), (60, 96, 108), (20, 18, 120),
                                  (120, 20, 125), (18, 125, 144), (20, 18, 180), (144, 18, 192), (18, 144, 200),
                                  (20, 18, 216), (225, 18, 225), (18, 20, 240)])
def test_equals_staged(grid, ntypes, tmp_path):
    rng = np.random.default_rng(sum(grid))
    box = tuple(0.5 * g for g in grid)
    pos, types, mols, bonds = tild_gen.diblock(rng, 300, 10, 0.5, box, 3)
    if ntypes == 1:
        types = np.ones_like(types)
    tild_gen.write_data(tmp_path / "input.data", pos, types, mols, bonds, box, ntypes, 3)
    styles = [("gaussian", 1, 1, 0.5, 0.5), ("gaussian", 2, 2, 0.5, 0.5), ("gaussian", 1, 2, 0.7, 0.5)][:1 if ntypes == 1 else 3]
    s = tild.System(tild_gen.deck("input.data", 3, grid, styles, "EM", 0.005, 3), tmp_path)
    f = []
    for staged in (False, True):
        e = tild.Engine(s, device=0, seed=7, fft_staged=staged)
        assert e.geometry()["last_reg"] == (0 if staged or grid[2] == 9 else 1)
        e.step(3)
        f.append([e.forces(), e.positions()] + [e.grid_field(t, a) for t in range(e.nfields) for a in range(3)])
        e.close()
    assert all(np.array_equal(a, b) for a, b in zip(*f))


@pytest.mark.parametrize("n", [n for n in LENGTHS if n <= 128])
def test_square_plane(n, tmp_path):
    g = _check(*decks.melt3d(tmp_path, grid=(n, n, 8), box=(0.5 * n, 0.5 * n, 4.0), n_chains=4 * n), want_last=0)
    assert g["grad_reg"] == 1
