"""Which register-resident forms of the FFT passes a replica runs, and that they give the bits of
the LDS-staged passes they stand for: films, charges, one to four types, uneven planes."""
import numpy as np
import pytest

import tild
import tild_gen

pytestmark = pytest.mark.gpu


def _system(d, grid, ntypes, charged):
    dim = len(grid)
    box = tuple(0.5 * n for n in grid) + ((1.0,) if dim == 2 else ())
    pos, types, mols, bonds = tild_gen.diblock(np.random.default_rng(sum(grid)), 300, 10, 0.5, box, dim)
    types = 1 + np.arange(len(types)) % ntypes
    styles = [("gaussian", i, j, 0.4 + 0.2 * i * j, 0.5) for i in range(1, ntypes + 1) for j in range(i, ntypes + 1)]
    q = np.where(mols % 2 == 0, 1.0, -1.0) if charged else None
    tild_gen.write_data(d / "input.data", pos, types, mols, bonds, box, ntypes, dim, charges=q)
    kw = dict(charges=(1.0, 0.7)) if charged else {}
    return tild.System(tild_gen.deck("input.data", dim, grid, styles, "EM", 0.005, 3, **kw), d)


# grid, types, charges, and the forms: fused last axis, plane_rect, yfwd_reg, plane_pair, c2r_reg.
# The last axes are none whose z pass fuses its products otherwise (24, 25, 30, 32, 40, 48, ...).
FILM = [((27, 45), 1, False), ((63, 54), 2, False), ((36, 100), 3, False), ((45, 60), 4, False), ((96, 240), 2, False),
        ((225, 72), 2, False), ((216, 96), 1, True), ((125, 144), 2, True), ((64, 45), 2, False), ((80, 96), 3, True),
        ((128, 63), 4, True), ((160, 27), 2, False), ((100, 75), 2, False), ((200, 90), 1, False)]
BOX = [((45, 36, 60), 1, True, 0), ((36, 45, 27), 4, True, 0), ((54, 27, 36), 3, False, 0),
       ((24, 32, 27), 2, False, 0), ((48, 64, 27), 2, False, 0), ((80, 40, 36), 1, True, 0),
       ((36, 30, 45), 4, False, 0), ((25, 24, 27), 3, True, 0), ((100, 128, 21), 2, False, 1),
       ((108, 100, 27), 1, True, 1), ((80, 160, 21), 3, False, 1)]


def _compare(s, geometry, passes):
    out = []
    for staged in (False, True):
        e = tild.Engine(s, device=0, seed=7, fft_staged=staged)
        g, p = e.geometry(), e.passes()
        if staged:
            assert not any(p.values()) and g["last_reg"] == 0, (g, p)
        else:
            assert {k: g[k] for k in geometry} == geometry and {k: p[k] for k in passes} == passes, (g, p)
        e.step(3)
        out.append([e.forces(), e.positions()] + [e.grid_field(t, a) for t in range(e.nfields) for a in range(s.dim)])
        e.close()
    assert all(np.array_equal(a, b) for a, b in zip(*out))


@pytest.mark.parametrize("grid,ntypes,charged", FILM)
def test_film_equals_staged(grid, ntypes, charged, tmp_path):
    last = int(ntypes <= (2 if grid[1] > 100 else 4))
    _compare(_system(tmp_path, grid, ntypes, charged), {"last_reg": last},
             {"plane_rect": 0, "yfwd_reg": 0, "plane_pair": 0, "c2r_reg": 1})


@pytest.mark.parametrize("grid,ntypes,charged,c2r", BOX)
def test_box_equals_staged(grid, ntypes, charged, c2r, tmp_path):
    _compare(_system(tmp_path, grid, ntypes, charged), {"last_reg": 1, "plane_reg": 0, "plane_inv": 0},
             {"plane_rect": int(grid[1] % 2 == 0), "yfwd_reg": int(grid[1] % 2 == 1), "plane_pair": 1 - c2r, "c2r_reg": c2r})


# in boxes the x C2R of 125 and 160 points runs staged, where that form is the faster one
@pytest.mark.parametrize("grid,c2r", [((125, 100, 9), 0), ((160, 80, 9), 0), ((120, 128, 9), 1), ((125, 27), 1), ((160, 27), 1)])
def test_x_c2r_rule(grid, c2r, tmp_path):
    _compare(_system(tmp_path, grid, 2, False), {"last_reg": int(len(grid) == 2)}, {"c2r_reg": c2r})


@pytest.mark.parametrize("n", [24, 25, 30, 32, 40, 48, 50, 64, 80, 128, 160])
def test_y_inverse_equals_staged(n, tmp_path):
    # the lengths whose z pass differs: the y passes of planes without plane passes do not
    _compare(_system(tmp_path, (20, n, 9), 2, False), {"last_reg": 0, "plane_reg": 0, "plane_inv": 0, "grad_reg": 1},
             {"plane_rect": 0, "yfwd_reg": n % 2, "plane_pair": 0, "c2r_reg": 0})


# the x transform of the deposit: staged for films of 80 and 160 points, whose staged form is the
# faster one, in registers for other compiled plans; none with the forward plane pass
@pytest.mark.parametrize("grid,xreg", [((80, 27), 0), ((160, 45), 0), ((64, 27), 1), ((128, 45), 1), ((100, 27), 1),
                                       ((80, 45, 21), 1), ((160, 27, 21), 1), ((80, 36, 21), 0), ((20, 45), 0)])
def test_deposit_x_transform_rule(grid, xreg, tmp_path):
    _compare(_system(tmp_path, grid, 2, False), {}, {"deposit_xreg": xreg})
