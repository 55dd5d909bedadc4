"""The momentum line passes at every segment length and tile width their
launch rule takes (pp_solve_ad): lines that do not fill their last segment,
odd and even row lengths, one-tile and many-tile planes, lines beyond 512
cells.  The converged fields are checked with the oracle's calc_residual_ad
(bit-exact with the library's, test_gpu_ad.py): a row solved with a wrong
neighbour, coefficient or line end does not reach the tolerance."""
import numpy as np
import pytest

import cases
from flow_structure_interaction_fem_ibm_amd import pp
from oracle_lib import Oracle
from test_gpu_ad import CN1, announce

pytestmark = pytest.mark.gpu


def setup(nx, ny, nz, dt):
    """Cells of about 1/64 in every direction, one sphere."""
    nodes = [pp.tanh_nodes(n, n / 64.0, b) for n, b in ((nx, 1.2), (ny, 0.9), (nz, 1.5))]
    L = [a[-1] for a in nodes]
    r = 0.3 * min(L)
    ib, _, gs, ex = pp.build_geometry(*nodes, [pp.Ellipsoid((0.5 * L[0], 0.47 * L[1], 0.53 * L[2]), (r, r, r), 0.0, 24)],
                                      mode=pp.PP_GEOM_ANALYTIC)
    s, o = pp.PressureSolver(*nodes), Oracle(*nodes)
    s.set_geometry(ib, gs)
    o.set_iblank(ib)
    o.set_stencils(gs)
    visc = np.full(o.shape, 0.01)
    for x in (s, o):
        x.set_vel_ghosts(ex["coeffD"], 2.0, 1.0)
    s.set_solve_ad(dt, visc, visc, visc, visc)
    return s, o, ib, gs, o.set_solve_ad(dt, visc, visc, visc, visc), np.random.default_rng(3)


@pytest.mark.parametrize("shape", [
    (21, 18, 17),      # few blocks: 2-cell segments in 4-line tiles
    (36, 100, 131),    # 4-cell segments in y, 2 in z
    (70, 150, 90),     # 16 in y, 4 in z
    (37, 129, 193),    # 16 in both, an odd row
    (14, 400, 258),
    (13, 520, 513),    # 16 in 8-line tiles
    (523, 13, 12),     # x-lines of 131 segments
], ids=str)
def test_line_segments_converge(shape):
    announce(f"solve_ad {shape}")
    dt = 1e-3
    s, o, ib, gs, coef, rng = setup(*shape, dt=dt)
    faces = [rng.standard_normal(ib.shape) * 0.5 for _ in range(3)]
    nl = [cases.random_field(ib.shape, 60 + q) for q in range(3)]
    u0 = [rng.standard_normal(ib.shape) * 0.1 for _ in range(3)]
    vbi = rng.standard_normal((gs.n, 3))
    u, v, w, st = s.solve_ad(CN1, *u0, *nl, *faces, vel_bi=vbi, itermax_ad=200, restol_ad=1e-12)
    assert st["status"] == "PP_OK", st
    for q, (got, r) in enumerate(zip((u, v, w), nl)):
        m, _, _ = o.calc_residual_ad(0.5 * dt, coef, faces, got, r)
        assert m <= 1e-12 and m == st["residual_uvw"][q]
        # blank cells off the ghosts are 0, the outer layer is the caller's
        solid = (ib == 1)
        solid.reshape(-1)[gs.ig + ib.shape[2] * (gs.jg + ib.shape[1] * gs.kg)] = False
        solid[[0, -1, -2]] = False
        solid[:, [0, -1, -2]] = False
        solid[:, :, [0, -1, -2]] = False
        assert not got[solid].any()
        assert np.array_equal(got[:, :, 0], u0[q][:, :, 0]) and np.array_equal(got[-2], u0[q][-2])
