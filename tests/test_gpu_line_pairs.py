"""GPU: line smoothing of small levels, where both colours of a direction run
in one launch: tiles of 8 x 4 lines cut short by the level, lines of one, two
and four cells per lane and one cell more or less, one step (whose z lines run
in place) and several, against the numpy restatement of the pass set; the
colour-split and the natural layout give the same solve bit for bit."""
import numpy as np
import pytest

import cases
from flow_structure_interaction_fem_ibm_amd import pp
from levels import Hierarchy
from test_gpu_levels import F32, F64, announce, close
from test_gpu_line_shapes import sphere
from test_gpu_split import assert_same, both_layouts

pytestmark = pytest.mark.gpu

GRIDS = [(16, 17, 18), (31, 33, 15), (32, 15, 48), (64, 20, 24), (15, 64, 33), (17, 14, 63), (25, 27, 26)]


@pytest.mark.parametrize("grid", GRIDS, ids=str)
def test_pass_set(grid):
    announce(f"pass set of a small level {grid}")
    nodes, ib, gs, s = sphere(*grid)
    ghost = np.zeros(ib.shape, bool)
    ghost[gs.kg, gs.jg, gs.ig] = True
    H = Hierarchy(*nodes, ib, ghost)
    rng = np.random.default_rng(8)
    shp = H.dims[0][::-1]
    gh = (H.flags[0] & 2) != 0
    for prec, tol in ((F64, 1e-10), (F32, 2e-4)):
        e = rng.standard_normal(shp) * (~H.blank[0] | gh)
        rhs = rng.standard_normal(shp) * ~H.blank[0]
        if prec == F32:
            e, rhs = e.astype(np.float32).astype(np.float64), rhs.astype(np.float32).astype(np.float64)
        for omega in (1.0, 1.3):
            got = s.level_apply(pp.PP_LOP_LINE_PASS, 0, e, rhs, precision=prec, omega=omega)
            assert close(got, H.line_pass(0, e, rhs, omega), tol), (prec, omega)
    # several steps: the z lines of all but the last in one launch as well
    ref = e
    pad = lambda a: np.pad(a, ((1, 2),) * 3)
    for sweeps in (1, 2, 3):
        ref = H.line_pass(0, ref, rhs, 1.3)
        got = s.smooth(pad(e), pad(rhs), smoother=pp.PP_SMOOTH_LINE, omega=1.3, sweeps=sweeps)
        assert close(got[1:-2, 1:-2, 1:-2], ref, 1e-10), sweeps


@pytest.mark.parametrize("shape", [(24, 24, 24), (64, 20, 24), (16, 36, 48)], ids=str)
def test_layouts_agree(shape):
    announce(f"split vs natural {shape}")
    _, ib, gs, s = sphere(*shape)
    b = cases.random_field(ib.shape, 7, ib)
    for nu in ({}, {"nu_pre": 1, "nu_post": 2}, {"nu_pre": 2, "nu_post": 0}, {"nu_pre": 0, "nu_post": 1}):
        assert_same(both_layouts(s, b, rel_tol=1e-9, max_outer=200, **nu))

