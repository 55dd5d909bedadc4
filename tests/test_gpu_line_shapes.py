"""The pressure line passes at every segment length and tile width their
launch rule takes: after one pass set with omega = 1 the lines solved last
(z-lines of the second colour) satisfy their rows exactly, by the oracle's
calc_residual; and the FP32 passes on the colour-split rows give the solves of
the natural-layout ones bit for bit on shapes that reach the long segments."""
import numpy as np
import pytest

import cases
from flow_structure_interaction_fem_ibm_amd import pp
from oracle_lib import Oracle
from test_gpu_split import announce, assert_same, both_layouts

pytestmark = pytest.mark.gpu


def sphere(nx, ny, nz):
    """Cells of about 1/64 in every direction, one sphere."""
    nodes = [pp.tanh_nodes(n, n / 64.0, b) for n, b in ((nx, 1.0), (ny, 0.8), (nz, 1.2))]
    L = [a[-1] for a in nodes]
    r = 0.3 * min(L)
    ib, _, gs, _ = pp.build_geometry(*nodes, [pp.Ellipsoid((0.5 * L[0], 0.47 * L[1], 0.53 * L[2]), (r, r, r), 0.0, 24)],
                                     mode=pp.PP_GEOM_ANALYTIC)
    s = pp.PressureSolver(*nodes)
    s.set_geometry(ib, gs)
    return nodes, ib, gs, s


@pytest.mark.parametrize("shape", [
    (20, 30, 15), (20, 30, 31), (21, 29, 127), (20, 30, 250), (18, 22, 600), (12, 20, 1000),  # few blocks: 1-16 cells
    (66, 500, 100), (64, 520, 141), (72, 480, 200),                                           # 8, 12 and 16 cells
], ids=str)
def test_last_lines_of_a_pass_satisfy_their_rows(shape):
    announce(f"one FP64 line pass set {shape}")
    nodes, ib, gs, s = sphere(*shape)
    o = Oracle(*nodes)
    o.set_iblank(ib)
    o.set_stencils(gs)
    e, b = cases.random_field(ib.shape, 5), cases.random_field(ib.shape, 6, ib)
    out = s.smooth(e, b, smoother=pp.PP_SMOOTH_LINE, omega=1.0, sweeps=1)
    res = o.calc_residual(out, b)[0]
    k, j, i = np.meshgrid(*[np.arange(n - 3) for n in ib.shape], indexing="ij")
    solved = ((i + j) % 2 == 1) & (cases.interior(ib) == 0)
    # backward stable elimination: a few dozen roundings of the row's largest term
    dmax = sum(4.0 / np.diff(a).min() ** 2 for a in nodes) * np.abs(out).max()
    assert np.abs(cases.interior(res)[solved]).max() <= 1e-12 * dmax


@pytest.mark.parametrize("shape", [(64, 260, 514), (500, 40, 24)], ids=str)
def test_long_segments_agree_between_layouts(shape):
    announce(f"split vs natural {shape}")
    _, ib, gs, s = sphere(*shape)
    b = cases.random_field(ib.shape, 7, ib)
    assert_same(both_layouts(s, b, rel_tol=1e-9, max_outer=100))
