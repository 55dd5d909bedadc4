"""pp_time_kernel times the launches that the solve smooths a level with: one
colour of the lines each, or both on small levels; the work arrays it overwrites
do not change a later solve."""
import numpy as np
import pytest

import cases
from flow_structure_interaction_fem_ibm_amd import pp
from test_gpu_line_shapes import sphere
from test_gpu_split import announce

pytestmark = pytest.mark.gpu


# (grid, level, colours per launch): 36864 cells and lines of 66 take one
@pytest.mark.parametrize("grid,level,colours", [
    ((24, 24, 24), 0, 2), ((25, 27, 26), 0, 2), ((64, 32, 16), 0, 2), ((64, 48, 48), 1, 2),
    ((64, 48, 48), 0, 1), ((48, 32, 24), 0, 1), ((66, 20, 24), 0, 1),
], ids=str)
def test_bytes_of_a_launch(grid, level, colours):
    announce(f"time_kernel {grid} level {level}")
    _, ib, _, s = sphere(*grid)
    b = cases.random_field(ib.shape, 3, ib)
    ref = np.zeros(ib.shape)
    s.solve(ref, b, rel_tol=1e-9)
    cells = float(np.prod(s.level_info()[level]))
    for prec, elem in ((pp.PP_PREC_MIXED, 4), (pp.PP_PREC_FP64, 8)):
        for cls in ("xline", "yline", "zline"):
            us, got = s.time_kernel(cls, level, prec, 5)
            assert us > 0 and got == pytest.approx(cells * (3 * elem + 1) * 0.5 * colours)
    p = np.zeros(ib.shape)
    s.solve(p, b, rel_tol=1e-9)
    assert np.array_equal(p, ref)
