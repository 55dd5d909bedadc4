"""The momentum solve reads the outer layer's faces and, where a ghost stencil
reaches them, its edges; every other entry of the outer layer (its twelve edges,
its corners, the layer behind the upper faces) is the caller's own, and what it
holds does not reach the cells: lines that do not fill their last segment,
with NaN and infinities there, against zeros there, bit for bit."""
import numpy as np
import pytest

import cases
from flow_structure_interaction_fem_ibm_amd import pp
from test_gpu_ad import AB2, CN1, announce
from test_gpu_ad_lines import setup

pytestmark = pytest.mark.gpu


def unread(shape):
    """Entries beside no cell: outer in two or three directions, or behind the
    upper outer layer."""
    count, behind = np.zeros(shape, int), np.zeros(shape, bool)
    for d, n in enumerate(shape):
        at = [slice(None)] * 3
        for q in (0, n - 2, n - 1):
            at[d] = q
            count[tuple(at)] += 1
        behind[tuple(at)] = True
    return (count >= 2) | behind


# 21x18x17 and 29x21x35: 2-cell y/z segments; 37x129x193: 16-cell ones;
# 130x98x82: 4-cell ones; x-lines of 1, 2 and 3 cells in their last segment;
# 24x32x48: every segment full
@pytest.mark.parametrize("shape", [(21, 18, 17), (29, 21, 35), (37, 129, 193), (130, 98, 82), (23, 70, 261),
                                   (24, 32, 48)], ids=str)
@pytest.mark.parametrize("scheme", ["AB2", "CN1", "CN2"])
def test_unread_outer_entries(shape, scheme):
    announce(f"{scheme} {shape} with non-finite outer edges")
    s, _, ib, gs, _, rng = setup(*shape, dt=1e-3)
    bad = unread(ib.shape)
    faces = [rng.standard_normal(ib.shape) * 0.5 for _ in range(3)]
    nl = [cases.random_field(ib.shape, 60 + q) for q in range(3)]
    u0 = [rng.standard_normal(ib.shape) * 0.1 for _ in range(3)]
    vbi = rng.standard_normal((gs.n, 3))
    p, bx, by, bz = (rng.standard_normal(ib.shape) * 0.1 for _ in range(4))
    out = {}
    for x in (0.0, np.nan, -np.inf):
        for a in u0 + nl:
            a[bad] = x
        kw = dict(vel_bi=vbi, itermax_ad=5, restol_ad=0.0)
        if scheme == "CN2":
            u, v, w, f, st = s.solve_ad_cn2(*u0, *nl, *faces, 1, p, bx, by, bz, **kw)
            got = (u, v, w) + f
        else:
            *got, st = s.solve_ad(AB2 if scheme == "AB2" else CN1, *u0, *nl, *faces, **kw)
        assert st["iterations"] == 5
        out[x] = [a[1:-2, 1:-2, 1:-2] for a in got], st["residual_uvw"]
    ref, res = out.pop(0.0)
    assert all(np.isfinite(a).all() for a in ref)
    for got, r in out.values():
        assert list(r) == list(res)
        assert all(np.array_equal(a, b) for a, b in zip(got, ref))
