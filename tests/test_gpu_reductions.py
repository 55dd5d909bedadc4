"""GPU: the divergence pass and the one-launch reduction of its partial sums,
at the edges of both: rows left over by the four rows of a thread, grids
wider than a workgroup, one workgroup of partials, exactly one chunk of them
(512), one more, and many chunks.  The field is the NumPy expression in the
same order (bit for bit: no operation is contracted), 0 on the outer layers;
the sum is that of the field's cells, within the N rounding errors that any
order of N additions may make.  Two calls in a row: the second finds the
workgroup counter as the first left it."""
import numpy as np
import pytest

from flow_structure_interaction_fem_ibm_amd import pp

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

# cells: workgroups of 64x16, 128x8 or 256x4 rows per plane
SHAPES = [(4, 4, 4),          # 4 partials, one row group
          (64, 16, 512),      # 512: one chunk exactly
          (63, 15, 513),      # 513: two chunks
          (130, 6, 10),       # a workgroup wider than the row
          (258, 5, 7),        # two workgroups per row, a single row left over
          (20, 18, 1000)]     # 2000: four chunks


@pytest.mark.parametrize("n", SHAPES, ids=lambda n: "x".join(map(str, n)))
def test_divergence_field_and_sum(n):
    print(f"[case] divergence {n}", flush=True)
    nodes = [pp.tanh_nodes(m, m / 64.0, b) for m, b in zip(n, (1.0, 0.8, 1.2))]
    s = pp.PressureSolver(*nodes)
    rng = np.random.default_rng(sum(n))
    ib = np.zeros(s.shape, np.int8)
    s.set_geometry(ib, pp.GhostSet(*[np.zeros(0, np.int32)] * 6, np.zeros((0, 8)), np.zeros(0)))
    f = [rng.standard_normal(s.shape) for _ in range(3)]
    assert s.shape == (n[2] + 3, n[1] + 3, n[0] + 3)
    d = [np.diff(x) for x in nodes]
    inv = [1.0 / q for q in d]
    dtinv = 3.0
    c = (slice(1, n[2] + 1), slice(1, n[1] + 1), slice(1, n[0] + 1))

    def diff(a, ax):
        sl = list(c)
        sl[ax] = slice(2, n[2 - ax] + 2)
        return a[tuple(sl)] - a[c]
    v = dtinv * (diff(f[0], 2) * inv[0] + diff(f[1], 1) * inv[1][:, None] + diff(f[2], 0) * inv[2][:, None, None])
    ref = np.zeros(s.shape)
    ref[c] = v
    terms = v * d[0] * d[1][:, None] * d[2][:, None, None]
    tol = terms.size * np.finfo(float).eps * np.abs(terms).sum()
    tf = [torch.from_numpy(a).cuda() for a in f]
    for _ in range(2):
        out = torch.full(s.shape, 7.0, dtype=torch.float64, device="cuda")
        got = s.divergence_noalloc(*tf, out, dtinv=dtinv)
        assert np.array_equal(out.cpu().numpy(), ref)
        assert abs(got - terms.sum()) <= tol
        host, hsum = s.divergence(*f, dtinv=dtinv)
        assert np.array_equal(host, ref) and hsum == got
