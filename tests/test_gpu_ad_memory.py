"""Device memory of the momentum entry points: a solve keeps its working copy
(13 padded FP64 arrays) with the context, a single residual keeps nothing, and
pp_destroy gives everything back."""
import numpy as np
import pytest

from flow_structure_interaction_fem_ibm_amd import pp
from test_gpu_ad import AB2, CN1, announce

pytestmark = pytest.mark.gpu


def context(n):
    s = pp.PressureSolver(*[np.linspace(0.0, 1.0, n + 1)] * 3)
    z = np.zeros(0, np.int32)
    s.set_geometry(np.zeros(s.shape, np.int8), pp.GhostSet(z, z, z, z, z, z, np.zeros((0, 8)), np.zeros(0)))
    visc = np.full(s.shape, 0.01)
    s.set_solve_ad(1e-3, visc, visc, visc, visc)
    return s, np.random.default_rng(1).standard_normal(s.shape)


def test_held_memory():
    import torch
    announce("device memory of calc_residual_ad and solve_ad, 128x128x128")
    free = lambda: torch.cuda.mem_get_info()[0]
    s, f = context(24)  # code objects and runtime pools load with the first calls
    s.calc_residual_ad(CN1, *[f] * 5)
    s.solve_ad(AB2, *[f] * 9, itermax_ad=1)
    s.close()
    start = free()
    s, f = context(128)
    copy = 13 * 8 * 130 * 130 * 128  # at least
    before = free()
    m0 = s.calc_residual_ad(CN1, *[f] * 5)
    assert before - free() < copy // 8
    s.solve_ad(AB2, *[f] * 9, itermax_ad=1)
    held = before - free()
    assert copy <= held < 2 * copy
    m1 = s.calc_residual_ad(CN1, *[f] * 5)
    assert abs(before - free() - held) < copy // 8  # the solve's copy stays
    assert m0[:2] == m1[:2] and np.array_equal(m0[2], m1[2])
    s.close()
    assert start - free() < copy // 8
