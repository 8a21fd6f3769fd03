"""Step sequences of groups that exchange faces, run as fused beta + alpha
pairs (from 240 MB of distributions, 84 where only x faces are exchanged in
FP32), against the same number of single steps, which launch the half-step
kernels and their copies.

Stated tolerance: 0, every stored bit of every slot and output: both paths
evaluate the same expressions in the same order."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

from tests.test_gpu_parity import build_gpu_group  # noqa: E402
from turbulent_lbm_multigpu_amd import _capi  # noqa: E402

F32, F64 = _capi.STORAGE_F32, _capi.STORAGE_F64
# domain, subdomains, periodic axes, storage, exchange mode, x faces in the kernel
CASES = [
    ((152, 146, 150), (2, 2, 2), (0, 0, 0), F32, 1, 1),  # edges and corners of three axes
    ((152, 146, 150), (2, 2, 2), (0, 0, 0), F32, 0, 0),  # every slot of the ghost layers is copied
    ((159, 144, 146), (3, 1, 2), (1, 1, 1), F32, 1, 2),  # every face has a neighbour, some the domain itself
    ((200, 130, 128), (1, 1, 1), (1, 0, 1), F32, 1, 0),  # a domain next to itself along two axes
    ((12, 520, 520), (1, 1, 1), (1, 1, 0), F32, 0, 0),
    ((16, 260, 270), (4, 1, 1), (0, 0, 0), F32, 1, 0),   # four cells wide: ghost and inner layers only
    ((300, 64, 60), (3, 1, 1), (1, 0, 0), F32, 0, 1),
    ((330, 100, 98), (1, 2, 1), (0, 0, 0), F32, 1, 1),   # several tile columns
    ((102, 122, 128), (2, 2, 1), (0, 1, 0), F64, 1, 2),
    ((24, 258, 260), (1, 2, 2), (1, 0, 0), F64, 0, 0),
]


def group(case, graph):
    size, nums, periodic, storage, mode, fused = case
    g, _, _ = build_gpu_group(size, nums, lid=0.08, amp=1e-2, seed=11, storage=storage, mode=mode, graph=graph,
                              periodic=tuple(bool(p) for p in periodic), inv_tau=1 / 0.51, tau=0.51,
                              smagorinsky_cs=0.17)
    for i, s in enumerate(g.solvers):
        s.place_spheres(5 + i, 0.04, 1.0, 2.5)
    g.set_fused_x(fused)
    return g


def same(a, b):
    for x, y in zip(a.solvers, b.solvers):
        assert x.step_counter == y.step_counter
        for field in (_capi.FIELD_DD_RAW, _capi.FIELD_VELOCITY, _capi.FIELD_DENSITY):
            np.testing.assert_array_equal(x.store(field), y.store(field))


@pytest.mark.parametrize("case,graph", [(c, True) for c in CASES] + [(CASES[0], False), (CASES[-1], False)])
def test_face_pairs_equal_single_steps(case, graph):
    print(f"case: {case} graph {graph}", flush=True)
    a, b = group(case, graph), group(case, graph)
    for n in (4, 1, 7):
        for _ in range(n):
            a.step(1)
        b.step(n)
        a.wait()
        b.wait()
        same(a, b)
    for g in (a, b):
        g.close()
