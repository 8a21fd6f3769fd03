"""What surrounds the fused pairs of a step sequence: threads with a solver
each, changes of a group between sequences.  Stated tolerance: 0, every stored
bit against single steps, which launch the half-step kernels."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

from turbulent_lbm_multigpu_amd import _capi  # noqa: E402
from turbulent_lbm_multigpu_amd.solver import LbmSolver  # noqa: E402

F32, F64 = _capi.STORAGE_F32, _capi.STORAGE_F64


def build(dims, storage, case=0, bc=(1,) * 6):
    s = LbmSolver(dims, bc, inv_tau=1 / 0.51, tau=0.51, smagorinsky_cs=0.17, lid_velocity=0.08, storage=storage)
    s.init_perturbed(0.01, 91, case)
    s.place_spheres(5 + case, 0.04, 1.0, 2.5)
    return s


def single_steps(s, n):
    for _ in range(n):
        s.step()


def same(a, b):
    assert a.step_counter == b.step_counter
    np.testing.assert_array_equal(a.store(_capi.FIELD_DD_RAW), b.store(_capi.FIELD_DD_RAW))


def test_threads_with_a_solver_each():
    """Walks and boxes from several threads at once, buffers taken and given
    back all the while."""
    cases = [((96, 90, 88), F32), ((64, 70, 72), F64), ((24, 20, 16), F32), ((90, 96, 71), F32)]

    def work(k, errors):
        dims, storage = cases[k]
        try:
            for _ in range(3):
                a, b = build(dims, storage, k), build(dims, storage, k)
                for n in (8, 5, 30):
                    single_steps(a, n)
                    b.run(n)
                same(a, b)
                a.close()
                b.close()
        except BaseException as e:  # noqa: BLE001 (reported by the test's own thread)
            errors.append((k, e))

    errors = []
    threads = [threading.Thread(target=work, args=(k, errors)) for k in range(len(cases))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors, errors
