"""What surrounds the fused pairs of a step sequence: threads with a solver
each, changes of a group between sequences, a caller's recording.  Stated
tolerance: 0, every stored bit against single steps, which launch the half-step
kernels."""
import ctypes as C
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

from tests.test_gpu_parity import build_gpu_group  # noqa: E402
from turbulent_lbm_multigpu_amd import _capi, serving  # noqa: E402
from turbulent_lbm_multigpu_amd.solver import LbmGroup, LbmSolver, release_kept_memory  # noqa: E402

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


def x_chain(dims, n, storage):
    """n members joined in x."""
    solvers = [build(dims, storage, i, (8 if i else 1, 8 if i < n - 1 else 1, 1, 1, 1, 1)) for i in range(n)]
    g = LbmGroup(solvers)
    size = (1, dims[1], dims[2])
    for i in range(n):
        if i:
            g.add_comm(i, i - 1, (1, 0, 0), (0, 0, 0), size, (1, 0, 0))
        if i < n - 1:
            g.add_comm(i, i + 1, (dims[0] - 2, 0, 0), (dims[0] - 1, 0, 0), size, (-1, 0, 0))
    return g


def test_a_stopping_member_joins_a_paired_group():
    """The plan of the two joined members, who run as pairs, does not outlive
    the third's arrival, whose stop refuses pairs; nor does the refusal."""
    dims = (130, 140, 140)
    a, b = x_chain(dims, 2, F32), x_chain(dims, 2, F32)
    late = [build((90, 80, 70), F32, 7) for _ in range(2)]

    def both(n):
        for _ in range(n):
            a.step(1)
        b.step(n)
        a.wait()
        b.wait()
        for x, y in zip(a.solvers, b.solvers):
            same(x, y)

    both(8)
    assert b.pair_count() == 4
    for g, s in ((a, late[0]), (b, late[1])):
        g.add_member(s)
        g.set_member_stop(2, 30)
    both(8)
    for g in (a, b):
        g.set_launch(128, 3)  # rebuilds the descriptors, not the plan
        g.set_alpha_work_group(256)
    both(8)
    for g in (a, b):
        g.set_member_stop(2, -1)
    assert b.pair_count() == 4
    both(8)
    assert b.pair_count() == 8
    for g in (a, b):
        g.remove_member(2)
    both(8)
    for g in (a, b):
        g.close()
    for s in a.solvers + b.solvers + late:
        s.close()


@pytest.mark.parametrize("paired_before", [False, True])
def test_a_recorded_sequence_steps_in_place(paired_before):
    """A caller who records the group's stream gets launches that do not
    depend on second buffers: replays after these are gone, with eager steps
    in between, are still the same."""
    dims, sizes = (96, 90, 88), 2
    a, b = [build(dims, F32, k) for k in range(sizes)], [build(dims, F32, k) for k in range(sizes)]
    g = LbmGroup(b)
    g.set_graph(False)
    first = 8 if paired_before else 2
    g.step(first)
    g.wait()
    lib, stream = _capi.load_library(), C.c_void_p()
    assert lib.lbm_group_get_stream(g._h, C.byref(stream)) == 0
    graph, replay = C.c_void_p(), C.c_void_p()
    assert lib.hipStreamBeginCapture(stream, 1) == 0
    g.step(8)
    assert lib.hipStreamEndCapture(stream, C.byref(graph)) == 0
    assert lib.hipGraphInstantiate(C.byref(replay), graph, None, None, C.c_size_t(0)) == 0
    n = first
    for k in range(4):
        assert lib.hipGraphLaunch(replay, stream) == 0
        g.wait()
        n += 8
        if k == 1:
            with pytest.raises(_capi.LbmError):
                serving.Server(4e12)  # takes the second buffers away
        if k % 2:
            g.step(2)
            g.wait()
            n += 2
        for x in a:
            single_steps(x, n - x.step_counter)
        for x, y in zip(a, b):
            np.testing.assert_array_equal(x.store(_capi.FIELD_DD_RAW), y.store(_capi.FIELD_DD_RAW))
    assert lib.hipGraphExecDestroy(replay) == 0 and lib.hipGraphDestroy(graph) == 0
    g.close()
    for s in a + b:
        s.close()


# Domains whose sequences take pairs: walks by runs of positions and by
# rectangles, one column wide to rows longer than a work-group, thin and ragged;
# then boxes.
@pytest.mark.parametrize("dims,storage", [
    ((83, 79, 77), F32), ((150, 141, 133), F32), ((12, 200, 210), F32), ((400, 401, 3), F32), ((500, 4, 250), F32),
    ((1100, 60, 30), F32), ((330, 100, 60), F32), ((61, 67, 63), F64), ((3, 700, 700), F64), ((520, 60, 40), F64),
    ((300, 61, 30), F64), ((24, 20, 16), F32), ((16, 16, 16), F64)])
def test_sequences_take_pairs(dims, storage):
    a, b = build(dims, storage), build(dims, storage)
    assert b.pair_count() == {"pairs": 0, "second_buffer": False}
    b.run(3)
    assert b.pair_count() == {"pairs": 0, "second_buffer": False}  # too short
    b.run(12)  # on an odd step: one half-step, then 2 x 2 pairs, then three half-steps
    assert b.pair_count() == {"pairs": 4, "second_buffer": True}
    b.step()
    b.run(8)
    assert b.pair_count()["pairs"] == 8
    single_steps(a, 24)
    assert a.pair_count() == {"pairs": 0, "second_buffer": False}
    same(a, b)
    a.close()
    b.close()


@pytest.mark.parametrize("graph", [True, False])
def test_groups_take_pairs(graph):
    """With and without exchange, in graphs and launched one by one."""
    free = LbmGroup([build((96, 70, 64), F32, k) for k in range(3)])
    joined = x_chain((130, 140, 140), 2, F32)
    two = LbmGroup([build((64, 70, 64), F64, k) for k in range(5)])
    for g in (free, joined, two):
        g.set_graph(graph)
        g.step(2)
        assert g.pair_count() == 0
        g.step(10)  # five pairs, of which the last has none to go back with
        assert g.pair_count() == 4
        g.step(64)
        assert g.pair_count() == 36
        g.set_timing(True)  # times the half-step kernels
        g.step(8)
        assert g.pair_count() == 36
        g.set_timing(False)
        assert all(s.pair_count() == {"pairs": 0, "second_buffer": True} for s in g.solvers)
        g.close()
        for s in g.solvers:
            s.close()


def test_a_failed_allocation_takes_the_second_buffers():
    """They are held, gone after an allocation that does not fit, and taken
    again by the next sequence."""
    a, b = build((96, 90, 88), F32), build((96, 90, 88), F32)
    for k in range(2):
        b.run(8)
        assert b.pair_count() == {"pairs": 4 * (k + 1), "second_buffer": True}
        with pytest.raises(_capi.LbmError):
            serving.Server(4e12)
        assert not b.pair_count()["second_buffer"]
    b.run(8)
    assert b.pair_count() == {"pairs": 12, "second_buffer": True}
    single_steps(a, 24)
    same(a, b)
    a.close()
    b.close()


# Walks of few columns, or of few planes beside the two of their halo, lose
# against the half-steps (by 3.5 and 11 times the first two), large boxes where
# several solvers run side by side.
@pytest.mark.parametrize("count,dims,storage", [(1500, (8, 8, 8), F32), (1, (4, 4, 60000), F32), (1, (1000, 1000, 3), F32),
                                                (200, (16, 16, 16), F32), (1, (300, 300, 3), F64), (400, (12, 12, 12), F64),
                                                (1, (48, 48, 48), F32), (1, (40, 40, 40), F64)])
def test_shapes_that_step_in_place(count, dims, storage):
    solvers = [build(dims, storage, k) for k in range(count)]
    if count == 1:
        solvers[0].run(8)
        assert solvers[0].pair_count() == {"pairs": 0, "second_buffer": False}
    else:
        g = LbmGroup(solvers)
        g.step(8)
        assert g.pair_count() == 0 and not any(s.pair_count()["second_buffer"] for s in solvers)
        g.close()
    for s in solvers:
        s.close()


# domain, subdomains, periodic axes, storage, exchange mode, x faces in the kernel, kernel variant
FACES = [
    ((170, 164, 166), (2, 2, 2), (0, 0, 0), F32, 1, 1, 0),  # edges and corners of three axes
    ((170, 164, 166), (2, 2, 2), (0, 0, 0), F32, 0, 0, 0),  # every slot of the ghost layers is copied
    ((180, 168, 166), (3, 1, 2), (1, 1, 1), F32, 1, 2, 0),  # every face has a neighbour, some the domain itself
    ((260, 150, 130), (1, 1, 1), (1, 0, 1), F32, 1, 0, 0),  # a domain next to itself along two axes
    ((16, 400, 420), (4, 1, 1), (0, 0, 0), F32, 1, 0, 3),   # four cells wide: ghost and inner layers only
    ((300, 64, 68), (3, 1, 1), (1, 0, 0), F32, 0, 1, 35),
    ((400, 112, 104), (1, 2, 1), (0, 0, 0), F32, 1, 1, 0),  # several tile columns
    ((122, 140, 150), (2, 2, 1), (0, 1, 0), F64, 1, 2, 0),
    ((60, 230, 240), (1, 2, 2), (1, 0, 0), F64, 0, 0, 0),
]


@pytest.mark.parametrize("case,graph", [(c, True) for c in FACES] + [(FACES[0], False), (FACES[-1], False)])
def test_groups_with_faces_take_pairs(case, graph):
    size, nums, periodic, storage, mode, fused, variant = case
    print(f"case: {case} graph {graph}", flush=True)
    groups = []
    for _ in range(2):
        g, _, _ = build_gpu_group(size, nums, lid=0.08, amp=1e-2, seed=11, storage=storage, mode=mode, graph=graph,
                                  periodic=tuple(bool(p) for p in periodic), inv_tau=1 / 0.51, tau=0.51,
                                  smagorinsky_cs=0.17, kernel_variant=variant)
        for i, s in enumerate(g.solvers):
            s.place_spheres(5 + i, 0.04, 1.0, 2.5)
        g.set_fused_x(fused)
        groups.append(g)
    a, b = groups
    for n in (4, 1, 7):
        for _ in range(n):
            a.step(1)
        b.step(n)
    a.wait()
    b.wait()
    assert a.pair_count() == 0 and b.pair_count() == 4
    for x, y in zip(a.solvers, b.solvers):
        same(x, y)
        for field in (_capi.FIELD_VELOCITY, _capi.FIELD_DENSITY):
            np.testing.assert_array_equal(x.store(field), y.store(field))
    for g in groups:
        g.close()
        for s in g.solvers:
            s.close()


@pytest.mark.parametrize("nums,dims,storage", [((5, 5, 5), (32, 32, 32), F32), ((10, 10, 1), (16, 16, 200), F32),
                                               ((2, 2, 2), (300, 300, 4), F64)])
def test_joined_shapes_that_step_in_place(nums, dims, storage):
    """Above 240 MB, and slower in pairs."""
    mono = tuple(n * d for n, d in zip(nums, dims))
    g, _, _ = build_gpu_group(mono, nums, lid=0.08, amp=1e-2, seed=11, storage=storage, mode=1, inv_tau=1 / 0.51,
                              tau=0.51, smagorinsky_cs=0.17)
    g.step(8)
    assert g.pair_count() == 0 and not any(s.pair_count()["second_buffer"] for s in g.solvers)
    g.close()
    for s in g.solvers:
        s.close()


def free_bytes():
    free, total = C.c_size_t(), C.c_size_t()
    assert _capi.load_library().hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    return free.value


def test_kept_memory_is_given_back():
    """A closed solver's second buffer (here 209 MB) is kept for the next one
    until it is asked for."""
    release_kept_memory()
    before = free_bytes()
    s = build((140, 140, 140), F32)
    s.run(8)
    assert s.pair_count()["second_buffer"]
    s.close()
    assert before - free_bytes() > 200e6
    release_kept_memory()
    assert before - free_bytes() < 50e6
    a, b = build((96, 90, 88), F32), build((96, 90, 88), F32)  # and goes on all the same
    b.run(8)
    single_steps(a, 8)
    same(a, b)
    assert b.pair_count()["second_buffer"]
    a.close()
    b.close()
