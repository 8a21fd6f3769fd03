"""What surrounds the fused pairs of a step sequence: threads with a solver
each, changes of a group between sequences, a caller's recording.  Stated
tolerance: 0, every stored bit against single steps, which launch the half-step
kernels."""
import ctypes as C
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

from oracle import oracle as orc  # noqa: E402
from tests import test_gpu_pairs as pairs  # noqa: E402
from tests.test_gpu_parity import build_gpu_group  # noqa: E402
from turbulent_lbm_multigpu_amd import _capi, serving  # noqa: E402
from turbulent_lbm_multigpu_amd import decomposition as dec  # noqa: E402
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


def settle(s, steps=500):
    """Half-steps that repay the second buffer many times over; returns their number."""
    s.run(steps)
    assert s.pair_count()["second_buffer"]
    return steps


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
                for n in (8, 5, 130, 30):
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

    both(100)
    taken = b.pair_count()
    assert taken == 50
    for g, s in ((a, late[0]), (b, late[1])):
        g.add_member(s)
        g.set_member_stop(2, 30)  # beyond the next call
    both(8)
    for g in (a, b):
        g.set_launch(128, 3)  # rebuilds the descriptors, not the plan
        g.set_alpha_work_group(256)
    both(8)
    for g in (a, b):
        g.set_member_stop(2, -1)
    assert b.pair_count() == taken
    both(100)
    assert b.pair_count() == taken + 50
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
    dims, sizes = (64, 64, 64), 2
    a, b = [build(dims, F32, k) for k in range(sizes)], [build(dims, F32, k) for k in range(sizes)]
    g = LbmGroup(b)
    g.set_graph(False)
    first = 200 if paired_before else 2
    g.step(first)
    assert (g.pair_count() > 0) == paired_before
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
    n = 3 + settle(b) + 1
    b.step()
    taken = b.pair_count()["pairs"]
    assert taken == 248  # from an odd step: one half-step, 2 x 124 pairs, then three half-steps
    b.run(11)
    assert b.pair_count()["pairs"] == taken + 4
    b.step()
    b.run(8)
    assert b.pair_count()["pairs"] == taken + 8
    single_steps(a, n + 20)
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
        g.prepare_steps(10)  # as a caller who has many steps in mind
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
        b.run(48)
        assert b.pair_count() == {"pairs": 24 * (k + 1), "second_buffer": True}
        with pytest.raises(_capi.LbmError):
            serving.Server(4e12)
        assert not b.pair_count()["second_buffer"]
    b.run(48)
    assert b.pair_count() == {"pairs": 72, "second_buffer": True}
    single_steps(a, 144)
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
        solvers[0].run(500)
        assert solvers[0].pair_count() == {"pairs": 0, "second_buffer": False}
    else:
        g = LbmGroup(solvers)
        g.prepare_steps(8)
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
    b.prepare_steps(4)
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
    g.prepare_steps(8)
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
    settle(s)
    s.close()
    assert before - free_bytes() > 200e6
    release_kept_memory()
    assert before - free_bytes() < 50e6
    a, b = build((96, 90, 88), F32), build((96, 90, 88), F32)  # and goes on all the same
    single_steps(a, settle(b))
    same(a, b)
    a.close()
    b.close()


@pytest.mark.parametrize("dims,storage", [((24, 24, 24), F32), ((96, 96, 96), F32), ((64, 64, 64), F64)])
def test_short_runs_of_new_states_step_in_place(dims, storage):
    """A second buffer costs a short run more than it gains: it is taken once
    the half-steps so far would have repaid it, by one run or by many."""
    with build(dims, storage) as s:
        s.run(4)
        assert s.pair_count() == {"pairs": 0, "second_buffer": False}
        for _ in range(60):
            s.run(4)
        assert s.pair_count()["second_buffer"]
    with build(dims, storage) as s:
        s.run(240)
        assert s.pair_count() == {"pairs": 120, "second_buffer": True}
    with build(dims, storage) as s, build(dims, storage, 1) as t:
        g = LbmGroup([s] if dims[0] > 64 else [s, t])
        g.step(4)
        assert g.pair_count() == 0
        g.close()


def test_a_buffer_at_hand_is_taken_sooner():
    """One that a destroyed solver left costs no allocation."""
    release_kept_memory()
    with build((128, 128, 128), F32) as s:
        s.run(8)
        assert s.pair_count()["pairs"] == 0
        settle(s)
    with build((128, 128, 128), F32) as a, build((128, 128, 128), F32) as b:
        a.run(8)
        assert a.pair_count()["pairs"] == 4
        single_steps(b, 8)
        same(a, b)


# Every form of a domain that pairs take, after a second buffer is there: forcing, outputs, faces of
# all kinds, BGK and LES; walks by runs and rectangles, boxes.
FORMS = [
    ((83, 79, 77), F32, {"outputs": True, "grav": (1e-4, -2e-4, 3e-5)}),
    ((96, 96, 96), F32, {"cs": 0.0, "bc": (8, 8, 1, 1, 1, 8)}),
    ((300, 90, 40), F32, {"forcing": 1, "grav": (1e-5, 0.0, 0.0), "outputs": True}),
    ((1100, 60, 30), F32, {"lid": False}),
    ((61, 67, 63), F64, {"outputs": True, "grav": (1e-4, -2e-4, 3e-5)}),
    ((520, 60, 40), F64, {"forcing": 1, "grav": (0.0, 1e-5, 0.0), "bc": (1, 1, 8, 8, 1, 1)}),
    ((3, 3, 3), F32, {}),
    ((24, 20, 16), F32, {"outputs": True, "grav": (1e-4, -2e-4, 3e-5)}),
    ((36, 36, 36), F32, {"bc": (8, 8, 1, 1, 8, 1)}),
    ((100, 20, 20), F32, {"forcing": 1, "grav": (1e-5, 0.0, 0.0), "outputs": True}),
    ((9, 90, 4), F32, {"cs": 0.0}),
    ((31, 33, 29), F64, {"outputs": True}),
    ((3, 4, 151), F64, {}),
    ((130, 9, 11), F64, {"cs": 0.0, "bc": (1, 1, 8, 8, 1, 1)}),
]


@pytest.mark.parametrize("dims,storage,kw", FORMS)
def test_pairs_of_every_form(dims, storage, kw):
    print(f"case: {dims} storage {storage} {kw}", flush=True)
    a, b = pairs.build(dims, storage, **kw), pairs.build(dims, storage, **kw)
    single_steps(a, settle(b))
    for first, steps in ((0, 4), (1, 7), (0, 12)):
        taken = b.pair_count()["pairs"]
        single_steps(a, first + steps)
        single_steps(b, first)
        b.run(steps)
        assert b.pair_count()["pairs"] > taken
        assert pairs.same(pairs.fields(a, kw.get("outputs")), pairs.fields(b, kw.get("outputs")))
    a.close()
    b.close()


@pytest.mark.parametrize("dims,storage", [((80, 81, 79), F32), ((80, 81, 79), F64), ((24, 20, 16), F32), ((24, 20, 16), F64)])
def test_special_values_in_pairs(dims, storage):
    """-0, infinities, NaN and the largest finite value among the populations
    go the same way through both paths, walks and boxes."""
    two = [build(dims, storage) for _ in range(2)]
    single_steps(two[0], settle(two[1]))
    dt = np.float64 if storage == F64 else np.float32
    rng = np.random.default_rng(3)
    dd = two[0].store(_capi.FIELD_DD)
    for v in (-0.0, np.inf, -np.inf, np.nan, np.finfo(dt).max, np.finfo(dt).tiny):
        dd[tuple(rng.integers(0, n, 40) for n in dd.shape)] = v
    for s in two:
        s.set(_capi.FIELD_DD, dd)
    taken = two[1].pair_count()["pairs"]
    single_steps(two[0], 4)
    two[1].run(4)
    assert two[1].pair_count()["pairs"] == taken + 2
    a, b = (s.store(_capi.FIELD_DD) for s in two)
    nan = np.isnan(a)
    assert np.array_equal(nan, np.isnan(b)) and nan.any()
    bits = np.uint64 if storage == F64 else np.uint32
    assert np.array_equal(a.view(bits)[~nan], b.view(bits)[~nan])
    for s in two:
        s.close()


def test_pairs_equal_the_oracle():
    dims = (83, 79, 77)
    kw = dict(inv_tau=1 / 0.5005, tau=0.5005, smagorinsky_cs=0.17, lid_velocity=0.1)
    s = LbmSolver(dims, pairs.WALLS, **kw)
    settle(s)  # then from the start again
    o = orc.OracleDomain(dims, pairs.WALLS, **kw)
    o.reset(amplitude=1e-3, seed=12)
    s.init_perturbed(1e-3, 12)
    origin, size = dec.lid_region(dims)
    o.set_flags(origin, size, orc.FLAG_INJECTION)
    s.set(_capi.FIELD_FLAGS, np.full(size[::-1], orc.FLAG_INJECTION, np.int32), origin, size)
    taken = s.pair_count()["pairs"]
    o.run(8)
    s.run(8)
    assert s.pair_count()["pairs"] == taken + 4
    assert np.array_equal(s.store(_capi.FIELD_DD).reshape(19, -1), o.dd)
    s.close()


@pytest.mark.parametrize("graph", [True, False])
@pytest.mark.parametrize("storage", [F32, F64])
def test_paired_groups_with_members_that_freeze(storage, graph):
    """Across several calls, an odd start, a member that is frozen and one that
    freezes on the way."""
    sizes = [(16, 30, 21), (90, 91, 94), (33, 80, 97), (70, 64, 66)]
    (sa, ga), (sb, gb) = pairs.group_of(sizes, storage), pairs.group_of(sizes, storage)
    gb.set_graph(graph)
    ga.set_graph(False)
    gb.prepare_steps(10)

    def both(n, paired):
        taken = gb.pair_count()
        for _ in range(n):
            ga.step(1)
        gb.step(n)
        assert (gb.pair_count() > taken) == paired
        for x, y in zip(sa, sb):
            assert pairs.same(pairs.fields(x, False), pairs.fields(y, False))

    both(10, True)
    both(7, True)
    both(13, True)
    for g in (ga, gb):
        g.set_member_stop(1, 5)
    both(12, False)  # member 1 freezes inside the call
    both(8, True)    # and is frozen in this one
    for g in (ga, gb):
        g.set_member_stop(1, -1)
    both(9, True)
    both(2, False)
    both(16, True)
    ga.close()
    gb.close()
    for s in sa + sb:
        s.close()
