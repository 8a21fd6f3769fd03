"""Step sequences that run as fused beta + alpha pairs (long enough, large
enough, FP32/FP64, no exchange) against the same number of single steps, which
launch the half-step kernels, and against the CPU oracle.

Stated tolerance: 0.  Both paths evaluate the same expressions in the same
order; every stored bit of every slot is compared, NaNs by their places."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

from oracle import oracle as orc  # noqa: E402
from turbulent_lbm_multigpu_amd import _capi  # noqa: E402
from turbulent_lbm_multigpu_amd import decomposition as dec  # noqa: E402
from turbulent_lbm_multigpu_amd import serving  # noqa: E402
from turbulent_lbm_multigpu_amd._capi import LbmError  # noqa: E402
from turbulent_lbm_multigpu_amd.solver import LbmGroup, LbmSolver  # noqa: E402

WALLS = (1,) * 6


def build(dims, storage, *, bc=WALLS, cs=0.17, forcing=0, grav=(0.0, 0.0, 0.0), outputs=False, lid=True, case=0):
    s = LbmSolver(dims, bc, inv_tau=1 / 0.51, tau=0.51, smagorinsky_cs=cs, lid_velocity=0.08, gravitation=grav,
                  forcing=forcing, storage=storage, store_velocity=outputs, store_density=outputs)
    s.init_perturbed(0.01, 91, case)
    if lid:
        o, sz = dec.lid_region(dims)
        s.set(_capi.FIELD_FLAGS, np.full(sz[::-1], _capi.FLAG_VELOCITY_INJECTION, np.int32), o, sz)
    s.place_spheres(5, 0.04, 1.0, 2.5)
    return s


def fields(s, outputs):
    out = [s.store(_capi.FIELD_DD_RAW), s.step_counter]
    return out + ([s.store(_capi.FIELD_VELOCITY), s.store(_capi.FIELD_DENSITY)] if outputs else [])


def single_steps(s, n):
    for _ in range(n):
        s.step()


def same(a, b):
    return all(np.array_equal(x, y, equal_nan=isinstance(x, np.ndarray) and x.dtype.kind == "f") for x, y in zip(a, b))


# Small domains pair up in boxes: one box, single cells over a full box, flat,
# long and ragged ones.
BOXES = [
    ((3, 3, 3), _capi.STORAGE_F32, {}),
    ((24, 20, 16), _capi.STORAGE_F32, {"outputs": True, "grav": (1e-4, -2e-4, 3e-5)}),
    ((48, 48, 48), _capi.STORAGE_F32, {"bc": (8, 8, 1, 1, 8, 1)}),
    ((200, 20, 20), _capi.STORAGE_F32, {"forcing": 1, "grav": (1e-5, 0.0, 0.0), "outputs": True}),
    ((9, 90, 4), _capi.STORAGE_F32, {"cs": 0.0}),
    ((3, 4, 151), _capi.STORAGE_F64, {}),
    ((31, 33, 29), _capi.STORAGE_F64, {"outputs": True}),
    ((130, 9, 11), _capi.STORAGE_F64, {"cs": 0.0, "bc": (1, 1, 8, 8, 1, 1)}),
]
# FP32 sequences walk planes in pairs from 480,000 cells, FP64 from 250,000: rows as runs of
# positions (short rows), rectangles with one, even and ragged tile columns,
# domains thinner than a walk, rows longer than a work-group.
CASES = [
    ((12, 200, 210), _capi.STORAGE_F32, {}),
    ((83, 79, 77), _capi.STORAGE_F32, {"outputs": True, "grav": (1e-4, -2e-4, 3e-5)}),
    ((96, 96, 96), _capi.STORAGE_F32, {"cs": 0.0, "bc": (8, 8, 1, 1, 1, 8)}),
    ((257, 130, 15), _capi.STORAGE_F32, {"forcing": 1, "grav": (1e-5, 0.0, 0.0), "outputs": True}),
    ((400, 401, 3), _capi.STORAGE_F32, {}),
    ((1100, 30, 16), _capi.STORAGE_F32, {"lid": False}),
    ((3, 200, 420), _capi.STORAGE_F64, {}),
    ((61, 67, 63), _capi.STORAGE_F64, {"outputs": True}),
    ((520, 33, 17), _capi.STORAGE_F64, {"forcing": 1, "grav": (0.0, 1e-5, 0.0), "bc": (1, 1, 8, 8, 1, 1)}),
]


@pytest.mark.parametrize("dims,storage,kw", CASES + BOXES)
@pytest.mark.parametrize("first,steps", [(0, 4), (0, 7), (1, 12)])
def test_pairs_equal_single_steps(dims, storage, kw, first, steps):
    print(f"case: {dims} storage {storage} {kw} from {first}, {steps} steps", flush=True)
    a, b = build(dims, storage, **kw), build(dims, storage, **kw)
    single_steps(a, first + steps)
    single_steps(b, first)
    b.run(steps)
    assert same(fields(a, kw.get("outputs")), fields(b, kw.get("outputs")))
    a.close()
    b.close()


def test_pairs_equal_oracle():
    dims = (83, 79, 77)
    kw = dict(inv_tau=1 / 0.5005, tau=0.5005, smagorinsky_cs=0.17, lid_velocity=0.1)
    o = orc.OracleDomain(dims, WALLS, **kw)
    s = LbmSolver(dims, WALLS, **kw)
    o.reset(amplitude=1e-3, seed=12)
    s.init_perturbed(1e-3, 12)
    origin, size = dec.lid_region(dims)
    o.set_flags(origin, size, orc.FLAG_INJECTION)
    s.set(_capi.FIELD_FLAGS, np.full(size[::-1], orc.FLAG_INJECTION, np.int32), origin, size)
    o.run(8)
    s.run(8)
    assert np.array_equal(s.store(_capi.FIELD_DD).reshape(19, -1), o.dd)
    s.close()


@pytest.mark.parametrize("storage", [_capi.STORAGE_F32, _capi.STORAGE_F64])
def test_special_values(storage):
    """-0, infinities, NaN and the largest finite value among the populations
    go the same way through both paths."""
    dims = (80, 81, 79)
    pair = [build(dims, storage) for _ in range(2)]
    dt = np.float64 if storage == _capi.STORAGE_F64 else np.float32
    rng = np.random.default_rng(3)
    dd = pair[0].store(_capi.FIELD_DD)
    for v in (-0.0, np.inf, -np.inf, np.nan, np.finfo(dt).max, np.finfo(dt).tiny):
        at = tuple(rng.integers(0, n, 40) for n in dd.shape)
        dd[at] = v
    for s in pair:
        s.set(_capi.FIELD_DD, dd)
    single_steps(pair[0], 4)
    pair[1].run(4)
    a, b = (s.store(_capi.FIELD_DD) for s in pair)
    nan = np.isnan(a)
    assert np.array_equal(nan, np.isnan(b)) and nan.any()
    bits = np.uint64 if dt == np.float64 else np.uint32
    assert np.array_equal(a.view(bits)[~nan], b.view(bits)[~nan])
    for s in pair:
        s.close()


def group_of(sizes, storage):
    solvers = [build(d, storage, case=k) for k, d in enumerate(sizes)]
    return solvers, LbmGroup(solvers)


@pytest.mark.parametrize("graph", [True, False])
@pytest.mark.parametrize("storage", [_capi.STORAGE_F32, _capi.STORAGE_F64])
def test_group_pairs(storage, graph):
    """A group without exchange, also across several calls, an odd start, a
    member that is frozen and one that freezes on the way."""
    sizes = [(16, 30, 21), (90, 71, 64), (33, 80, 47)]
    sa, ga = group_of(sizes, storage)
    sb, gb = group_of(sizes, storage)
    gb.set_graph(graph)
    ga.set_graph(False)

    def both(n):
        for _ in range(n):
            ga.step(1)
        gb.step(n)
        for x, y in zip(sa, sb):
            assert same(fields(x, False), fields(y, False))

    both(10)
    both(7)
    both(13)
    for g in (ga, gb):
        g.set_member_stop(1, 5)
    both(12)   # member 1 freezes inside the call
    both(8)    # and is frozen in this one
    for g in (ga, gb):
        g.set_member_stop(1, -1)
    both(9)
    before = gb.launch_counts()
    gb.step(2)
    ga.step(1)
    ga.step(1)
    both(16)
    after = gb.launch_counts()
    assert after["graph_launches"] > before["graph_launches"] or not graph
    ga.close()
    gb.close()
    single_steps(sa[1], 6)  # on its own again
    sb[1].run(6)
    assert same(fields(sa[1], False), fields(sb[1], False))
    for s in sa + sb:
        s.close()


def test_second_buffers_are_given_back():
    """An allocation that does not fit takes the second buffers of idle
    solvers before it fails; they go on all the same."""
    dims = (96, 90, 88)
    a, b = build(dims, _capi.STORAGE_F32), build(dims, _capi.STORAGE_F32)
    b.run(8)
    b.wait()
    with pytest.raises(LbmError):
        serving.Server(4e12)
    b.run(8)
    g = LbmGroup([b])
    g.step(8)
    g.wait()
    with pytest.raises(LbmError):
        serving.Server(4e12)
    g.step(6)
    g.close()
    b.run(6)
    single_steps(a, 36)
    assert same(fields(a, False), fields(b, False))
    a.close()
    b.close()
