"""Transfers between host and device go in chunks of one megabyte (two from
32 MB on), in turn through the lanes of several threads: regions of one chunk,
exactly full ones, one cell more, and many, from any origin.

Stated tolerance: 0, fields are copied bit for bit, and a moment depends on its
own cell alone."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

from turbulent_lbm_multigpu_amd import _capi  # noqa: E402
from turbulent_lbm_multigpu_amd.solver import LbmSolver  # noqa: E402

MB = 1 << 20


def chunk(bytes_per_cell):
    return MB // bytes_per_cell // 64 * 64


# domain, region origin, region size: 13,760 cells fill a chunk of FP32
# distributions, 6,848 of FP64, 27,584 of FP16
CASES = [
    ((5, 4, 3), (0, 0, 0), (1, 1, 1), _capi.STORAGE_F32),
    ((42, 45, 9), (1, 2, 1), (40, 43, 8), _capi.STORAGE_F32),
    ((140, 10, 100), (1, 1, 0), (139, 9, 11), _capi.STORAGE_F32),
    ((64, 107, 3), (0, 0, 2), (64, 107, 1), _capi.STORAGE_F64),
    ((61, 47, 53), (0, 1, 2), (61, 45, 50), _capi.STORAGE_F64),
    ((97, 61, 83), (3, 0, 1), (94, 61, 82), _capi.STORAGE_F16_SHIFTED),
    ((101, 67, 71), (0, 0, 0), (101, 67, 71), _capi.STORAGE_F32),
]


def test_the_regions_meet_the_edges_of_chunks():
    assert 40 * 43 * 8 == chunk(76) and 139 * 9 * 11 == chunk(76) + 1 and 64 * 107 == chunk(152)


def solver(dims, storage, seed):
    s = LbmSolver(dims, (1,) * 6, inv_tau=1 / 0.51, tau=0.51, smagorinsky_cs=0.17, lid_velocity=0.08,
                  storage=storage, store_velocity=True, store_density=True)
    s.init_perturbed(0.01, seed)
    return s


def bits(rng, like):
    raw = rng.integers(0, 256, like.nbytes, dtype=np.uint8)
    return raw.view(like.dtype).reshape(like.shape)


def check_region(dims, origin, size, storage, seed):
    rng = np.random.default_rng(seed)
    box = (Ellipsis,) + tuple(slice(o, o + n) for o, n in zip(origin[::-1], size[::-1]))
    with solver(dims, storage, seed) as s:
        rho, j = s.moments()
        r, k = s.moments(origin, size)
        assert np.array_equal(r, rho[box]) and np.array_equal(k, j[box])
        for field in (_capi.FIELD_DD_RAW, _capi.FIELD_FLAGS, _capi.FIELD_VELOCITY, _capi.FIELD_DENSITY):
            whole = s.store(field)
            part = s.store(field, origin, size)
            assert part.tobytes() == np.ascontiguousarray(whole[box]).tobytes()
            if field == _capi.FIELD_FLAGS:
                new = rng.integers(0, 256, part.shape).astype(part.dtype)
            elif field == _capi.FIELD_DD_RAW:
                new = bits(rng, part)
            else:
                new = rng.random(part.shape).astype(part.dtype)
            s.set(field, new, origin, size)
            whole[box] = new
            assert s.store(field).tobytes() == whole.tobytes()


@pytest.mark.parametrize("dims,origin,size,storage", CASES)
def test_regions_come_and_go_bit_for_bit(dims, origin, size, storage):
    check_region(dims, origin, size, storage, 11)


def test_threads_share_the_lanes():
    """Eight threads with a solver each want more lanes than there are."""
    failed = []

    def work(seed):
        try:
            check_region((97, 61, 53), (3, 0, 1), (94, 61, 52), _capi.STORAGE_F32, seed)
        except BaseException as e:  # noqa: BLE001
            failed.append(e)

    threads = [threading.Thread(target=work, args=(i,)) for i in range(8)]
    for t in threads:
        t.start()
    for t in threads:
        t.join(100)
    assert not failed and not any(t.is_alive() for t in threads)
