"""Host arrays of 4 MB and more go into a solver in chunks of 2 MB, a lane for
each up to six: sizes on both sides of the limits, whole chunks and remainders.
Stated tolerance: 0, what was set is read back (FP32 and FP64 store it as it is)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

from turbulent_lbm_multigpu_amd import _capi  # noqa: E402
from turbulent_lbm_multigpu_amd.solver import LbmSolver  # noqa: E402

# 4 MB are just over 55,188 cells of FP32 and 27,594 of FP64; 27,584 and 13,760 fill a chunk
CASES = [((6132, 3, 3), _capi.STORAGE_F32), ((6133, 3, 3), _capi.STORAGE_F32), ((431, 64, 3), _capi.STORAGE_F32),
         ((47, 53, 23), _capi.STORAGE_F32), ((61, 67, 83), _capi.STORAGE_F32), ((3066, 3, 3), _capi.STORAGE_F64),
         ((3067, 3, 3), _capi.STORAGE_F64), ((71, 73, 61), _capi.STORAGE_F64)]


@pytest.mark.parametrize("dims,storage", CASES)
def test_set_reads_back(dims, storage):
    print(f"case: {dims} storage {storage}", flush=True)
    s = LbmSolver(dims, inv_tau=1.2, storage=storage)
    dtype = np.float64 if storage == _capi.STORAGE_F64 else np.float32
    for seed in (1, 2):
        dd = np.random.default_rng(seed).random((19,) + tuple(dims[::-1])).astype(dtype)
        s.set(_capi.FIELD_DD, dd)
        np.testing.assert_array_equal(s.store(_capi.FIELD_DD), dd)
    o, sz = (1, 1, 0), (dims[0] - 2, dims[1] - 1, dims[2])  # a region: x rows are not whole
    part = np.random.default_rng(3).random((19,) + tuple(sz[::-1])).astype(dtype)
    s.set(_capi.FIELD_DD, part, o, sz)
    dd[:, 0:sz[2], 1:1 + sz[1], 1:1 + sz[0]] = part
    np.testing.assert_array_equal(s.store(_capi.FIELD_DD), dd)
    s.close()
