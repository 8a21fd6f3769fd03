"""Periodic rows of two-byte storages with two cells per work-item, whose x
faces the step kernel exchanges inside a wavefront, against the copy exchange:
rows of an even and an odd count of pairs, the shortest and some over several
wavefronts, split ones, and domains over the ends of layout blocks.

Stated tolerance: 0, every stored bit of every slot."""
import pytest

pytestmark = pytest.mark.gpu

from tests.test_gpu_parity import fused_vs_copy  # noqa: E402
from turbulent_lbm_multigpu_amd import _capi  # noqa: E402


@pytest.mark.parametrize("storage", [_capi.STORAGE_F16_SHIFTED, _capi.STORAGE_BF16_SHIFTED])
@pytest.mark.parametrize("domain_size,wg", [
    ((130, 9, 8), 256),    # 65 pairs a row, the fewest that are not split
    ((132, 37, 11), 64),
    ((134, 33, 14), 512),
    ((190, 41, 13), 256),
    ((254, 18, 15), 128),  # 127 pairs: every other seam one place earlier
    ((256, 35, 9), 256),   # split, over several layout blocks
    ((322, 21, 12), 256),
])
def test_seams_equal_the_copies(storage, domain_size, wg):
    for variant in (8, 11):
        fused_vs_copy(domain_size, (1, 1, 1), 1, wg=wg, periodic=(True, False, False), storage=storage,
                      variant=variant, step_runs=(3, 4))
