"""The batch splits of the slab backward take every S-th tile of 16 samples (csrc/bwd_slab.hip, csrc/bwd_slab8.hip): splits of
unequal tile counts, a cut last tile that belongs to any of them, as many splits as tiles; against the oracle and the other
path.  Reference backward: src/python/mhc/ops.py:276-361."""
import pytest

from test_gpu_resident_bwd import K_RESIDENT, _both_paths

pytestmark = pytest.mark.gpu
K_SLAB_SPLITS, K_SLAB_WIDTH, K_SLAB8 = 3, 11, 12


# (tiles, splits, split of the last tile): (6, 4, 1), (6, 6, 5), (7, 3, 0), (2, 2, 1)
@pytest.mark.parametrize("B,splits", [(83, 4), (96, 6), (97, 3), (17, 2)])
@pytest.mark.parametrize("n,C", [(4, 136), (1, 64), (5, 72), (8, 64)])
def test_splits_of_every_sth_tile(B, splits, n, C):
    from mhc._lib import tuning_lib

    lib = tuning_lib()
    key, names = (K_SLAB_WIDTH, ("64 channels", "128 channels")) if n <= 4 else (K_SLAB8, ("general kernels", "slab"))
    try:
        assert lib.mhc_tuning_set(K_RESIDENT, 1) == 0 and lib.mhc_tuning_set(K_SLAB_SPLITS, splits) == 0
        _both_paths(key, names, B, n, C, False, False)
    finally:
        lib.mhc_tuning_set(K_RESIDENT, 0)
        lib.mhc_tuning_set(K_SLAB_SPLITS, 0)
