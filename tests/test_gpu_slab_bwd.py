"""The slab backward of n <= 4 (csrc/bwd_slab.hip): both channel widths at the edges of its tiles (16 samples, 64 / 128
channels), of its ring of tiles in flight (1 .. 5 tiles per batch split) and of its splits, against the oracle and
each other.  Reference backward: src/python/mhc/ops.py:276-361."""
import pytest

from test_gpu_resident_bwd import K_RESIDENT, _both_paths

pytestmark = pytest.mark.gpu
K_SLAB_SPLITS, K_SLAB_WIDTH = 3, 11

# (B, n, C, splits; 0 = as the library chooses)
SHAPES = [(1, 4, 8, 0), (16, 4, 128, 1), (17, 4, 136, 1), (33, 3, 64, 1), (50, 4, 72, 1), (65, 2, 200, 1), (80, 1, 40, 1),
          (49, 3, 264, 2), (47, 4, 192, 3), (161, 2, 128, 4), (100, 1, 320, 0), (1000, 4, 1280, 7), (515, 3, 1928, 0)]


@pytest.mark.parametrize("B,n,C,splits", SHAPES)
@pytest.mark.parametrize("inject,w_f32", [(False, False), (False, True), (True, False)])
def test_slab_backward_widths(B, n, C, splits, inject, w_f32):
    from mhc._lib import tuning_lib

    lib = tuning_lib()
    try:
        assert lib.mhc_tuning_set(K_RESIDENT, 1) == 0 and lib.mhc_tuning_set(K_SLAB_SPLITS, splits) == 0
        _both_paths(K_SLAB_WIDTH, ("64 channels", "128 channels"), B, n, C, inject, w_f32)
    finally:
        lib.mhc_tuning_set(K_RESIDENT, 0)
        lib.mhc_tuning_set(K_SLAB_SPLITS, 0)
