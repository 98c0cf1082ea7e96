"""The tiled backward of n <= 4.  The slab kernel (csrc/bwd_slab.hip): both channel widths at the edges of its tiles (16 samples, 64 / 128
channels), of its ring of tiles in flight (1 .. 5 tiles per batch split) and of its splits, against the oracle and
each other.  The channel sums with the coefficient backward of several samples per workgroup (gram_quad_kernel,
csrc/mix_bwd_reduce.hip): against the two launches.  The slab
kernel of five to eight streams: against the general kernels.  Reference backward: src/python/mhc/ops.py:276-361."""
import pytest
import torch

from test_gpu_resident_bwd import K_RESIDENT, _both_paths

pytestmark = pytest.mark.gpu
K_GRAM, K_SLAB_SPLITS, K_SLAB_WIDTH, K_SLAB8 = 2, 3, 11, 12

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


# one to four samples in the last workgroup; rows of one step, of whole and cut steps, of one to three steps per wave
@pytest.mark.parametrize("B,n,C", [(1, 4, 8), (2, 4, 128), (3, 2, 136), (5, 4, 904), (9, 3, 1032), (6, 4, 2560), (7, 1, 2688),
                                   (4, 4, 4096), (10, 2, 4224)])
@pytest.mark.parametrize("inject,w_f32", [(False, False), (False, True), (True, False)])
def test_channel_sums_of_several_samples_per_workgroup(B, n, C, inject, w_f32):
    from mhc._lib import tuning_lib

    lib = tuning_lib()
    try:
        assert lib.mhc_tuning_set(K_RESIDENT, 1) == 0
        _both_paths(K_GRAM, ("two launches", "several samples"), B, n, C, inject, w_f32)
    finally:
        lib.mhc_tuning_set(K_RESIDENT, 0)


# fewer than four streams, whose sums share a 4 x 4 product with nobody's: a sum of stream 0 that overflows stays infinite where the
# two launches have infinity (NaN comes from an infinity times the zero coefficient of a stream that is not there)
@pytest.mark.parametrize("n", [1, 2, 3])
def test_overflow_of_one_sum_stays_where_it_is(n):
    from mhc._lib import tuning_lib
    from test_gpu_resident_bwd import _step

    lib, got = tuning_lib(), []
    st = _step(6, n, 136, False, False)
    st.forward()
    st.dy.zero_()
    st.x[4, :, 7] = 0
    st.x[4, 0, 7], st.dy[4, n - 1, 7] = 8.0, 1e38  # dy x^T of streams (n - 1, 0) only
    try:
        assert lib.mhc_tuning_set(K_RESIDENT, 1) == 0
        for mode in (1, 2):
            assert lib.mhc_tuning_set(K_GRAM, mode) == 0
            st.backward()
            got.append(st.dbias[n:2 * n].cpu())  # of H_post
    finally:
        lib.mhc_tuning_set(K_RESIDENT, 0)
        lib.mhc_tuning_set(K_GRAM, 0)
    for g in got:
        assert g[n - 1] == float("inf") and not g[:n - 1].any(), got


# slots of a tile beyond the batch repeat its last sample: one whose df overflows adds its infinity to dw and the slots nothing
@pytest.mark.parametrize("n", [2, 4, 5, 8])
def test_slots_beyond_the_batch_add_nothing(n):
    from mhc._lib import tuning_lib
    from test_gpu_resident_bwd import _step

    lib, got = tuning_lib(), []
    st = _step(17, n, 72, False, False)
    st.forward()
    st.dy[16, :, 7] = 3e38
    st.x[16, :, 7] = 1.0
    try:
        for mode in (1, 2):
            assert lib.mhc_tuning_set(K_RESIDENT, mode) == 0
            st.backward()
            got.append(st.dw.cpu())
    finally:
        lib.mhc_tuning_set(K_RESIDENT, 0)
    for g in got:
        assert g[7] == float("inf") and torch.isfinite(g[:7]).all() and torch.isfinite(g[8:]).all(), g


# n = 5 .. 8 (csrc/bwd_slab8.hip): one to four tiles of 16 samples per split, cut tiles, channels beyond the row, several slabs
@pytest.mark.parametrize("B,n,C,splits", [(1, 5, 8, 1), (16, 8, 64, 1), (17, 8, 72, 1), (33, 6, 136, 1), (50, 7, 64, 1), (49, 8, 200, 2),
                                          (130, 5, 264, 3), (65, 7, 320, 0), (200, 8, 1280, 0), (300, 6, 1928, 0)])
@pytest.mark.parametrize("inject,w_f32", [(False, False), (False, True), (True, False)])
def test_slab_backward_of_five_to_eight_streams(B, n, C, splits, inject, w_f32):
    from mhc._lib import tuning_lib

    lib = tuning_lib()
    try:
        assert lib.mhc_tuning_set(K_RESIDENT, 1) == 0 and lib.mhc_tuning_set(K_SLAB_SPLITS, splits) == 0
        _both_paths(K_SLAB8, ("general kernels", "slab"), B, n, C, inject, w_f32)
    finally:
        lib.mhc_tuning_set(K_RESIDENT, 0)
        lib.mhc_tuning_set(K_SLAB_SPLITS, 0)
