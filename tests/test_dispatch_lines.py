"""Which launch path a call takes, on either side of the lines at which two paths cost the same (mhc_tuning_route of the tuning
build: the built-in rules, no GPU needed).  Every row is a size at which one of the two was measured to be the faster one; the
figures stand beside the rules (csrc/capi.hip)."""
import pytest

F32, BF16, F32_AS_BF16 = 0, 1, 2
BACKWARD = 0
RESIDENT, TILED = 0, 1


def _route(which, dtype, B, n, C):
    from mhc._lib import tuning_lib

    return tuning_lib().mhc_tuning_route(which, dtype, B, n, C)


@pytest.mark.parametrize("n,C,rows", [
    # full rounds of the resident path, and the first sizes of the round behind them
    (4, 2048, [(420, RESIDENT), (512, RESIDENT), (513, TILED)]), (4, 1984, [(512, RESIDENT), (600, TILED)]),
    (4, 1600, [(512, RESIDENT), (600, TILED)]), (4, 1536, [(600, RESIDENT), (768, RESIDENT), (800, TILED)]),
    (3, 2048, [(384, RESIDENT), (512, RESIDENT), (540, TILED)]), (3, 1536, [(700, RESIDENT), (800, TILED)]),
    (4, 2624, [(512, RESIDENT), (768, TILED)]), (4, 512, [(1536, TILED), (1600, RESIDENT), (1800, TILED)]),
    (2, 2624, [(512, RESIDENT), (800, TILED)]), (1, 2624, [(1024, RESIDENT), (1060, TILED)]),
    (1, 64, [(2000, RESIDENT), (2100, TILED)]), (4, 64, [(4000, RESIDENT), (4200, TILED)]),
    # more streams: rows of another form of the resident kernel
    (5, 512, [(1150, TILED), (1250, RESIDENT), (1300, TILED)]), (5, 1664, [(460, RESIDENT), (540, TILED)]),
    (6, 896, [(600, RESIDENT), (768, RESIDENT), (1024, TILED)]), (6, 384, [(768, TILED), (1300, RESIDENT), (1500, TILED)]),
    (7, 896, [(768, RESIDENT), (1280, RESIDENT), (1700, TILED)]), (7, 1792, [(600, RESIDENT), (800, TILED)]),
    (8, 1792, [(1400, RESIDENT), (1800, TILED)]), (8, 3072, [(2000, RESIDENT)]), (8, 1024, [(1024, RESIDENT), (1060, TILED)]),
    (8, 960, [(8000, RESIDENT)]), (8, 1025, [(8000, RESIDENT)]),  # C % 64 != 0: always the resident path
])
def test_backward_of_float32_storage(n, C, rows):
    for B, want in rows:
        assert _route(BACKWARD, F32_AS_BF16, B, n, C) == want, B
