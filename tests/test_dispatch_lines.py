"""Which launch path a call takes, on either side of the lines at which two paths cost the same (mhc_tuning_route of the tuning
build: the built-in rules, no GPU needed).  Every row is a size at which one of the two was measured to be the faster one; the
figures stand beside the rules (csrc/capi.hip, csrc/layer_fwd_held.hip, csrc/layer_fwd_onepass.hip,
csrc/mix_bwd_reduce.hip)."""
import subprocess
import sys

import pytest

F32, BF16, F32_AS_BF16 = 0, 1, 2
BACKWARD, FORWARD, SUMS = 0, 1, 2
RESIDENT, TILED = 0, 1
TWO, ONE, ONE_READS, HELD = 0, 1, 2, 3
APART, FUSED, WAVE = 0, 1, 2

_CHILD = """
import ctypes, sys
lib = ctypes.CDLL(sys.argv[1])
for line in sys.stdin:
    print(lib.mhc_tuning_route(*map(int, line.split())), flush=True)
"""


@pytest.fixture(scope="module")
def route():
    """In a process of its own: this one keeps to the product library."""
    import os

    from mhc import _lib

    path = os.path.join(os.path.dirname(_lib.LIB_PATH), "libmhc_hip_tuning.so")
    child = subprocess.Popen([sys.executable, "-c", _CHILD, path], stdin=subprocess.PIPE, stdout=subprocess.PIPE, text=True)

    def ask(*query):
        child.stdin.write(" ".join(map(str, query)) + "\n")
        child.stdin.flush()
        return int(child.stdout.readline())

    yield ask
    child.stdin.close()
    assert child.wait(timeout=60) == 0


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
def test_backward_of_float32_storage(route, n, C, rows):
    for B, want in rows:
        assert route(BACKWARD, F32_AS_BF16, B, n, C) == want, B


@pytest.mark.parametrize("dtype,n,C,rows", [
    (F32, 2, 640, [(1000, TWO), (1060, HELD)]), (F32, 2, 896, [(1000, TWO), (1150, TWO), (1500, HELD)]),
    (F32, 2, 1152, [(1100, TWO), (1250, HELD)]), (F32, 2, 1664, [(1150, TWO), (1300, HELD)]), (F32, 2, 2560, [(1000, TWO), (1060, HELD)]),
    (F32, 3, 576, [(1150, TWO), (1250, HELD)]), (F32, 3, 768, [(1200, TWO), (1500, HELD)]), (F32, 3, 1152, [(1100, TWO), (1250, HELD)]),
    (F32, 4, 448, [(1950, TWO), (2100, HELD)]), (F32, 4, 1280, [(1500, TWO), (1850, HELD)]),
    (F32_AS_BF16, 3, 576, [(1700, TWO), (2100, HELD)]), (F32_AS_BF16, 3, 1024, [(1700, TWO), (1850, HELD)]),
    (F32_AS_BF16, 3, 1152, [(1500, TWO), (1600, HELD)]), (F32_AS_BF16, 4, 320, [(2300, TWO), (2400, HELD)]),
    (F32_AS_BF16, 4, 1536, [(1150, TWO), (1330, HELD)]),
    # the one-launch forward: phi up to 120 KB, up to 150, up to 256, and beyond
    (BF16, 4, 256, [(7, ONE_READS), (4000, ONE_READS), (4200, HELD)]), (BF16, 4, 64, [(5000, ONE)]),
    (BF16, 4, 704, [(1024, TWO), (1100, ONE_READS)]), (BF16, 3, 1600, [(1024, TWO), (1100, ONE_READS)]),
    (BF16, 2, 4096, [(1024, TWO), (1100, ONE_READS)]), (BF16, 2, 5120, [(1024, TWO), (1100, ONE)]),
    (BF16, 2, 6144, [(1100, TWO)]), (BF16, 4, 1280, [(1100, TWO), (1280, TWO), (1400, ONE), (2048, ONE)]),
    (BF16, 3, 2560, [(1200, TWO), (1300, ONE)]), (BF16, 4, 1408, [(1400, TWO)]),
])
def test_forward(route, dtype, n, C, rows):
    for B, want in rows:
        assert route(FORWARD, dtype, B, n, C) == want, B


@pytest.mark.parametrize("n,C,rows", [
    (1, 512, [(1500, FUSED), (4096, WAVE), (4200, APART)]), (4, 768, [(1000, FUSED), (4096, WAVE), (4200, APART)]),
    (4, 1280, [(700, FUSED), (2560, WAVE)]), (1, 1600, [(1100, WAVE)]), (1, 1920, [(1100, APART), (1500, WAVE)]),
    (1, 2816, [(1300, APART), (1800, WAVE)]), (1, 3072, [(2000, APART)]), (2, 3072, [(1100, APART), (1400, WAVE)]),
    (2, 2048, [(600, APART), (700, FUSED)]), (5, 1600, [(384, APART), (400, FUSED), (800, APART)]),
    (5, 1280, [(450, APART), (540, FUSED)]), (6, 2112, [(450, APART), (540, FUSED)]), (5, 1285, [(450, APART), (540, APART)]), (2, 1283, [(800, APART)]),
    (4, 128, [(4311, APART)]), (6, 640, [(1000, FUSED), (1100, APART)]),
])
def test_channel_sums_of_the_float32_tier(route, n, C, rows):
    for B, want in rows:
        assert route(SUMS, F32, B, n, C) == want, B


@pytest.mark.parametrize("n,C,rows", [(7, 192, [(2126, RESIDENT), (2400, RESIDENT), (3000, TILED)]), (7, 256, [(2400, RESIDENT), (3000, TILED)]),
                                      (8, 320, [(1500, RESIDENT), (1600, TILED)]), (8, 512, [(1500, TILED)])])
def test_backward_of_bf16_storage(route, n, C, rows):
    for B, want in rows:
        assert route(BACKWARD, BF16, B, n, C) == want, B
