"""The rules by which launches choose their shape, on the CPU: each against
times measured on an MI355X, so that a change of a rule shows where it gives
time away. The choice has to be within 6 % of the fastest measured one (the
spread of repeated measurements is about 3 %)."""
import ctypes
import os

import pytest

LIB = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "evo.cpp_amd",
                   "lib", "libevo_hip_testing.so")
SLACK = 1.06


@pytest.fixture(scope="module")
def rules():
    lib = ctypes.CDLL(LIB)
    size = ctypes.c_size_t
    lib.evo_test_hcs_stream_segment.argtypes = [size, size] + 3 * [ctypes.c_int]
    lib.evo_test_hcs_stream_segment.restype = ctypes.c_uint
    lib.evo_test_hcm_stream_two_groups.argtypes = [size, size] + 3 * [ctypes.c_int]
    lib.evo_test_linear_plan.argtypes = [size, size, size, ctypes.c_int, ctypes.c_int, size,
                                         ctypes.POINTER(ctypes.c_int), ctypes.POINTER(size)]
    lib.evo_test_linear_plan_ns.argtypes = 4 * [size] + [ctypes.c_int]
    lib.evo_test_linear_plan_ns.restype = ctypes.c_double
    lib.evo_test_fp8_tile.argtypes = [size, size, size, ctypes.c_int]
    return lib


# (width, length, kind): us with segments of 16, 32, 64 and 128 rows. Kinds:
# 0 BF16 rows, 5 taps (padded windows) or 7 (exact); 1 F32 rows, 7 taps, 16-bit
# outputs; 2 F32 rows and outputs, 7 taps; 3 those with 5 taps.
HCS_KINDS = [(0, 0, 0), (1, 1, 0), (1, 1, 1), (1, 0, 1)]  # F32 rows, exact, F32 outputs
HCS_SEGMENTS = [
    (4096, 130, 0, (8.7, 11.6, 17.4, 28.9)), (4096, 611, 0, (11.2, 12.2, 17.7, 29.2)),
    (4096, 1024, 0, (12.6, 13.1, 18.1, 29.3)), (4096, 1500, 0, (18.9, 16.1, 18.7, 29.6)),
    (4096, 3000, 0, (31.5, 27.6, 24.1, 31.0)), (4096, 4096, 0, (40.0, 32.9, 25.4, 31.3)),
    (4096, 8192, 0, (73.2, 60.0, 51.8, 43.6)), (960, 6000, 0, (19.1, 16.0, 18.6, 29.5)),
    (4096, 2049, 0, (26.0, 25.6, 23.3, 30.1)), (4096, 2049, 0, (19.5, 17.4, 17.3, 21.0)),
    (4096, 3000, 0, (25.2, 20.8, 19.2, 23.6)), (4096, 8192, 0, (52.2, 51.6, 44.3, 39.9)),
    (1920, 6000, 0, (22.8, 20.0, 19.0, 23.4)), (1920, 8192, 0, (28.1, 26.0, 23.0, 25.1)),
    (4096, 611, 1, (12.5, 12.0, 17.7, 30.2)), (4096, 2049, 1, (32.5, 29.7, 34.0, 39.4)),
    (4096, 3000, 1, (39.9, 33.6, 35.7, 41.5)), (4096, 6000, 1, (72.6, 63.1, 57.4, 62.9)),
    (1920, 611, 1, (8.9, 11.7, 18.3, 31.4)), (1920, 6000, 1, (38.0, 32.9, 34.6, 39.9)),
    (4096, 3500, 1, (43.9, 39.5, 32.4, 32.7)), (4096, 4000, 1, (55.7, 50.5, 50.9, 51.2)),
    (4096, 950, 2, (17.7, 18.0, 22.0, 34.9)), (4096, 1100, 2, (17.4, 16.9, 16.2, 25.3)),
    (4096, 1800, 2, (29.8, 28.9, 26.9, 37.8)), (4096, 2700, 2, (43.1, 40.4, 41.0, 42.7)),
    (4096, 3000, 2, (39.5, 36.1, 31.9, 31.8)), (4096, 3500, 2, (54.6, 50.4, 46.1, 46.0)),
    (4096, 1800, 3, (36.1, 31.3, 29.1, 40.0)), (4096, 3000, 3, (53.4, 52.2, 45.1, 46.5)),
]


@pytest.mark.parametrize("width,length,kind,times", HCS_SEGMENTS)
def test_hcs_stream_segment(rules, width, length, kind, times):
    rows = rules.evo_test_hcs_stream_segment(width, length, *HCS_KINDS[kind])
    assert times[(16, 32, 64, 128).index(rows)] <= SLACK * min(times)


# (group size, length, taps, F32 rows, caches): us tap by tap and on the row
# stream.
HCM_TWO_GROUPS = [
    (15, 2, 40, 1, 1, (18.1, 19.2)), (24, 2, 40, 1, 1, (17.9, 19.1)),
    (17, 2, 40, 1, 1, (18.0, 19.1)), (15, 5, 40, 1, 1, (21.3, 20.8)),
    (15, 2, 128, 1, 1, (29.7, 25.6)), (15, 17, 40, 1, 1, (32.4, 23.1)),
    (15, 2, 128, 0, 1, (31.2, 25.0)), (15, 5, 40, 0, 1, (21.9, 20.0)),
    (15, 2, 10, 0, 1, (14.2, 16.5)), (24, 4, 10, 0, 0, (8.3, 8.7)), (15, 7, 10, 0, 1, (16.7, 17.3)),
    (24, 4, 20, 0, 1, (15.6, 16.6)), (15, 2, 20, 0, 0, (8.9, 8.2)),
    (24, 3, 33, 0, 1, (17.0, 17.8)),
    (15, 7, 20, 0, 1, (18.4, 17.4)), (24, 2, 64, 0, 1, (21.1, 19.2)),
    (15, 3, 33, 1, 1, (16.5, 18.3)),
    (24, 4, 33, 1, 0, (8.6, 9.0)), (15, 4, 40, 1, 1, (17.7, 18.6)), (15, 5, 20, 1, 0, (9.6, 8.9)),
    (15, 5, 20, 1, 1, (17.3, 18.1)), (24, 3, 64, 1, 1, (19.9, 19.7)),
    (15, 5, 40, 1, 1, (20.6, 19.3)), (15, 3, 40, 1, 0, (9.5, 8.8)),
]


@pytest.mark.parametrize("group_size,length,taps,f32,caches,times", HCM_TWO_GROUPS)
def test_hcm_stream_two_groups(rules, group_size, length, taps, f32, caches, times):
    streamed = rules.evo_test_hcm_stream_two_groups(group_size, length, taps, f32, caches)
    assert times[streamed] == min(times)


def test_hcm_stream_leaves_small_groups(rules):
    """A slice of 16 channels may touch three groups of 14."""
    assert not rules.evo_test_hcm_stream_two_groups(14, 1000, 128, 0, 1)


LARGE = "256 x 256"
# (rows, N, K, activation planes, workspace or not): us of the fastest (block
# tile, K parts), and of choices the rule made before.
LINEAR = [
    (5, 22528, 4096, 2, 0, {(1, 1): 37.9, (4, 1): 38.2, (0, 1): 40.6, (6, 1): 41.7}),
    (16, 22528, 4096, 2, 0, {(4, 1): 38.7, (1, 1): 40.8, (6, 1): 42.3, (2, 1): 44.4, (0, 1): 48.8}),
    (32, 22528, 4096, 1, 0, {(4, 1): 39.1, (6, 1): 41.6, (2, 1): 42.5, (5, 1): 42.6, (1, 1): 49.8}),
    (61, 22528, 4096, 2, 0, {(6, 1): 50.4, (4, 1): 56.9, (8, 1): 57.5, (7, 1): 60.2}),
    (300, 22528, 4096, 2, 0, {(6, 1): 146.2, (7, 1): 146.7, (9, 1): 161.0, LARGE: 162.6}),
    (16, 12288, 4096, 2, 0, {(3, 1): 23.5, (1, 1): 25.0, (5, 1): 26.9, (4, 1): 27.0, (0, 1): 27.8}),
    (24, 12288, 4096, 1, 0, {(3, 1): 22.4, (5, 1): 25.1, (2, 1): 26.1, (4, 1): 26.2}),
    (48, 512, 4096, 1, 1, {(1, 4): 8.3, (2, 4): 8.7, (0, 4): 8.7, (0, 2): 8.8, (1, 8): 9.4}),
    (128, 512, 4096, 2, 1, {(2, 4): 9.7, (0, 1): 10.3, (1, 2): 10.5, (3, 8): 10.6}),
    (300, 512, 1920, 2, 0, {(2, 1): 8.6, (1, 1): 10.0, (3, 1): 10.5, (4, 1): 12.7}),
    (5, 4096, 11264, 2, 1, {(1, 2): 20.6, (1, 4): 21.6, (0, 1): 21.9, (3, 4): 22.0}),
    (32, 4096, 11264, 1, 1, {(3, 4): 21.6, (5, 4): 22.3, (2, 2): 22.4, (4, 4): 23.8, (1, 2): 27.2}),
    (61, 4096, 11264, 2, 0, {(2, 1): 38.4, (1, 1): 49.4, (3, 1): 52.0, (4, 1): 62.9}),
    (300, 4096, 11264, 2, 1, {(7, 2): 73.8, LARGE: 78.7, (8, 2): 80.7, (7, 4): 82.0}),
    (5, 1920, 5120, 2, 1, {(1, 4): 9.8, (0, 2): 10.0, (0, 4): 10.3, (2, 4): 10.5}),
    (61, 1920, 1920, 2, 1, {(1, 1): 8.1, (2, 1): 9.3, (2, 2): 9.5, (0, 1): 9.5}),
    (1000, 1920, 1920, 2, 1, {(6, 1): 22.5, (7, 1): 28.2, (8, 2): 28.2, (5, 1): 29.5}),
    (300, 4096, 4096, 2, 1, {(7, 2): 33.7, (6, 1): 36.5, (8, 2): 37.6, LARGE: 41.0}),
    (2000, 4096, 4096, 2, 1, {(8, 1): 123.8, (7, 1): 153.3, (8, 2): 158.8, (9, 1): 163.4}),
    (3000, 4096, 11264, 2, 0, {LARGE: 493.4, (8, 1): 525.9, (7, 1): 655.1, (6, 1): 670.8}),
    (1000, 22528, 4096, 2, 1, {LARGE: 313.5, (9, 1): 358.6, (8, 1): 360.3, (7, 1): 403.6}),
    (5000, 4096, 4096, 2, 0, {LARGE: 370.1, (7, 1): 377.8, (9, 1): 383.7, (8, 1): 407.3}),
    (4400, 4096, 11264, 2, 0, {(7, 1): 852.8, (6, 1): 979.6, (8, 1): 1011.9, LARGE: 1051.0}),
    (8192, 512, 4096, 2, 1, {LARGE: 79.0, (8, 1): 85.9, (6, 1): 91.5, (9, 1): 95.6}),
    (2500, 4096, 11264, 1, 1, {LARGE: 291.4, (8, 1): 308.9, (9, 1): 365.4, (6, 1): 396.5}),
    (5700, 4096, 11264, 1, 0, {LARGE: 627.8, (8, 1): 666.5, (7, 1): 786.1, (9, 1): 817.7}),
    (4096, 1920, 1920, 2, 0, {(8, 1): 81.8, (7, 1): 84.4, LARGE: 89.2, (6, 1): 91.4}),
    (1000, 512, 4096, 2, 1, {(6, 4): 21.2, (7, 4): 23.3, (8, 8): 24.6, (6, 2): 24.6, LARGE: 30.8}),
    (777, 4096, 11264, 1, 1, {(8, 1): 95.2, (8, 2): 108.0, LARGE: 112.8, (8, 4): 126.2, (6, 1): 139.4}),
    (100, 4096, 4096, 1, 1, {(3, 1): 16.0, (6, 4): 17.4, (5, 2): 17.8, (5, 4): 17.8, LARGE: 26.8}),
    (3000, 5760, 1920, 1, 0, {(8, 1): 116.1, (9, 1): 118.3, LARGE: 129.2, (7, 1): 131.9, (6, 1): 141.1}),
]


@pytest.mark.parametrize("m,n,k,planes,workspace,times", LINEAR)
def test_linear_tile(rules, m, n, k, planes, workspace, times):
    """Few rows are bound by the weight's bytes; which tile streams them
    fastest still differs by up to a third. The costs are fits with a median
    error of 2 to 6 %: within 10 % of the fastest here, and not above 256 x
    256."""
    parts, tail = ctypes.c_int(), ctypes.c_size_t()
    tile = rules.evo_test_linear_plan(m, n, k, planes == 2, 0, workspace << 26,
                                      ctypes.byref(parts), ctypes.byref(tail))
    choice = LARGE if tile < 0 else (tile, parts.value)
    assert choice in times and times[choice] <= 1.10 * min(times.values())
    assert times[choice] <= 1.02 * times.get(LARGE, times[choice])


# (rows, N, K, promotion every 128 K or 32): us on the six block tiles of the
# FP8 product, 128 x 192 first, weights that no cache holds.
FP8 = [
    (5, 12288, 4096, 1, (39.5, 33.9, 19.6, 13.5, 15.0, 13.1)),
    (64, 12288, 4096, 1, (40.7, 34.7, 21.0, 14.7, 16.3, 19.0)),
    (200, 12288, 4096, 1, (41.8, 34.6, 27.5, 29.3, 32.5, 41.1)),
    (300, 12288, 4096, 1, (40.9, 35.4, 30.0, 37.2, 41.8, 55.2)),
    (520, 12288, 4096, 1, (46.5, 67.9, 52.8, 59.8, 73.6, 89.0)),
    (640, 12288, 4096, 1, (50.0, 68.3, 55.8, 66.3, 72.7, 102.7)),
    (1024, 12288, 4096, 1, (56.2, 92.2, 78.7, 97.0, 110.8, 156.8)),
    (8192, 12288, 4096, 1, (418.5, 484.3, 550.4, 679.1, 727.7, 1178.4)),
    (130, 5760, 1920, 1, (21.5, 17.6, 10.9, 10.6, 8.5, 9.8)),
    (777, 5760, 1920, 1, (22.7, 19.4, 22.5, 25.0, 24.9, 34.8)),
    (1300, 5760, 1920, 1, (27.7, 35.2, 28.7, 35.3, 36.1, 54.3)),
    (2049, 5760, 1920, 1, (32.2, 39.4, 42.3, 52.4, 59.2, 83.3)),
    (1024, 3072, 1024, 1, (15.7, 12.2, 10.5, 11.7, 12.0, 17.0)),
    (16, 12288, 4096, 0, (51.2, 35.5, 24.6, 17.6, 18.0, 17.5)),
    (200, 12288, 4096, 0, (53.2, 44.4, 33.9, 35.5, 38.8, 54.1)),
    (400, 12288, 4096, 0, (54.3, 48.3, 52.8, 57.6, 60.3, 88.7)),
    (900, 12288, 4096, 0, (86.2, 90.8, 95.5, 113.0, 117.6, 187.2)),
    (3000, 12288, 4096, 0, (251.0, 261.9, 276.7, 327.3, 341.9, 591.4)),
    (640, 5760, 1920, 0, (28.9, 24.5, 19.9, 23.1, 24.8, 37.4)),
    (1300, 5760, 1920, 0, (41.8, 38.2, 35.3, 42.1, 43.1, 69.2)),
]


@pytest.mark.parametrize("m,n,k,k128,times", FP8)
def test_fp8_tile(rules, m, n, k, k128, times):
    tile = rules.evo_test_fp8_tile(m, n, k, k128)
    assert times[tile] <= SLACK * min(times) and times[tile] <= 1.02 * times[0]


def test_linear_choice_is_cheap(rules):
    """A product of a few rows is over in 6 us: the choice of its tile may not
    take a good part of that (0.55 us; 3.6 us with a root per candidate). The
    least of 20 batches, so that a busy host does not count."""
    times = [rules.evo_test_linear_plan_ns(5, 512, 4096, 1 << 26, 500) for _ in range(20)]
    assert min(times) < 1800
