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
    lib.evo_test_hcs_stream_segment.argtypes = [size, size, ctypes.c_int]
    lib.evo_test_hcs_stream_segment.restype = ctypes.c_uint
    lib.evo_test_hcm_stream_two_groups.argtypes = [size, size, ctypes.c_int, ctypes.c_int]
    return lib


# (width, length, F32 rows and exact windows): us with segments of 16, 32, 64
# and 128 rows. BF16 rows with 5 taps (padded windows) or 7 (exact), F32 with 7.
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
]


@pytest.mark.parametrize("width,length,f32_exact,times", HCS_SEGMENTS)
def test_hcs_stream_segment(rules, width, length, f32_exact, times):
    rows = rules.evo_test_hcs_stream_segment(width, length, f32_exact)
    assert times[(16, 32, 64, 128).index(rows)] <= SLACK * min(times)


# (group size, length, taps, F32 rows): us tap by tap and on the row stream,
# with the caches.
HCM_TWO_GROUPS = [
    (15, 2, 40, 1, (18.1, 19.2)), (24, 2, 40, 1, (17.9, 19.1)), (17, 2, 40, 1, (18.0, 19.1)),
    (15, 5, 40, 1, (21.3, 20.8)), (15, 2, 128, 1, (29.7, 25.6)), (15, 17, 40, 1, (32.4, 23.1)),
    (15, 2, 128, 0, (31.2, 25.0)), (15, 5, 40, 0, (21.9, 20.0)),
]


@pytest.mark.parametrize("group_size,length,taps,f32,times", HCM_TWO_GROUPS)
def test_hcm_stream_two_groups(rules, group_size, length, taps, f32, times):
    streamed = rules.evo_test_hcm_stream_two_groups(group_size, length, taps, f32)
    assert times[streamed] == min(times)


def test_hcm_stream_leaves_small_groups(rules):
    """A slice of 16 channels may touch three groups of 14."""
    assert not rules.evo_test_hcm_stream_two_groups(14, 1000, 128, 0)
