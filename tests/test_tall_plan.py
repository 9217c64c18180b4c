"""Heights of the row tiles of grouped int8 products (caifx_gemm_tall_plan.hpp), which the host chooses without knowing the segments."""
import itertools

# (rows, experts, columns, reduction): us with heights of 64, 96 .. 256, segments drawn uniformly or unevenly; where the number of tiles taken
# at its mean misses a second round
MEASURED = {
    (5472, 16, 896, 1280): [38.1, 41.3, 25.3, 27.2, 29.2, 31.5, 38.4], (5616, 16, 1024, 512): [24.0, 25.4, 16.6, 17.7, 18.8, 19.2, 24.5],
    (5874, 33, 1024, 512): [23.6, 25.1, 16.3, 17.4, 18.0, 20.1, 25.4], (3552, 16, 1024, 512): [23.6, 14.3, 15.3, 16.6, 16.0, 18.7, 22.5],
    (23232, 64, 256, 1280): [39.9, 43.3, 26.5, 28.6, 30.1, 31.7, 31.3], (7968, 12, 512, 1024): [33.6, 19.8, 21.6, 23.3, 24.9, 27.3, 33.4],
    (8118, 33, 1536, 1024): [64.7, 54.1, 43.3, 43.9, 46.4, 49.9, 57.0], (3824, 16, 896, 1280): [38.6, 22.9, 24.8, 27.0, 28.9, 31.2, 30.8],
    (9100, 5, 1408, 512): [44.0, 36.4, 29.0, 31.4, 34.0, 36.4, 28.7], (3888, 16, 1408, 512): [23.4, 23.9, 16.3, 16.8, 16.7, 19.5, 24.4]}


def test_a_round_that_segments_may_begin_is_counted(tall_plans):
    for (call, us), (height, _) in zip(MEASURED.items(), tall_plans(list(MEASURED))):
        assert us[(int(height) - 64) // 32] <= 1.12 * min(us), (call, height)


def test_heights_over_the_range(tall_plans):
    calls = list(itertools.product([0, 1, 17, 100, 999, 24576, 1 << 20, 1 << 30], [1, 2, 33, 64, 65, 4096], [256, 640, 14336], [256, 1408, 1 << 22]))
    for call, (height, us) in zip(calls, tall_plans(calls)):
        assert height in range(64, 257, 32) and 0.0 < us < float("inf"), call
