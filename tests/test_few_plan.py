"""Which forward calls the few-row kernel takes, and how it cuts them (caifx_gemm_few_plan.hpp)."""
import itertools

INT4, INT8, INT8_ONE = 0, 1, 2


# (rows, columns, reduction, kind): us tiled / here, repeated and with other code in between
#   17.6 / 19.7, 17.6 / 21.1;  19.6 / 18.8, 19.5 / 21.8;  19.8 / 20.3, 18.9 / 21.4;  20.4 / 20.2, 18.8 / 21.5;  20.3 / 21.3, 21.5 / 22.8;
#   19.6 / 20.0, 20.6 / 21.6;  23.4 / 21.2, 21.0 / 22.5
def test_calls_that_the_tiled_kernel_takes_as_fast(few_plans):
    calls = [(97, 2752, 4096, INT4), (100, 4096, 4096, INT4), (398, 960, 4096, INT4), (778, 512, 4096, INT4), (444, 1024, 3968, INT8),
             (816, 512, 3840, INT8), (490, 1024, 4096, INT8)]
    assert not any(parts for _, _, parts, _ in few_plans(calls))


#   22.5 / 18.2;  20.7 / 17.3;  23.0 / 20.2;  25.8 / 21.5;  18.1 / 16.7;  20.2 / 17.9;  41 / 23 (one scale)
def test_calls_that_it_takes(few_plans):
    calls = [(64, 4096, 4096, INT4), (248, 3584, 2048, INT4), (183, 2112, 4096, INT4), (698, 704, 4096, INT8), (881, 448, 3968, INT4),
             (531, 768, 3200, INT8), (444, 1024, 3968, INT8_ONE)]
    assert all(parts for _, _, parts, _ in few_plans(calls))


def test_every_plan_is_one_round_and_fits_the_tiled_kernels_room(few_plans):
    calls = [c for c in itertools.product([17, 32, 33, 100, 112, 113, 255, 700, 1024, 28672], [8, 64, 200, 1024, 4096, 8456, 16384],
                                          [512, 640, 1152, 4096, 14336], [INT4, INT8, INT8_ONE])]
    taken = 0
    for (M, N, K, kind), (row_tiles, blocks, parts, units) in zip(calls, few_plans(calls)):
        if parts == 0:
            continue
        taken += 1
        total = K // (128 if kind == INT4 else 64)
        assert 2 <= blocks <= 7 and 16 * blocks * row_tiles >= M > 16 * blocks * (row_tiles - 1)
        assert row_tiles * -(-N // 64) * parts <= 256 and (parts - 1) * units < total <= parts * units
        if parts > 1:      # up to 8 parts of at least 8 steps of 64 for at most 128 tiles of 128 x 128
            tiles = -(-M // 128) * -(-N // 128)
            assert tiles <= 128 and parts <= min(256 // tiles, 8, K // 64 // 8)
    assert taken > 300
