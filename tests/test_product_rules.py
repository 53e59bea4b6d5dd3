"""The rules that choose how a bfloat16 product of many rows is laid out: host code, asked through the library's queries."""

import random

import pytest

from bitwise_amd.csrc import ops

GATED_TILES = {(128, 128), (128, 256), (160, 256), (192, 256), (256, 256), (128, 64), (64, 128)}


def sizes(n, seed):
    rng = random.Random(seed)
    for _ in range(n):
        yield rng.randint(65, 2048), int(2 ** rng.uniform(6, 14)), 64 * max(1, int(2 ** rng.uniform(0, 7.8)))


def test_every_tile_a_rule_gives_is_one_that_the_gpu_tests_cover():
    for M, N, K in sizes(4000, 1):
        assert ops.gemm_prompt_tile(M, N, K) in GATED_TILES | {(256, 192)}
        assert ops.gemm_prompt_tile(M, 2 * N, K, gated=True) in GATED_TILES
        if K > 2048:
            assert ops.gemm_prompt_tile(M, N, K) != (256, 256), "no registers there for the sums of earlier segments"


def test_few_rows_of_a_long_inner_size_do_not_take_64_x_128_tiles_where_128_x_64_pull_the_weights_faster():
    # 320 rows of 4096 x 4096: 29 us and 25; of K = 14336 101 and 78
    assert ops.gemm_prompt_tile(320, 4096, 4096) == ops.gemm_prompt_tile(320, 4096, 14336) == (128, 64)


def test_tiles_of_one_or_two_steps_along_k():
    # 1,600 rows of 2048 columns, K = 64: 5.1 us in 128 x 128, 6.5 in 128 x 256
    assert ops.gemm_prompt_tile(1600, 2048, 64) == ops.gemm_prompt_tile(700, 4096, 128) == (128, 128)


@pytest.mark.parametrize("M,N,K", [(257, 14336, 512), (450, 14336, 512), (777, 8192, 512), (450, 8192, 256)])
def test_part_empty_rounds_of_a_short_inner_size_do_not_take_the_larger_of_two_tiles(M, N, K):
    # (160 x 256 took 8 to 12 % longer; 450 x 8192 x 256 with rotation 12.8 us for 9.1)
    assert ops.gemm_prompt_tile(M, N, K) in ((128, 256), (128, 128))
