"""The rules that choose how a bfloat16 product of many rows is laid out: host code, asked through the library's queries."""

import random

import pytest
import torch

from bitwise_amd.csrc import ops
from bitwise_amd.parts.linear import Linear

GATED_TILES = {(128, 128), (128, 256), (160, 256), (192, 256), (256, 256), (128, 64), (64, 128)}
SPLIT_TILES = {(128, 64), (128, 128), (128, 256), (160, 256), (192, 256), (256, 192), (256, 256)}


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
            for store in (False, True):
                tile = ops.gemm_split_tile.__wrapped__(M, 4 * (N // 4), K, store)
                assert tile is None or tile in SPLIT_TILES


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


def test_gated_gelu_in_the_epilogue_only_where_it_is_faster():
    # both ways timed, us behind the store and in the epilogue
    for (M, inter, K), wins in {(128, 512, 14336): False,         # 19.7 and 69.9
                                (192, 1024, 14336): False,        # 30.1 and 101
                                (65, 512, 2048): False,           # 7.2 and 13.6
                                (96, 512, 1024): False,           # 6.4 and 8.8
                                (128, 2048, 4096): False,         # 64 workgroups with all of K
                                (2048, 8192, 2048): True,         # 151 and 111
                                (117, 8192, 2048): True,
                                (2048, 512, 64): True, (65, 512, 72): True}.items():
        assert ops.gelu_glu_in_epilogue(M, inter, K) == wins, (M, inter, K)
    for M in (1, 16, 64):
        assert not ops.gelu_glu_in_epilogue(M, 8192, 2048)        # (no epilogue for steps of so few rows)


class Workspace:
    """Keeps what is asked of it, as the real one does: a buffer by name and size, for good."""

    def __init__(self, max_rows):
        self.max_rows, self.buffers = max_rows, {}

    def buffer(self, name, cols, dtype, rows=None):
        return self.buffers.setdefault((name, cols, dtype, rows), torch.empty(rows, cols, dtype=dtype, device="meta"))


@pytest.mark.parametrize("store", (False, True))
@pytest.mark.parametrize("N,K", [(2048, 8192), (4096, 14336), (8192, 4096), (4096, 4096), (2048, 2048)])
def test_scratch_for_a_split_is_held_only_where_products_split(N, K, store):
    """A product that goes whole brings no scratch (it held 67 MB for 2,048 rows of 2048 x 8192); those that split share one
    buffer, large enough for each of them; a few blocks of 64 rows at once keep theirs."""
    lin = object.__new__(Linear)
    lin.out_features, lin.in_features = N, K
    ws = Workspace(2048)
    split = 0
    for rows in range(65, 2049):
        got = lin._scratch(ws, rows, store)
        floats, counters = ops.gemm_add_scratch.__wrapped__(rows, N, K)
        if counters == 1 and ops.gemm_split_tile.__wrapped__(rows, N, K, store) is None:
            assert got is None
            continue
        assert (got is None) == (floats == 0)
        if got is not None:
            assert got[0].numel() >= floats and got[1].numel() >= counters
            split += counters == 1
    sums = {cols for name, cols, _, _ in ws.buffers if name == "gemm_add_split"}
    most = ops.gemm_split_rows(2048, N, K, store)
    assert len(sums) <= 1 and (split > 0) == (most > 0)
    if sums:
        assert sums == {max((K + 2047) // 2048 * most * N, 512 * 4096)}
    if (N, K) == (2048, 8192):
        assert lin._scratch(ws, 2048, store) is None and most < 2048


def test_the_most_rows_that_split():
    for N, K in ((2048, 8192), (4096, 14336), (8192, 4096)):
        for most in (2048, 1000, 300, 64):
            got = ops.gemm_split_rows(most, N, K)
            splits = [M for M in range(65, most + 1) if ops.gemm_split_tile.__wrapped__(M, N, K) is not None]
            assert got == max(splits, default=0)
    with pytest.raises(RuntimeError):
        ops.gemm_split_tile(100, 0, 4096)
