"""The rules that choose how a 32-bit product is laid out: host code, held against the measured times of the kernels they choose from."""

import pytest
import torch

from bitwise_amd.csrc import ops

# bfloat16 weights, rows, columns, K, microseconds in tiles of the matrix cores, as chains
CHAINS = [(False, 2, 16321, 64, 3.9, 3.3), (False, 4, 16321, 1024, 12.7, 13.9), (False, 2, 18000, 64, 5.8, 3.7), (False, 2, 24000, 2048, 46.0, 41.4),
          (False, 4, 24000, 1024, 25.5, 24.0), (False, 2, 32768, 4096, 99.8, 119.4), (False, 8, 24000, 512, 13.1, 14.3),
          (False, 8, 65000, 256, 18.5, 15.5), (False, 6, 65000, 512, 31.4, 27.2), (False, 2, 100000, 64, 16.9, 9.2), (True, 2, 24000, 64, 4.4, 3.8),
          (True, 2, 100000, 1024, 42.6, 38.7), (True, 4, 100000, 64, 10.7, 9.7), (True, 4, 24000, 2048, 24.0, 25.2),
          (True, 8, 24000, 1024, 15.0, 22.4), (True, 8, 65000, 2048, 45.6, 90.3), (False, 2, 16384, 1824, 29.3, 24.4),
          (False, 8, 39549, 1824, 59.3, 53.2), (False, 6, 49152, 1056, 43.3, 39.2), (False, 8, 65000, 1824, 82.4, 88.0)]


@pytest.mark.parametrize("bf16,rows,columns,K,tiles,chains", CHAINS)
def test_few_rows_of_many_columns_go_the_faster_way(bf16, rows, columns, K, tiles, chains):
    assert ops.gemm_f32_by_chains(rows, columns, K, bf16) == (chains < tiles)


def test_chains_are_for_whole_stages_of_up_to_eight_rows_and_a_chip_of_columns():
    for bf16 in (False, True):
        assert all(ops.gemm_f32_by_chains(1, n, k, bf16) for n in (16321, 49152) for k in (64, 2048, 8192))
        assert not ops.gemm_f32_by_chains(9, 100000, 64, bf16) and not ops.gemm_f32_by_chains(1, 16320, 64, bf16)
        assert ops.gemm_f32_by_chains(1, 20000, 96, bf16) == (not bf16) and not ops.gemm_f32_by_chains(1, 20000, 80, bf16)


# bfloat16 weights, rows, outputs, K, microseconds with SwiGLU in the tiles' epilogue, in a kernel behind the product
SWIGLU = [(False, 1, 8192, 2048, 30.0, 32.3), (False, 1, 8200, 64, 6.1, 5.5), (False, 1, 8200, 4096, 68.3, 51.1), (False, 1, 16384, 1024, 42.4, 31.4),
          (False, 2, 50000, 256, 32.9, 23.9), (False, 1, 14336, 8192, 162.0, 212.8), (False, 8, 8200, 64, 6.5, 6.0), (False, 8, 16384, 256, 11.0, 11.4),
          (False, 8, 50000, 512, 49.1, 45.3), (True, 1, 8192, 2048, 16.3, 17.2), (True, 1, 8200, 4096, 42.5, 29.4), (True, 1, 9000, 1024, 14.4, 13.9),
          (True, 1, 14336, 1024, 14.6, 16.1), (True, 8, 8200, 1024, 14.1, 16.1)]


@pytest.mark.parametrize("bf16,rows,outputs,K,tiles,apart", SWIGLU)
def test_swiglu_goes_the_faster_way(bf16, rows, outputs, K, tiles, apart):
    w = torch.empty(2 * outputs, K, dtype=torch.bfloat16 if bf16 else torch.float32, device="meta")
    assert ops.gemm_f32_swiglu_in_tiles(torch.empty(rows, K, device="meta"), w, rows) == (tiles < apart)
