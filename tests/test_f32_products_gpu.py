"""32-bit products of up to 64 rows: every kernel that the rule on rows, columns and K picks, at the edges of its rows, columns and
stages, against the scalar std::fma program, bit for bit."""

import numpy as np
import pytest
import torch

import plain_scalar as ps
from bitwise_amd.csrc import ops

pytestmark = pytest.mark.gpu

SHAPES = [
    # strips of 32 columns: one to five stages, columns around a strip and a half strip, row blocks around 16, 32, 48
    (1, 1, 64), (3, 31, 128), (8, 32, 192), (15, 33, 256), (16, 2048, 64), (17, 47, 320), (33, 96, 64), (48, 65, 192), (64, 49, 704), (16, 8192, 64),
    # 16 x 64 tiles: more than 256 strips of up to 16 rows
    (2, 8193, 64), (9, 8256, 128), (16, 8255, 384), (16, 16384, 448),
    # 32 x 32 tiles: 17 rows and more
    (17, 4097, 64), (31, 4128, 128), (33, 2754, 320), (49, 2080, 192), (64, 2049, 64),
    # 64 x 64 tiles: 33 rows and more of many columns, and K in stages of 32 only
    (33, 16384, 64), (64, 16400, 192), (17, 50, 96), (40, 200, 32), (5, 16390, 96),
    # chains: up to eight rows of many columns (two to eight with 32-bit weights, some with bfloat16 ones)
    (1, 16385, 128), (1, 16321, 704), (2, 16385, 64), (3, 16330, 128), (4, 16449, 1024), (5, 16400, 256), (7, 16385, 96), (8, 16390, 192),
]


@pytest.mark.parametrize("M,N,K", SHAPES)
@pytest.mark.parametrize("wdt", [torch.bfloat16, torch.float32])
def test_few_rows_are_the_scalar_chains(gpu, M, N, K, wdt):
    g = torch.Generator().manual_seed(M * 31 + N + K)
    wide = torch.randn(M, K + 8, generator=g)
    wide[0, :4] = torch.tensor([-0.0, 1e-38, -3e38, 1e-42])
    w = (torch.randn(N, K, generator=g) * 0.2).to(wdt)
    want = ps.linear(wide[:, :K].contiguous().numpy(), w.float().numpy())
    out = torch.full((M, N + 4), 5.0, device=gpu)
    x = wide.to(gpu)[:, :K]                                     # rows farther apart than they are long
    ops.gemm_f32(x, w.to(gpu), out[:, :N], M)
    got = out.cpu().numpy()
    assert np.array_equal(got[:, :N].view(np.uint32), want.view(np.uint32))
    assert (got[:, N:] == 5.0).all()
    ops.gemm_f32(x, w.to(gpu), out[:, :N], M, accumulate=True)
    assert np.array_equal(out.cpu().numpy()[:, :N], want + want)
