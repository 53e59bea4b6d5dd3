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
    (3, 16384, 1056),
]


def _check(gpu, x, w, wdt):
    """``x`` (rows farther apart than they are long) times ``w`` against std::fma, written and added."""
    (M, K), N = x.shape, w.shape[0]
    want = ps.linear(x.contiguous().numpy(), w.float().numpy())
    out = torch.full((M, N + 4), 5.0, device=gpu)
    wide = torch.zeros(M, K + 8)
    wide[:, :K] = x
    there, weight = wide.to(gpu)[:, :K], w.to(wdt).to(gpu)
    ops.gemm_f32(there, weight, out[:, :N], M)
    got = out.cpu().numpy()
    assert np.array_equal(got[:, :N].view(np.uint32), want.view(np.uint32))
    assert (got[:, N:] == 5.0).all()
    ops.gemm_f32(there, weight, out[:, :N], M, accumulate=True)
    assert np.array_equal(out.cpu().numpy()[:, :N], want + want)
    return want


@pytest.mark.parametrize("M,N,K", SHAPES)
@pytest.mark.parametrize("wdt", [torch.bfloat16, torch.float32])
def test_few_rows_are_the_scalar_chains(gpu, M, N, K, wdt):
    g = torch.Generator().manual_seed(M * 31 + N + K)
    x, w = torch.randn(M, K, generator=g), (torch.randn(N, K, generator=g) * 0.2).to(wdt)
    want = _check(gpu, x, w, wdt)
    # (what a missing, repeated or exchanged step of k would give is another number in nearly every output)
    swapped = x.clone()
    swapped[:, [0, K - 1]] = x[:, [K - 1, 0]]
    assert (ps.linear(swapped.numpy(), w[:8].float().numpy()) != want[:, :8]).mean() > 0.5


# a shape for every kernel that takes a 32-bit product
KERNELS = [(1, 33, 64), (8, 40, 192), (1, 16385, 128), (4, 16330, 128), (8, 16390, 64), (9, 8256, 128), (20, 4128, 128), (40, 16400, 64), (5, 40, 72),
           (30, 50, 72), (70, 200, 96), (100, 130, 48), (1000, 2040, 64), (257, 300, 64)]


@pytest.mark.parametrize("M,N,K", KERNELS)
@pytest.mark.parametrize("wdt", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("kind", ["denormal sums", "denormal operands", "cancelling", "infinite", "zeros"])
def test_special_values_are_the_scalar_chains(gpu, M, N, K, wdt, kind):
    g = torch.Generator().manual_seed(M + N + K)
    x, w = torch.randn(M, K, generator=g), (torch.randn(N, K, generator=g) * 0.2).to(wdt).float()
    if kind == "denormal sums":                                 # products of about 1e-41: sums that are denormal throughout
        x, w = x * 1e-20, (w * 5e-21).to(wdt).float()
    elif kind == "denormal operands":
        x = x * 1e-40
    elif kind == "cancelling":                                  # huge steps next to each other take each other back: their order shows
        at = torch.randint(0, K // 2, (M,), generator=g) * 2
        w[:, 1::2] = w[:, 0::2]
        rows = torch.arange(M)
        x[rows, at], x[rows, at + 1] = 1e7, -1e7
    elif kind == "infinite":                                    # one a row: no sum is the difference of two
        x[torch.arange(M), torch.randint(0, K, (M,), generator=g)] = float("inf")
        w[w == 0] = 1.0
    else:
        x[:] = torch.where(torch.rand(M, K, generator=g) < 0.5, 0.0, -0.0)
    want = _check(gpu, x, w, wdt)
    if kind.startswith("denormal"):
        assert (want != 0).mean() > 0.9 and (np.abs(want) < np.finfo(np.float32).tiny).all()
    elif kind == "infinite":
        assert np.isinf(want).all()
