"""SwiGLU in the 32-bit product's epilogue: the bits of the product and the activation as two kernels, for every kernel that the rules
choose, at the edges of its tiles, and where no tile takes the product."""

import pytest
import torch

from bitwise_amd.csrc import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("rows,inter,K,offset", [
    (1, 8192, 64, 0), (8, 4104, 128, 0), (16, 4097, 192, 0),           # tiles of 16 x 64; outputs that fill no block
    (17, 3001, 64, 0), (32, 4100, 320, 0),                             # 32 x 32
    (33, 8200, 64, 0), (64, 8193, 128, 0),                             # 64 x 64 of few rows
    (65, 97, 32, 0), (100, 1000, 96, 0), (450, 1021, 64, 0),           # 64 x 64 and 128 x 64 of a prompt
    (300, 4099, 32, 0), (1000, 2050, 96, 0), (2050, 700, 64, 0),       # 128 x 128, and three 64 x 64 a compute unit
    (1, 8200, 1024, 0), (4, 8193, 128, 0), (8, 18000, 64, 0),             # more than 8,192 outputs: the epilogue or two kernels
    (8, 200, 256, 0), (3, 4104, 100, 0), (70, 130, 50, 0), (70, 130, 64, 1), (9, 5000, 96, 0),   # strips; no tile
])
def test_bits_of_two_kernels(gpu, dtype, rows, inter, K, offset):
    g = torch.Generator(device=gpu).manual_seed(rows + inter + K)
    x = torch.randn(rows, K + offset + (-(K + offset)) % 4, generator=g, device=gpu)[:, offset:offset + K]
    w = (torch.randn(2 * inter, K, generator=g, device=gpu) * 2 * K ** -0.5).to(dtype)
    x[0, 0] = -200.0                                                   # (gates far out: the exponential's ends)
    sums = torch.empty(rows, 2 * inter, device=gpu)
    want = torch.empty(rows, inter, device=gpu)
    ops.gemm_f32(x, w, sums, rows)
    ops.swiglu_f32(sums, want, rows)
    got = torch.full((rows + 1, inter), 7.0, device=gpu)
    ops.gemm_f32_swiglu(x, w, torch.empty_like(sums), got, rows)
    assert torch.equal(got[:rows].view(torch.int32), want.view(torch.int32)) and bool((got[rows] == 7.0).all())
