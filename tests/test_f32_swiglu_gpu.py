"""SwiGLU in the 32-bit product's epilogue: the bits of the product and the activation as two kernels, for every kernel that the rules
choose, at the edges of its tiles, and where no tile takes the product."""

import pytest
import torch

from bitwise_amd.csrc import ops
from bitwise_amd.parts.linear import Linear
from bitwise_amd.parts.mlp import SwiGLU
from bitwise_amd.runtime import Runtime, Workspace

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


def _feed_forward(gpu, width, inter, bias=None):
    rt = Runtime("float32", gpu)
    g = torch.Generator(device=gpu).manual_seed(width)
    part = SwiGLU({"width": width, "inter": inter}, rt)
    part.bind({n: torch.randn(*s.shape, generator=g, device=gpu) * 0.1 for n, s in part.tensors().items()})
    if bias is not None:
        part.gate_up = Linear(part.gate_up.weight, rt, bias=bias)
    return part, torch.randn(300, width, generator=g, device=gpu)


def test_no_room_is_held_for_sums_that_never_reach_memory(gpu):
    width, inter = 256, 4200
    part, x = _feed_forward(gpu, width, inter)
    ws = Workspace(gpu, max_rows=300, page_size=16)
    act = torch.empty(300, inter, device=gpu)
    for rows in (1, 8, 40, 64, 65, 300):
        part.gate_up.store_swiglu(ws, x, act, rows)
    assert ws.nbytes() == 0
    small, y = _feed_forward(gpu, 128, 200)                             # strips up to 64 rows, tiles for more
    for rows in (1, 64, 65, 300):
        small.gate_up.store_swiglu(ws, y, act.view(-1)[:300 * 200].view(300, 200), rows)
    assert ws.nbytes() == 64 * 2 * 200 * 4


def test_a_bias_of_the_stacked_projection_counts(gpu):
    width, inter = 256, 4200
    bias = torch.linspace(-1, 1, 2 * inter, device=gpu)
    part, x = _feed_forward(gpu, width, inter, bias)
    ws, act, want = Workspace(gpu, max_rows=300, page_size=16), torch.empty(300, inter, device=gpu), torch.empty(300, inter, device=gpu)
    sums = torch.empty(300, 2 * inter, device=gpu)
    part.gate_up.store(ws, x, sums, 300)
    ops.swiglu_f32(sums, want, 300)
    for rows in (300, 40):
        act.zero_()
        part.gate_up.store_swiglu(ws, x, act, rows)
        assert torch.equal(act[:rows].view(torch.int32), want[:rows].view(torch.int32))
