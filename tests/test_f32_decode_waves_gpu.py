"""32-bit decode attention in workgroups of four and of eight waves: the same bits for a row, whichever the launch's size picks, at the
edges of the chunks of keys; and near the softmax in 64 bits."""

import pytest
import torch

from bitwise_amd.csrc import ops

pytestmark = pytest.mark.gpu
PAGE = 16


@pytest.mark.parametrize("hd,chunk", [(16, 256), (160, 48), (192, 40), (224, 36), (256, 32)])
@pytest.mark.parametrize("window,sinks", [(0, False), (0, True), (50, False)])
def test_four_and_eight_waves(gpu, hd, chunk, window, sinks):
    lens = [n for m in (1, 2, 3, 4, 7) for n in (m * chunk - 1, m * chunk, m * chunk + 1)] + [1, 2, 17, 64, 65]
    heads, kv_heads = 14, 7
    rows, per = len(lens), -(-max(lens) // PAGE) + 3
    assert rows * heads > 256
    g = torch.Generator(device=gpu).manual_seed(hd + window)
    need = [-(-n // PAGE) for n in lens]
    k = torch.randn(sum(need), kv_heads, PAGE, hd, generator=g, device=gpu)
    v = torch.randn(sum(need), kv_heads, PAGE, hd, generator=g, device=gpu)
    order = torch.randperm(sum(need), generator=g, device=gpu).int()
    table, at = torch.zeros(rows, per, dtype=torch.int32, device=gpu), 0
    for i, n in enumerate(need):
        table[i, :n] = order[at:at + n]
        at += n
    q = torch.randn(rows, heads * hd, generator=g, device=gpu)
    positions = torch.tensor([n - 1 for n in lens], dtype=torch.int32, device=gpu)
    positions[3] = -1                                                   # a padding row
    seq = torch.arange(rows, dtype=torch.int32, device=gpu)
    sink = torch.randn(heads, generator=g, device=gpu) if sinks else None

    def run(first, count, table):
        out = torch.full((count, heads * hd), 7.0, device=gpu)
        ops.attention_f32(q[first:first + count], positions[first:first + count], seq[:count], table[first:first + count].contiguous(), k, v, out, count,
                          heads, kv_heads, hd, PAGE, window, hd ** -0.5, sink=sink)
        return out

    capacity = window or per * PAGE
    assert ops.attention_f32_waves(hd, rows * heads, capacity) == 4
    assert ops.attention_f32_waves(hd, 5 * heads, capacity) == (4 if window and hd >= 160 else 8)
    many = run(0, rows, table)
    few = torch.cat([run(a, min(5, rows - a), table) for a in range(0, rows, 5)])
    assert torch.equal(many.view(torch.int32), few.view(torch.int32)) and bool((many[3] == 7.0).all())
    if not window:                                                      # tables of at most 64 keys
        short = run(rows - 4, 3, table[:, :4])
        assert torch.equal(short.view(torch.int32), many[rows - 4:rows - 1].view(torch.int32))
    for i, n in enumerate(lens):
        if i == 3:
            continue
        lo = max(0, n - window) if window else 0
        pages = table[i, :need[i]].long()
        keys = k[pages].transpose(0, 1).reshape(kv_heads, -1, hd)[:, lo:n].double()
        values = v[pages].transpose(0, 1).reshape(kv_heads, -1, hd)[:, lo:n].double()
        s = (q[i].view(kv_heads, 2, hd).double() * hd ** -0.5) @ keys.transpose(1, 2).contiguous()
        if sinks:
            s = torch.cat([s, sink.view(kv_heads, 2, 1).double()], 2)
        want = (torch.softmax(s, -1)[:, :, :n - lo] @ values).reshape(-1)
        # (sums of up to 1,793 terms in 32 bits)
        assert (many[i].double() - want).norm() <= 1e-5 * want.norm()
