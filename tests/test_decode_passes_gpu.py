"""Decode attention at the edges of what a workgroup folds at once: one pass over a context's partials or several, split over
workgroups or not, the same bits; and near the softmax in 64 bits."""

import pytest
import torch

from bitwise_amd.csrc import ops

pytestmark = pytest.mark.gpu
PAGE = 16


@pytest.mark.parametrize("heads,kv_heads,hd,lens", [
    (4, 1, 128, (4500, 640)),              # 71 partitions of four heads: one pass
    (8, 2, 128, (64 * 72, 64 * 73, 64 * 74)),   # about what one pass takes
    (4, 1, 128, (64 * 150 + 1,)),          # several
    (2, 2, 64, (64 * 256, 64 * 257 + 5)),  # a workgroup's most partitions
    (8, 1, 96, (3001, 577)),
    (16, 1, 64, (2500,)),
    (1, 1, 16, (1500, 9)),                 # partials of 72 bytes: the last load of a pass is part empty
    (3, 3, 48, (1111, 705)),
    (2, 1, 256, (2000,)),
])
def test_passes_and_splits_give_the_same_bits(gpu, heads, kv_heads, hd, lens):
    g = torch.Generator(device=gpu).manual_seed(heads + hd + sum(lens))
    per = -(-max(lens) // PAGE)
    rows, need = len(lens), [-(-n // PAGE) for n in lens]
    k = torch.randn(sum(need), kv_heads * PAGE * hd, generator=g, device=gpu).bfloat16()
    v = torch.randn(sum(need), kv_heads * hd * PAGE, generator=g, device=gpu).bfloat16()
    order = torch.randperm(sum(need), generator=g, device=gpu).int()
    table, at = torch.zeros(rows, per, dtype=torch.int32, device=gpu), 0
    for i, n in enumerate(need):
        table[i, :n] = order[at:at + n]
        at += n
    positions = torch.tensor([n - 1 for n in lens], dtype=torch.int32, device=gpu)
    q = torch.randn(rows, heads * hd, generator=g, device=gpu).bfloat16()

    def run(scratch):
        out = torch.zeros(rows, heads * hd, dtype=torch.bfloat16, device=gpu)
        ops.attention_bf16(q, positions, table, None, rows, k, v, out, heads, kv_heads, hd, PAGE, 0, hd ** -0.5, decode=True, scratch=scratch)
        return out

    floats, counters = ops.attention_decode_scratch(rows, heads, kv_heads, hd, per, PAGE)
    assert floats > 0
    scratch = (torch.full((floats,), float("nan"), device=gpu), torch.zeros(counters, dtype=torch.int32, device=gpu))
    whole, split, again = run(None), run(scratch), run(scratch)
    assert torch.equal(whole, split) and torch.equal(whole, again) and not scratch[1].any()
    for i, n in enumerate(lens):
        pages = table[i, :need[i]].long()
        keys = k[pages].view(-1, kv_heads, PAGE, hd).permute(1, 0, 2, 3).reshape(kv_heads, -1, hd)[:, :n].double()
        values = v[pages].view(-1, kv_heads, hd, PAGE).permute(1, 0, 3, 2).reshape(kv_heads, -1, hd)[:, :n].double()
        rep = heads // kv_heads
        p = torch.softmax((q[i].view(kv_heads, rep, hd).double() * hd ** -0.5) @ keys.transpose(1, 2).contiguous(), -1)
        want = (p @ values).reshape(-1)
        # (probabilities and the result are rounded to bfloat16, 2^-9 each)
        assert (whole[i].double() - want).norm() <= 2 ** -7 * want.norm()
