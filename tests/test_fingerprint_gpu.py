"""Logits fingerprints at the edges of the kernel that chains a row bit by bit: rows that fill its passes to the last word but one,
exactly, and one beyond, odd lengths, rows that start on any element, words of every kind; and the number of rows on either side
of the rule."""

import numpy as np
import plain_llama as pl
import pytest
import torch

from bitwise_amd.csrc import ops

pytestmark = pytest.mark.gpu
BASES = [1469598103934665603, 0, 2 ** 64 - 1]


def device_prints(rows, bases):
    h_in = torch.from_numpy(np.asarray(bases, np.uint64).view(np.int64)).to(rows.device)
    h_out = torch.zeros_like(h_in)
    ops.fingerprint(rows, len(bases), h_in, h_out)
    return h_out.cpu().numpy().view(np.uint64).tolist()


@pytest.mark.parametrize("vocab", [4096, 4097, 16380, 16382, 16383, 16384, 16386, 32763, 32766, 32767, 32768, 65532, 65534, 65535, 65536,
                                   131068, 131071])
def test_rows_around_a_pass(gpu, vocab):
    g = torch.Generator().manual_seed(vocab)
    rows = torch.randn(3 * vocab + 1, generator=g)[1:].view(3, vocab)     # (a float past an even address)
    rows[1] = torch.from_numpy(np.random.default_rng(vocab).integers(0, 2 ** 32, vocab, dtype=np.uint32).view(np.float32))
    rows[2] = 0.0
    there = torch.empty(3 * vocab + 1, device=gpu)[1:].view(3, vocab)
    there.view(torch.int32).copy_(rows.view(torch.int32))
    assert device_prints(there, BASES) == [pl.hash_floats(b, rows[i].numpy()) for i, b in enumerate(BASES)]


@pytest.mark.parametrize("count,vocab", [(256, 5000), (257, 5000), (700, 9001), (2500, 4100)])
def test_many_rows(gpu, count, vocab):
    g = torch.Generator().manual_seed(count)
    few = torch.randn(5, vocab, generator=g)
    which = torch.arange(count) % 5
    want = [pl.hash_floats(BASES[0], few[i].numpy()) for i in range(5)]
    assert device_prints(few[which].contiguous().to(gpu), [BASES[0]] * count) == [want[i] for i in which.tolist()]
