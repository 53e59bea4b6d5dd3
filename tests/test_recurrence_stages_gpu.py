"""Matrix memories walked in stages against the walk, bit for bit: read-outs and states, portions around the edges of the chunks,
several requests in a step, slots that are skipped, shared keys, and layouts that the stages do not take."""

import pytest
import torch

from bitwise_amd.csrc import ops

pytestmark = pytest.mark.gpu

GIVEN, GATES = ops.RECUR_DECAY_GIVEN, ops.RECUR_SCALAR_GATES


def _both(gpu, mode, heads, dim, vdim, counts, heads_per_key=1, kscale=1.0, q_off=0, skip=None):
    g = torch.Generator(device=gpu).manual_seed(heads * dim + vdim + sum(counts))
    rows, nseq, keys = sum(counts), len(counts), heads // heads_per_key * dim
    k_off, v_off = q_off + keys, q_off + 2 * keys
    width = (v_off + heads * vdim + 2 * heads + 3) // 4 * 4
    proj = torch.randn(rows, width, generator=g, device=gpu)
    decays = torch.sigmoid(torch.randn(rows, heads * dim, generator=g, device=gpu)).pow(1 / 8)
    bias = torch.randn(2, heads, generator=g, device=gpu)
    state = torch.randn(nseq, ops.recurrence_state(mode if mode == GATES else GIVEN, heads, dim, vdim), generator=g, device=gpu)
    base, copy = heads * dim * vdim, heads * dim + heads
    state[:, :base:7] = -0.0
    if mode == GATES:                                                # every workgroup's copy of the normaliser and the maximum is alike
        state[:, base:] = state[:, base:base + copy].repeat(1, (state.shape[1] - base) // copy)
    bounds = [0]
    for n in counts:
        bounds.append(bounds[-1] + n)
    seq_rows = torch.tensor([x for a, n in zip(bounds, counts) for x in (a, n)], dtype=torch.int32, device=gpu)
    slots = torch.arange(nseq, dtype=torch.int32, device=gpu).flip(0).contiguous()
    if skip is not None:
        slots[skip] = -1
    positions = torch.arange(rows, dtype=torch.int32, device=gpu)
    results = []
    for stages in (False, True):
        out, s = torch.full((rows, heads * vdim), 7.0, device=gpu), state.clone()
        gate, goff, g2, b1, b2 = (decays, 0, 0, None, None) if mode == GIVEN else (proj, v_off + heads * vdim, v_off + heads * vdim + heads, bias[0], bias[1] + 3)
        gates = torch.full((rows, 3 * heads), float("nan"), device=gpu) if stages and mode == GATES else None
        ops.linear_recurrence(mode, proj, q_off, k_off, v_off, gate, goff, g2, b1, b2, 15.0, dim ** -0.5, s, out, seq_rows, slots, positions, nseq, heads,
                              dim, vdim, kscale=kscale, heads_per_key=heads_per_key, in_stages=stages, gates=gates)
        results.append((out.view(torch.int32), s.view(torch.int32)))
    (o0, s0), (o1, s1) = results
    assert torch.equal(o0, o1) and torch.equal(s0, s1)


@pytest.mark.parametrize("mode", [GIVEN, GATES])
@pytest.mark.parametrize("heads,dim,vdim", [(8, 64, 16), (3, 64, 72), (2, 128, 24), (8, 128, 8)])
@pytest.mark.parametrize("counts", [(1,), (13,), (14, 15, 16, 17), (29, 31, 32, 33), (63, 5), (64, 1, 80), (257,), (2049, 45)])
def test_stages_are_the_walk(gpu, mode, heads, dim, vdim, counts):
    _both(gpu, mode, heads, dim, vdim, counts)


@pytest.mark.parametrize("mode", [GIVEN, GATES])
def test_stages_with_shared_keys_scaled_keys_and_slots_to_skip(gpu, mode):
    _both(gpu, mode, 4, 64, 16, (40, 70), heads_per_key=2, kscale=0.37)
    _both(gpu, mode, 4, 128, 16, (40, 70, 33), heads_per_key=4, skip=1)


@pytest.mark.parametrize("mode", [GIVEN, GATES])
@pytest.mark.parametrize("heads,dim,vdim,q_off", [(2, 64, 12, 0), (2, 96, 16, 0), (2, 64, 16, 1), (2, 32, 16, 0), (2, 256, 16, 0)])
def test_layouts_that_the_stages_do_not_take(gpu, mode, heads, dim, vdim, q_off):
    _both(gpu, mode, heads, dim, vdim, (70, 9), q_off=q_off)
