"""The bfloat16 products of prompt portions, tile by tile: every epilogue in every tile that the rules choose, whole and split along
K, against the same rows given sixteen at a time (kernels for few rows) and against float64, with guard rows and columns around
the outputs.  Each case names the tile it is there for and asserts that the rule still gives it."""

import pytest
import torch

from bitwise_amd.csrc import ops

pytestmark = pytest.mark.gpu

# tile -> (M, columns, K): last tiles ragged in rows and columns, several segments of K where the tile joins them
STORED = {
    (64, 128): (257, 6100, 4160),
    (128, 64): (500, 2100, 2112),
    (128, 128): (600, 4090, 4160),
    (128, 256): (300, 16000, 4160),
    (160, 256): (700, 12000, 2112),
    (192, 256): (513, 16000, 4096),
    (256, 192): (2040, 6136, 2112),
    (256, 256): (1500, 8200, 192),
}
# tile -> (M, columns of the output, K); columns in whole 16-byte pieces and not
GATED = {
    (64, 128): [(77, 68, 2560), (88, 104, 64)],
    (128, 64): [(147, 75, 2112), (500, 1056, 2112)],
    (128, 128): [(65, 8317, 2112), (65, 8424, 64)],
    (128, 256): [(257, 5643, 64), (132, 8224, 2112)],
    (160, 256): [(389, 8288, 2112), (385, 8439, 64)],
    (192, 256): [(515, 6549, 2112), (485, 8224, 64)],
    (256, 256): [(581, 8271, 64), (1345, 4104, 192)],
}
# tile -> (M, columns, K): a workgroup per tile and segment of K, the last segment shorter
SPLIT = {
    (128, 128): [(86, 224, 3200), (321, 2052, 8256)],
    (128, 256): [(66, 8260, 6336), (130, 6148, 8256)],
    (128, 64): [(292, 80, 3968)],
    (160, 256): [(1814, 516, 10304)],
    (192, 256): [(1301, 524, 14400), (700, 3004, 8256)],
    (256, 192): [(194, 5512, 10304)],
    (256, 256): [(386, 4140, 10304)],
}
GUARD = 77.0


def operands(gpu, M, N, K, apart=16):
    g = torch.Generator(device=gpu).manual_seed(M + N + K)
    x = torch.randn(M, K + apart, generator=g, device=gpu).bfloat16()[:, :K]      # rows farther apart than they are long
    return x, (torch.randn(N, K, generator=g, device=gpu) * K ** -0.5).bfloat16(), g


def by_sixteen(x, w, out, epilogue):
    for r in range(0, out.shape[0], 16):
        n = min(16, out.shape[0] - r)
        ops.gemm_bf16(x[r:r + n], w, out[r:r + n], n, epilogue)
    return out


def store(entry, x, w, M, N, dtype, pad, *more):
    """The C entry itself into the corner of a guarded buffer: an output whose rows are ``pad`` longer than N, two rows more."""
    buf = torch.full((M + 2, N + pad), GUARD, device=x.device, dtype=dtype)
    rc = ops._fn(entry)(x.data_ptr(), w.data_ptr(), buf.data_ptr(), M, N, x.shape[1], x.stride(0), N + pad, *more, ops._stream())
    assert rc == 0
    assert (buf[M:] == GUARD).all() and (buf[:, N:] == GUARD).all(), "a store past the output"
    return buf[:M, :N]


@pytest.mark.parametrize("tile", list(STORED))
def test_stores_and_adds_row_by_row(gpu, tile):
    M, N, K = STORED[tile]
    assert ops.gemm_prompt_tile(M, N, K) == tile and ops.gemm_prompt_parts(M, N, K) == 0
    x, w, g = operands(gpu, M, N, K)
    want = by_sixteen(x, w, torch.zeros(M, N, device=gpu), ops.EPI_F32)
    got = store("bw_gemm_bf16", x, w, M, N, torch.float32, 4, ops.EPI_F32)
    assert torch.equal(got, want)
    ref = x.double() @ w.double().T
    assert (got.double() - ref).abs().max() <= 2e-6 * K ** 0.5 * ref.abs().max()      # (32-bit sums of exact products)
    del ref
    rounded = store("bw_gemm_bf16", x, w, M, N, torch.bfloat16, 3, ops.EPI_BF16)
    assert torch.equal(rounded, want.bfloat16())
    base = torch.randn(M, N, generator=g, device=gpu)
    added = torch.full((M + 2, N + 4), GUARD, device=gpu)
    added[:M, :N] = base
    rc = ops._fn("bw_gemm_bf16")(x.data_ptr(), w.data_ptr(), added.data_ptr(), M, N, K, x.stride(0), N + 4, ops.EPI_ADD_F32, ops._stream())
    assert rc == 0 and (added[M:] == GUARD).all() and (added[:, N:] == GUARD).all()
    assert torch.equal(added[:M, :N], by_sixteen(x, w, base, ops.EPI_ADD_F32))


@pytest.mark.parametrize("tile", list(STORED))
def test_exact_gelu_of_every_tile(gpu, tile):
    M, N, K = STORED[tile]
    assert ops.gemm_prompt_tile(M, N, K, erf=True) == tile and ops.gemm_prompt_parts(M, N, K, erf=True) == 0
    x, w, _ = operands(gpu, M, N, K)
    sums = by_sixteen(x, w, torch.zeros(M, N, device=gpu), ops.EPI_F32)
    want = torch.zeros(M, N, device=gpu, dtype=torch.bfloat16)
    ops.activate(sums, want, M, ops.PLAIN_GELU_ERF)
    assert torch.equal(store("bw_gemm_bf16", x, w, M, N, torch.bfloat16, 5, ops.EPI_GELU_BF16), want)


@pytest.mark.parametrize("tile,M,N,K", [(t, *s) for t, shapes in GATED.items() for s in shapes])
def test_gated_epilogues_of_every_tile(gpu, tile, M, N, K):
    """SwiGLU, the clamped unit and the gated GELU: stores of 16 bytes (rows of whole pieces) and element by element."""
    assert ops.gemm_prompt_tile(M, 2 * N, K, gated=True) == tile and ops.gemm_prompt_parts(M, 2 * N, K, gated=True) == 0
    x, w, _ = operands(gpu, M, 2 * N, K)
    w = w * 3.0                                                     # (sums large enough for the clamps to bite)
    sums = by_sixteen(x, w, torch.zeros(M, 2 * N, device=gpu), ops.EPI_F32)
    limit, alpha = 1.5, 1.702
    pads = (8, 3) if N % 8 == 0 else (3,)
    for act, entry, more in ((ops.ACT_SILU, "bw_gemm_bf16", (ops.EPI_SWIGLU_BF16,)), (ops.ACT_CLAMPED_SWISH, "bw_gemm_clamped_glu_bf16", (limit, alpha)),
                             (ops.ACT_GELU_TANH, "bw_gemm_gelu_glu_bf16", ())):
        want = torch.zeros(M, N, device=gpu, dtype=torch.bfloat16)
        if act == ops.ACT_SILU:
            by_sixteen(x, w, want, ops.EPI_SWIGLU_BF16)
        else:
            ops.glu(sums, want, M, act, **({"limit": limit, "alpha": alpha} if act == ops.ACT_CLAMPED_SWISH else {}))
        for pad in pads:
            got = store(entry, x, w, M, N, torch.bfloat16, pad, *more)
            assert torch.equal(got.contiguous().view(torch.int16), want.view(torch.int16)), (act, pad)


def test_gated_epilogues_pass_on_infinities_and_nan(gpu):
    """Sums that are infinite or no number, and gates of every size, through the epilogues themselves."""
    M, N, K = 581, 8264, 64
    assert ops.gemm_prompt_tile(M, 2 * N, K, gated=True) == (256, 256) and ops.gemm_prompt_parts(M, 2 * N, K, gated=True) == 0
    x, w, _ = operands(gpu, M, 2 * N, K, apart=0)
    x, w = x.contiguous(), w.contiguous()
    x[3], x[40], x[300, 5], x[301, 6], x[580] = float("inf"), float("nan"), 3e38, -3e38, 1e20
    x[4] = 0.0
    x[4, 5] = float("inf")                                          # (one infinite product a sum: infinite sums of both signs)
    x[7] *= 1e-30
    sums = by_sixteen(x, w, torch.zeros(M, 2 * N, device=gpu), ops.EPI_F32)
    assert sums.isnan().any() and sums.isinf().any()
    for act, entry, more in ((ops.ACT_CLAMPED_SWISH, "bw_gemm_clamped_glu_bf16", (7.0, 1.702)), (ops.ACT_GELU_TANH, "bw_gemm_gelu_glu_bf16", ())):
        want = torch.zeros(M, N, device=gpu, dtype=torch.bfloat16)
        ops.glu(sums, want, M, act, **({"limit": 7.0, "alpha": 1.702} if more else {}))
        got = store(entry, x, w, M, N, torch.bfloat16, 8, *more)
        assert torch.equal(got.isnan(), want.isnan()) and want.isnan().any()
        assert torch.equal(got.nan_to_num(nan=9.0), want.nan_to_num(nan=9.0))


@pytest.mark.parametrize("M,N,K", [(256, 4096, 2048), (257, 4096, 2048), (192, 8192, 2048), (193, 8190, 2048), (512, 4096, 512), (513, 4096, 512),
                                   (448, 4100, 1024), (320, 4096, 4160), (321, 4090, 4160), (65, 16384, 64)])
def test_stores_on_both_sides_of_the_limits_of_blocks(gpu, M, N, K):
    """64-row blocks in one launch up to so many workgroups (of 64 columns; the limit goes by K and the epilogue), tiles beyond."""
    x, w, _ = operands(gpu, M, N, K)
    sums = by_sixteen(x, w, torch.zeros(M, N, device=gpu), ops.EPI_F32)
    assert torch.equal(store("bw_gemm_bf16", x, w, M, N, torch.float32, 4, ops.EPI_F32), sums)
    assert torch.equal(store("bw_gemm_bf16", x, w, M, N, torch.bfloat16, 3, ops.EPI_BF16), sums.bfloat16())
    want = torch.zeros(M, N, device=gpu, dtype=torch.bfloat16)
    ops.activate(sums, want, M, ops.PLAIN_GELU_ERF)
    assert torch.equal(store("bw_gemm_bf16", x, w, M, N, torch.bfloat16, 3, ops.EPI_GELU_BF16), want)


@pytest.mark.parametrize("add", (True, False))
@pytest.mark.parametrize("tile,M,N,K", [(t, *s) for t, shapes in SPLIT.items() for s in shapes])
def test_sums_of_a_split_in_every_tile(gpu, tile, M, N, K, add):
    """A workgroup per tile and segment, the sums in scratch (full of NaN, larger than needed), joined in order: the bits of the
    rows given sixteen at a time, twice on the same scratch; nothing behind the scratch is written."""
    assert ops.gemm_split_tile(M, N, K, store=not add) == tile
    floats, counters = ops.gemm_add_scratch(M, N, K)
    assert (floats, counters) == ((K + 2047) // 2048 * M * N, 1)
    x, w, g = operands(gpu, M, N, K)
    base = torch.randn(M, N, generator=g, device=gpu)
    epilogue = ops.EPI_ADD_F32 if add else ops.EPI_F32
    want = by_sixteen(x, w, base.clone() if add else torch.zeros(M, N, device=gpu), epilogue)
    scratch = (torch.full((floats + 1000,), float("nan"), device=gpu), torch.zeros(counters, dtype=torch.int32, device=gpu))
    scratch[0][floats:] = GUARD
    for _ in range(2):
        got = base.clone()
        ops.gemm_bf16(x, w, got, M, epilogue, scratch=scratch)
        assert torch.equal(got, want) and not scratch[1].any()
        assert not scratch[0][:floats].isnan().any() and (scratch[0][floats:] == GUARD).all()


@pytest.mark.parametrize("M,N,K", [(2048, 2048, 8192), (513, 8192, 4096)])
def test_products_that_go_whole_leave_the_scratch_alone(gpu, M, N, K):
    assert ops.gemm_split_tile(M, N, K) is None
    floats, counters = ops.gemm_add_scratch(M, N, K)
    x, w, g = operands(gpu, M, N, K)
    scratch = (torch.full((floats,), float("nan"), device=gpu), torch.zeros(counters, dtype=torch.int32, device=gpu))
    got = torch.randn(M, N, generator=g, device=gpu)
    want = got.clone()
    ops.gemm_bf16(x, w, got, M, ops.EPI_ADD_F32, scratch=scratch)
    ops.gemm_bf16(x, w, want, M, ops.EPI_ADD_F32)
    assert torch.equal(got, want) and scratch[0].isnan().all()
