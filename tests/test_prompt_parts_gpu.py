"""Prompt products whose columns go in two launches of differently shaped tiles: the bits of the same rows given sixteen at a time, on
both sides of the boundary and at the ragged ends, whatever the epilogue."""

import pytest
import torch

from bitwise_amd.csrc import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,N,K,gated", [
    (514, 22414, 512, False), (568, 22484, 512, False), (654, 22136, 512, False), (641, 22343, 512, False),
    (1360, 16490, 1024, False), (961, 19014, 1024, False), (580, 16500, 2112, False), (785, 14194, 2112, False),
    (911, 16396, 2048, False), (586, 19048, 4160, False), (1286, 12304, 4160, False),
    (518, 10962, 512, True), (535, 11246, 512, True), (642, 11141, 512, True), (650, 11361, 512, True),
    (395, 11323, 2112, True), (390, 11495, 2112, True), (1287, 5927, 2048, True), (769, 7709, 4160, True), (777, 14336, 4096, True),
])
def test_both_launches_keep_the_bits(gpu, M, N, K, gated):
    first = ops.gemm_prompt_parts(M, 2 * N if gated else N, K, gated)
    assert 0 < first < (2 * N if gated else N)
    g = torch.Generator(device=gpu).manual_seed(M + N + K)
    x = torch.randn(M, K + 16, generator=g, device=gpu).bfloat16()[:, :K]
    w = (torch.randn(2 * N if gated else N, K, generator=g, device=gpu) * K ** -0.5).bfloat16()
    kinds = ((ops.EPI_SWIGLU_BF16, torch.bfloat16),) if gated else ((ops.EPI_F32, torch.float32), (ops.EPI_BF16, torch.bfloat16),
                                                                    (ops.EPI_ADD_F32, torch.float32))
    for epi, dtype in kinds:
        base = torch.full((M + 1, N), 7.0, device=gpu, dtype=dtype)
        got = base.clone()
        ops.gemm_bf16(x, w, got, M, epi)
        assert bool((got[M] == 7.0).all())
        for r in sorted({0, 112, 240, M // 32 * 16, (M - 1) // 16 * 16}):
            n = min(16, M - r)
            want = base[r:r + n].clone()
            ops.gemm_bf16(x[r:r + n], w, want, n, epi)
            assert torch.equal(got[r:r + n], want), (epi, r)


@pytest.mark.parametrize("M,N,K", [(514, 22414, 512), (641, 22343, 512), (961, 19014, 1024), (911, 16396, 2048)])
def test_exact_gelu_of_both_launches(gpu, M, N, K):
    assert 0 < ops.gemm_prompt_parts(M, N, K, erf=True) < N
    g = torch.Generator(device=gpu).manual_seed(M + N + K)
    x = torch.randn(M, K + 16, generator=g, device=gpu).bfloat16()[:, :K]
    w = (torch.randn(N, K, generator=g, device=gpu) * K ** -0.5).bfloat16()
    got, sums = torch.zeros(M, N, device=gpu, dtype=torch.bfloat16), torch.zeros(M, N, device=gpu)
    ops.gemm_bf16(x, w, got, M, ops.EPI_GELU_BF16)
    for r in range(0, M, 16):
        n = min(16, M - r)
        ops.gemm_bf16(x[r:r + n], w, sums[r:r + n], n, ops.EPI_F32)
    want = torch.zeros_like(got)
    ops.activate(sums, want, M, ops.PLAIN_GELU_ERF)
    assert torch.equal(got, want)


@pytest.mark.parametrize("M,N,K", [(518, 10962, 512), (642, 11141, 512), (395, 11323, 2112), (1287, 5927, 2048), (777, 14336, 4096)])
def test_other_gated_epilogues_of_both_launches(gpu, M, N, K):
    assert 0 < ops.gemm_prompt_parts(M, 2 * N, K, gated=True) < 2 * N
    g = torch.Generator(device=gpu).manual_seed(M + N + K)
    x = torch.randn(M, K + 16, generator=g, device=gpu).bfloat16()[:, :K]
    w = (torch.randn(2 * N, K, generator=g, device=gpu) * 3 * K ** -0.5).bfloat16()
    sums = torch.zeros(M, 2 * N, device=gpu)
    for r in range(0, M, 16):
        n = min(16, M - r)
        ops.gemm_bf16(x[r:r + n], w, sums[r:r + n], n, ops.EPI_F32)
    for act, entry, more in ((ops.ACT_CLAMPED_SWISH, "bw_gemm_clamped_glu_bf16", (1.5, 1.702)), (ops.ACT_GELU_TANH, "bw_gemm_gelu_glu_bf16", ())):
        want, got = torch.zeros(M, N, device=gpu, dtype=torch.bfloat16), torch.full((M + 1, N), 7.0, device=gpu, dtype=torch.bfloat16)
        ops.glu(sums, want, M, act, **({"limit": 1.5, "alpha": 1.702} if more else {}))
        assert ops._fn(entry)(x.data_ptr(), w.data_ptr(), got.data_ptr(), M, N, K, x.stride(0), N, *more, ops._stream()) == 0
        assert torch.equal(got[:M], want) and bool((got[M] == 7.0).all()), act
