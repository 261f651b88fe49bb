"""Small- and mid-M tiles of the quantised GEMM (gemm_skq_kernel): every row equals the bf16 GEMM on the
dequantised weights bit for bit -- the same bf16 weights, the same MFMA sums over K -- at sizes on both
sides of each tile's limit, with partial tiles, and at K values that leave stages or tiles out."""

import pytest
import torch

from yapd_amd import kernels
from yapd_amd.quant import dequant_affine, qgemm_affine, quantize_affine

pytestmark = pytest.mark.gpu
BF = torch.bfloat16


def inputs(dev, M, N, K, bits):
    g = torch.Generator(device=dev).manual_seed(M + N + K + bits)
    w = torch.randn(N, K, generator=g, device=dev) * torch.logspace(-2, 0, K, device=dev)
    w += torch.randn(N, 1, generator=g, device=dev) * 0.1
    A = torch.randn(M, K, generator=g, device=dev).to(BF)
    return A, quantize_affine(w, bits)


@pytest.mark.parametrize("bits", [4, 8])
# N = 1024: 16 x 16 tiles up to M = 64, 32 x 16 to 128, 32 x 32 to 256, 64 x 32 to 512, 64 x 64 to 1024, 128 x 64 to
# 2048 (not at 8 bits and K = 4096, whose scales do not fit beside its ring), 128 x 128 to 4096.  K: one stage short
# of the deep tiles' rings (768, 192), odd numbers of k-tiles, scales past one batch (4096)
@pytest.mark.parametrize("N,K", [(1024, 1024), (1000, 4096), (1024, 2048), (72, 768), (1024, 192), (200, 1344), (3072, 512)])
def test_rows_equal_the_bf16_gemm_on_dequantised_weights(dev, bits, N, K):
    A, codes = inputs(dev, 4096, N, K, bits)
    W = dequant_affine(*codes, bits)
    ref = torch.empty(4096, N, dtype=BF, device=dev)
    kernels.gemm_bf16(A, W, ref)
    for M in (1, 15, 16, 17, 64, 65, 100, 113, 127, 128, 129, 256, 257, 511, 513, 1000, 1025, 1900, 2049, 3000, 4096):
        assert torch.equal(qgemm_affine(A[:M], *codes, bits), ref[:M]), M


@pytest.mark.parametrize("bits", [4, 8])
def test_strided_rows(dev, bits):
    """A and C with row pitches of their own; columns past N stay untouched."""
    A, codes = inputs(dev, 50, 200, 1024, bits)
    wide = torch.full((50, 1024 + 40), float("nan"), dtype=BF, device=dev)
    wide[:, :1024] = A
    out = torch.full((50, 256), 7.0, dtype=BF, device=dev)
    qgemm_affine(wide[:, :1024], *codes, bits, out=out[:, :200])
    assert torch.equal(out[:, :200], qgemm_affine(A, *codes, bits))
    assert (out[:, 200:] == 7.0).all()


@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("N,K", [(1024, 64), (1000, 128), (3072, 192), (200, 704), (1024, 832), (1024, 896), (1024, 1088),
                                 (1024, 1152), (136, 9216), (520, 16384)])
def test_k_outside_the_rings(dev, bits, N, K):
    """K too short for the ring, and too long for its scales: 128 x 128 tiles of gemm_dlq_kernel, of which one k-tile
    is the shortest.  Against fp64 on the dequantised weights, half a bf16 ulp and the error of K fp32 sums, and bit
    for bit between row counts."""
    A, codes = inputs(dev, 4000, N, K, bits)
    W = dequant_affine(*codes, bits).double()
    got = [qgemm_affine(A[:M], *codes, bits) for M in (4000, 1000, 129, 3)]
    for C in got[1:]:
        assert torch.equal(C, got[0][: len(C)]), len(C)
    A = A[:1000].double()
    ref, mag = A @ W.T, A.abs() @ W.abs().T
    assert ((got[1].double() - ref).abs() <= ref.abs() * 2.0 ** -8 + mag * K * 2.0 ** -24).all()
