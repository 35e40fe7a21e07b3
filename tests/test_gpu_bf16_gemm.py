"""The bf16 products that move both operands by LDS-DMA (gemm_dd.h): every tile
shape at its edges, reductions that end inside a stage, split reductions."""

import pytest
import torch

pytestmark = pytest.mark.gpu

# M, N, K: the forward reduces over K and tiles (M, N), the dgrad reduces over
# N and tiles (M, K)
CASES = [
    (1, 8, 8), (129, 136, 72), (128, 128, 64), (300, 264, 200),   # one tile and its remainders, partial stages
    (257, 1288, 520),                                              # split reductions, both directions
    (4100, 1288, 1272), (4096, 1280, 1280),                        # 192 x 128
    (2048, 5120, 1288), (2056, 1280, 5120),                        # 256 x 160 / 256 x 256 and split
    (8200, 2568, 648),                                             # several rounds of the largest tiles
]


@pytest.mark.parametrize("M,N,K", CASES)
def test_bf16_products(M, N, K):
    from concord_amd import packed_b as pb
    g = torch.Generator().manual_seed(M + N + K)
    x = torch.randn(M, K, generator=g).bfloat16().cuda()
    dy = torch.randn(M, N, generator=g).bfloat16().cuda()
    W = torch.randn(N, K, generator=g).bfloat16().cuda()
    bias = torch.randn(N, generator=g).bfloat16().cuda()
    y = pb._gemm_fwd(x, None, None, None, 15, bias, W)
    dx = pb._gemm_dgrad(dy, None, None, None, 15, W)
    for got, a, b, add in ((y, x, W.t(), bias), (dx, dy, W, None)):
        ref = a.double() @ b.double()
        mag = a.double().abs() @ b.double().abs()
        if add is not None:
            ref, mag = ref + add.double(), mag + add.double().abs()
        R = a.shape[1]
        # one rounding to bf16 (2^-8 of the value) and R fp32 additions
        bound = ref.abs() * 2.0 ** -8 + mag * R * 2.0 ** -24
        assert torch.all((got.double() - ref).abs() <= bound)
