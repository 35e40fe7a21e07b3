"""The bf16 products that move both operands by LDS-DMA (gemm_dd.h): every tile
shape at its edges (test_cases_reach_every_tile_shape holds the cases to that),
reductions that end inside a stage, split reductions."""
import re

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
    (2044, 1272, 5128),                                            # forward in split 256 x 128
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


def test_cases_reach_every_tile_shape():
    from torch.profiler import ProfilerActivity, profile
    from concord_amd import packed_b as pb
    seen = {3: set(), 4: set()}   # kernel mode: forward, dgrad
    for M, N, K in CASES:
        x, dy, W = (torch.zeros(s, dtype=torch.bfloat16, device="cuda") for s in ((M, K), (M, N), (N, K)))
        with profile(activities=[ProfilerActivity.CUDA], acc_events=True) as prof:
            pb._gemm_fwd(x, None, None, None, 15, None, W)
            pb._gemm_dgrad(dy, None, None, None, 15, W)
            torch.cuda.synchronize()
        for e in prof.key_averages():
            m = re.search(r"gemm_dd_kernel<(\d+), (\d+), (\d+),", e.key)
            if m:
                seen[int(m[1])].add((int(m[2]), int(m[3])))
    dgrad = {(256, 256), (256, 128), (192, 128), (128, 128)}
    assert seen == {3: dgrad | {(256, 160)}, 4: dgrad}


@pytest.mark.parametrize("M,N,K", [(4096, 1280, 1280), (8192, 3072, 704)])
def test_decoding_layer_with_a_small_workspace(M, N, K):
    """Packed products whose workspace has no room for the decoded weight run
    on the packed words, with the same bits (neither is split)."""
    import concord_amd as ca
    from concord_amd import _lib as C, packed_b as pb
    torch.manual_seed(K)
    la = ca.ConcordLinearPackedB(K, N, bias=False, device="cuda")
    x, dy = (torch.randn(M, k, device="cuda").bfloat16() for k in (K, N))
    y, dx = torch.empty(M, N, device="cuda").bfloat16(), torch.empty(M, K, device="cuda").bfloat16()
    ws = torch.zeros(16384, dtype=torch.uint8, device="cuda")   # the tile counters alone
    w = (C.ptr(la.packed_w), la.packed_w.stride(0), C.ptr(la.row_exp), C.ptr(la.col_exp), 15)
    st = C.stream_of(x.device)
    C.check(C.lib().concord_dqgemm_fwd(C.ptr(x), K, *w, None, C.ptr(y), N, M, N, K, C.ptr(ws), ws.numel(), st), "fwd")
    C.check(C.lib().concord_dqgemm_dgrad(C.ptr(dy), N, *w, C.ptr(dx), K, M, N, K, C.ptr(ws), ws.numel(), st), "dgrad")
    args = (la.packed_w, la.row_exp, la.col_exp, 15)
    assert torch.equal(y, pb._gemm_fwd(x, *args, None, None))
    assert torch.equal(dx, pb._gemm_dgrad(dy, *args, None))


@pytest.mark.parametrize("M,N,K", [(4096, 1280, 1280), (4104, 1288, 1272), (2048, 1280, 5120), (4096, 640, 2560),
                                   (2056, 5128, 1288), (16384, 640, 640), (8200, 2568, 1272)])
def test_packed_products_on_a_decoded_copy(M, N, K):
    """Large packed products decode the weight first: the bits of the product
    on the materialised weight (power-of-two scales, same sums), in the
    separate and the combined backward entry."""
    import concord_amd as ca
    from concord_amd import packed_b as pb
    torch.manual_seed(N)
    la = ca.ConcordLinearPackedB(K, N, bias=True, device="cuda", lr=5e-4)
    x = torch.randn(M, K, device="cuda").bfloat16()
    dy = (torch.randn(M, N, device="cuda") * 1e-3).bfloat16()
    W = la.get_weight()
    la.bias.data.normal_()
    args = (la.packed_w, la.row_exp, la.col_exp, 15)
    y = pb._gemm_fwd(x, *args, la.bias, None)
    assert torch.equal(y, pb._gemm_fwd(x, None, None, None, 15, la.bias, W))
    dx = pb._gemm_dgrad(dy, *args, None)
    assert torch.equal(dx, pb._gemm_dgrad(dy, None, None, None, 15, W))
    gw = pb._wgrad(dy, x)
    dx2, gw2, gb2 = pb._dgrad_wgrad_vhat(dy, x, *args, la.v_row, la.v_col, la._sum_v_inv, 0.999, la._row_max_buf,
                                         la._col_max_buf, pb._get_step_counter("cuda"), True)
    assert torch.equal(dx, dx2) and torch.equal(gw, gw2)
    ref = dy.double().sum(0)
    assert torch.all((gb2.double() - ref).abs() <= ref.abs() * 2.0 ** -8 + dy.double().abs().sum(0) * M * 2.0 ** -24)
