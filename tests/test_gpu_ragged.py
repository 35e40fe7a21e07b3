"""Layers whose widths are no multiples of 8: the products run on zero-padded
copies in the workspace (ragged operands, csrc/gemm.hip)."""
import numpy as np
import pytest
import torch

from gpu_util import DEV, dev, host, rand_state, sync

pytestmark = pytest.mark.gpu

# (M, N, K): the edges of the 8-column chunks and of the rule that makes the
# copies (more than 64 terms, 512 rows, 4096 elements of work), one row or
# column, a vocabulary head, 4-channel patch rows, odd widths past a tile
SHAPES = [(1, 5, 3), (4, 32, 31), (4, 33, 31), (511, 65, 40), (511, 30, 64), (511, 30, 66), (512, 30, 64),
          (512, 65, 384), (64, 9, 1001), (300, 2050, 645), (513, 1, 36), (1030, 4, 2880), (700, 129, 7), (600, 8, 9), (777, 100, 770),
          (2050, 320, 36), (640, 257, 131), (520, 36, 1)]


def _bound(exact, terms, n):
    """One fp32 sum of n terms in any order (each addition rounds at most by
    2^-24 of the magnitudes' sum) rounded once to bf16."""
    return 2.0 ** -8 * np.abs(exact) + n * 2.0 ** -24 * terms + 1e-30


def _f64(t):
    return t.detach().double().cpu().numpy()


@pytest.mark.parametrize("M,N,K", SHAPES)
def test_ragged_products_match_float64(oracle, M, N, K):
    from concord_amd import packed_b as pb
    rng = np.random.default_rng(M + 3 * N + 7 * K)
    packed, re, ce = rand_state(rng, N, K, exp=(-2, 2), col=(-2, 2))
    pk, red, ced = dev(packed), dev(re), dev(ce)
    gen = torch.Generator().manual_seed(M)
    x = torch.randn(M, K, generator=gen).to(torch.bfloat16).to(DEV)
    dy = torch.randn(M, N, generator=gen).to(torch.bfloat16).to(DEV)
    b = torch.randn(N, generator=gen).to(torch.bfloat16).to(DEV)
    W = oracle.bf16_bits_to_f32(oracle.materialize(packed, re, ce)).astype(np.float64)
    Wb = torch.from_numpy(W).to(torch.bfloat16).to(DEV)
    xd, dyd, bd = _f64(x), _f64(dy), _f64(b)
    y_ref, y_terms = xd @ W.T + bd, np.abs(xd) @ np.abs(W).T + np.abs(bd)
    dx_ref, dx_terms = dyd @ W, np.abs(dyd) @ np.abs(W)
    gw_ref, gw_terms = dyd.T @ xd, np.abs(dyd).T @ np.abs(xd)
    for wbuf in (None, Wb):
        y = pb._gemm_fwd(x, pk, red, ced, 15, b, wbuf)
        dx = pb._gemm_dgrad(dy, pk, red, ced, 15, wbuf)
        assert (np.abs(_f64(y) - y_ref) <= _bound(y_ref, y_terms, K + 1)).all()
        assert (np.abs(_f64(dx) - dx_ref) <= _bound(dx_ref, dx_terms, N)).all()
    gw = pb._wgrad(dy, x)
    sync()
    assert (np.abs(_f64(gw) - gw_ref) <= _bound(gw_ref, gw_terms, M)).all()


@pytest.mark.parametrize("M,N,K", SHAPES)
def test_ragged_backward_entry_matches_separate_calls(oracle, M, N, K):
    """The combined entry, the v-hat entry and the plain product agree bit for
    bit on dx, grad_W and v-hat; the bias gradient matches the float64 sum."""
    from concord_amd import packed_b as pb
    rng = np.random.default_rng(M + N + K)
    packed, re, ce = rand_state(rng, N, K, exp=(-3, 3), col=(-1, 1))
    pk, red, ced = dev(packed), dev(re), dev(ce)
    gen = torch.Generator().manual_seed(K)
    x = torch.randn(M, K, generator=gen).to(torch.bfloat16).to(DEV)
    dy = (torch.randn(M, N, generator=gen) * 1e-2).to(torch.bfloat16).to(DEV)
    outs, gbs = [], []
    for combined in (True, False):
        vr, vc = torch.full((N,), 1e-4, device=DEV), torch.full((K,), 2e-4, device=DEV)
        svi = torch.ones(1, device=DEV)
        rm = torch.full((N,), 77, dtype=torch.int32, device=DEV)
        cm = torch.full((K,), 88, dtype=torch.int32, device=DEV)
        salt = torch.full((1,), 5, dtype=torch.int32, device=DEV)
        args = (vr, vc, svi, 0.999, rm, cm, salt)
        if combined:
            dx, gw, gb = pb._dgrad_wgrad_vhat(dy, x, pk, red, ced, 15, *args, with_bias=True)
        else:
            dx = pb._gemm_dgrad(dy, pk, red, ced, 15, None)
            gw, gb = pb._wgrad_vhat(dy, x, *args, with_bias=True)
        sync()
        outs.append([host(t) for t in (dx, gw, vr, vc, svi, rm, cm, salt)])
        gbs.append(_f64(gb))
    for a, b in zip(*outs):
        np.testing.assert_array_equal(a, b)
    np.testing.assert_array_equal(outs[0][1], host(pb._wgrad(dy, x)))
    vr, vc = np.full(N, 1e-4, np.float32), np.full(K, 2e-4, np.float32)
    oracle.vhat_ema(outs[0][1], vr, vc, 0.999)
    np.testing.assert_array_equal(outs[0][2], vr)
    np.testing.assert_array_equal(outs[0][3], vc)
    gb_ref, terms = _f64(dy).sum(0), np.abs(_f64(dy)).sum(0)
    for gb in gbs:
        assert (np.abs(gb - gb_ref) <= _bound(gb_ref, terms, M)).all()


@pytest.mark.parametrize("M,N,K", [(600, 65, 40), (900, 30, 33)])
def test_ragged_strided_and_small_workspace(oracle, M, N, K):
    """Operands with their own row strides and unaligned bases, and a
    workspace without room for the copies (the generic kernel), give the
    products of the plain call."""
    from concord_amd import _lib as C, packed_b as pb
    rng = np.random.default_rng(N)
    packed, re, ce = rand_state(rng, N, K, exp=(-2, 2), col=(-1, 1))
    pk, red, ced = dev(packed), dev(re), dev(ce)
    x = torch.randn(M, K, device=DEV).to(torch.bfloat16)
    base = pb._gemm_fwd(x, pk, red, ced, 15, None, None).double()
    xs = torch.zeros(M, K + 5, dtype=torch.bfloat16, device=DEV)
    xs[:, 1:K + 1] = x
    view = xs[:, 1:K + 1]
    need = int(C.lib().concord_gemm_workspace_bytes(M, N, K))
    for nbytes in (need, 16384):
        ws = torch.zeros(nbytes, dtype=torch.uint8, device=DEV)
        y = torch.full((M, N + 3), 7.0, dtype=torch.bfloat16, device=DEV)
        C.check(C.lib().concord_dqgemm_fwd(C.ptr(view), view.stride(0), C.ptr(pk), pk.stride(0), C.ptr(red), C.ptr(ced),
                                           15, None, C.ptr(y), y.stride(0), M, N, K, C.ptr(ws), nbytes,
                                           C.stream_of(torch.device(DEV))), "fwd")
        sync()
        assert (y[:, N:] == 7.0).all()
        err = (y[:, :N].double() - base).norm() / base.norm()
        assert err.item() < 2.0 ** -8


def test_ragged_forwards_on_two_streams():
    """Forwards of two ragged layers in flight on two streams, one of them
    replayed from a graph, give what each gives alone."""
    import concord_amd as ca
    torch.manual_seed(1)
    layers = [ca.ConcordLinearPackedB(k, n, bias=True, device=DEV) for n, k in ((320, 36), (257, 645))]
    xs = [torch.randn(m, k, device=DEV).to(torch.bfloat16) for m, k in ((32768, 36), (4096, 645))]
    with torch.no_grad():
        alone = [la(x).clone() for la, x in zip(layers, xs)]
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            captured = layers[0](xs[0])
        sync()
        streams = [torch.cuda.Stream() for _ in range(2)]
        for _ in range(20):
            with torch.cuda.stream(streams[0]):
                graph.replay()
                got = captured.clone()
            with torch.cuda.stream(streams[1]):
                ys = [layers[1](xs[1]) for _ in range(4)]
            sync()
            assert torch.equal(got, alone[0])
            for y in ys:
                assert torch.equal(y, alone[1])


@pytest.mark.parametrize("M,N,K", [(4096, 1280, 1280), (16384, 640, 640)])
def test_split_counters_of_an_uncleared_workspace(M, N, K):
    """A layer with a workspace of its own whose operands only the generic
    kernel takes (an odd base): its two-way split, from uncleared memory."""
    from concord_amd import _lib as C, packed_b as pb
    gen = torch.Generator().manual_seed(N)
    dy = torch.randn(M, N, generator=gen).to(torch.bfloat16).to(DEV)
    x = torch.empty(M * K + 1, dtype=torch.bfloat16, device=DEV)[1:].view(M, K)
    x.copy_(torch.randn(M, K, generator=gen))
    need = int(C.lib().concord_gemm_workspace_bytes(M, N, K))
    outs = []
    for fill in (0, 0xA5):
        ws = torch.full((need,), fill, dtype=torch.uint8, device=DEV)
        gw = torch.empty(N, K, dtype=torch.bfloat16, device=DEV)
        C.check(C.lib().concord_wgrad(C.ptr(dy), N, C.ptr(x), K, C.ptr(gw), K, M, N, K, C.ptr(ws), need,
                                      C.stream_of(torch.device(DEV))), "wgrad")
        outs.append(gw)
    sync()
    assert torch.equal(*outs)
    ref = dy.double().T @ x.double()
    assert ((outs[0].double() - ref).norm() / ref.norm()).item() < 2.0 ** -8


def test_ragged_operand_beyond_the_extents():
    """dy's padded copy would pass the 2^30 bytes that the fast kernels address:
    the dgrad and the weight gradient run on the operands as they are."""
    from concord_amd import packed_b as pb
    M, N, K = 1 << 20, 513, 9
    gen = torch.Generator(device=DEV).manual_seed(0)
    x = torch.randn(M, K, device=DEV, generator=gen).to(torch.bfloat16)
    dy = torch.randn(M, N, device=DEV, generator=gen).to(torch.bfloat16)
    W = torch.randn(N, K, device=DEV, generator=gen).to(torch.bfloat16)
    y = pb._gemm_fwd(x, None, None, None, 15, None, W)
    dx = pb._gemm_dgrad(dy, None, None, None, 15, W)
    gw = pb._wgrad(dy, x)
    sync()
    for at in (slice(0, 1000), slice(M - 1000, M)):
        for got, a, b in ((y[at], x[at], W.T), (dx[at], dy[at], W)):
            ref, terms = a.double() @ b.double(), a.double().abs() @ b.double().abs()
            assert ((got.double() - ref).abs() <= ref.abs() * 2.0 ** -8 + terms * a.shape[1] * 2.0 ** -24).all()
    ref = sum(dy[i:i + 65536].double().T @ x[i:i + 65536].double() for i in range(0, M, 65536))
    assert ((gw.double() - ref).norm() / ref.norm()).item() < 2.0 ** -8


@pytest.mark.parametrize("M,N,K,copies", [(512, 65, 384, 2), (600, 65, 37, 3), (640, 320, 36, 1)])
def test_backward_pads_each_operand_once(M, N, K, copies):
    """Copies a ragged backward launches: dy and x where their widths are no
    whole chunks, and the weight where the dgrad reads it padded."""
    from torch.profiler import ProfilerActivity, profile
    from concord_amd import packed_b as pb
    rng = np.random.default_rng(N)
    pk, red, ced = (dev(t) for t in rand_state(rng, N, K, exp=(-2, 2), col=(-1, 1)))
    x = torch.randn(M, K, device=DEV).to(torch.bfloat16)
    dy = torch.randn(M, N, device=DEV).to(torch.bfloat16)
    args = (torch.ones(N, device=DEV), torch.ones(K, device=DEV), torch.ones(1, device=DEV), 0.999, None, None,
            torch.ones(1, dtype=torch.int32, device=DEV))
    pb._dgrad_wgrad_vhat(dy, x, pk, red, ced, 15, *args, with_bias=True)
    sync()
    with profile(activities=[ProfilerActivity.CUDA], acc_events=True) as prof:
        pb._dgrad_wgrad_vhat(dy, x, pk, red, ced, 15, *args, with_bias=True)
        sync()
    assert sum(e.count for e in prof.key_averages() if "pad_rows_kernel" in e.key) == copies
