"""CPU-side checks of the product: the C-ABI library loads and exports every
declared symbol, host-side argument validation rejects bad calls before any
GPU work, flag numbering agrees across header / binding / oracle, and the
drop-in module refuses CPU devices instead of falling back."""
import os
import re

import pytest
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HEADER = os.path.join(ROOT, "include", "concord_amd.h")
DIAG_HEADER = os.path.join(ROOT, "include", "concord_amd_diag.h")


def _declared(headers=(HEADER, DIAG_HEADER)):
    names = set()
    for h in headers:
        src = re.sub(r"/\*.*?\*/", "", open(h).read(), flags=re.S)
        names |= set(re.findall(r"\b(concord_[a-z0-9_]+)\s*\(", src))
    return sorted(names)


def _header_flags():
    src = open(HEADER).read()
    return {m.group(1): int(m.group(2)) for m in
            re.finditer(r"#define CONCORD_([A-Z0-9_]+) \(1u << (\d+)\)", src)}


@pytest.fixture(scope="module")
def L():
    from concord_amd import _lib as C
    return C.lib()


def test_library_exports_every_declared_symbol(L):
    from concord_amd import _lib as C
    decl = _declared()
    assert len(decl) >= 16
    for name in decl:
        assert hasattr(L, name), f"{name} declared in include/ but not exported"
    assert sorted(C.exported_symbols()) == decl


def test_flag_numbering_consistent(oracle):
    from concord_amd import _lib as C
    hf = _header_flags()
    for name, bit in hf.items():
        assert getattr(C, name) == 1 << bit, name
        if hasattr(oracle, name):
            assert getattr(oracle, name) == 1 << bit, name


def test_version_and_workspace(L):
    assert L.concord_version() == 1
    a = L.concord_workspace_bytes(5120, 1280, 0)
    # v-hat partials dominate: (K/64) N + (N/128) K floats + 256 B of counters
    assert a >= 256 + (20 * 5120 + 40 * 1280) * 4
    assert a % 256 == 0
    assert L.concord_workspace_bytes(0, 0, 0) >= 256


def test_invalid_arguments_rejected_without_launch(L):
    from concord_amd import _lib as C
    P = None
    rc = L.concord_materialize(P, 10, P, P, -1, 10, 15, 0, P, 10, P)
    assert rc == C.EINVAL
    assert b"bad size" in L.concord_last_error()
    rc = L.concord_materialize(P, 10, P, P, 4, 10, 15, 0, P, 10, P)
    assert rc == C.EINVAL and b"NULL" in L.concord_last_error()
    rc = L.concord_dqgemm_fwd(P, 3, P, 3, P, P, 15, P, P, 3, 4, 4, 8, P, 0, P)
    assert rc == C.EINVAL
    rc = L.concord_vhat_ema(P, 8, 4, 8, 0.999, P, P, P, P, P, P, P, 0, P)
    assert rc == C.EINVAL
    ws = (ctypes_buf := __import__("ctypes").create_string_buffer(16))
    rc = L.concord_rebalance(ws, 8, ws, ws, ws, ws, P, P, ws, 4, 8, 24000, 7, -8, 0, 1, ws, 16, P)
    assert rc == C.EWORKSPACE
    assert b"workspace" in L.concord_last_error()
    # empty problems are valid no-ops
    assert L.concord_materialize(P, 0, P, P, 0, 0, 15, 0, P, 0, P) == C.OK
    assert L.concord_wgrad(P, 0, P, 0, P, 0, 5, 0, 7, P, 0, P) == C.OK
    # tile counters always; split-K partials only for products with few tiles
    ws = L.concord_gemm_workspace_bytes(2048, 5120, 1280)
    assert ws >= 16384 and ws % 256 == 0
    assert L.concord_gemm_workspace_bytes(128, 128, 1 << 16) >= 16384 + 2 * 128 * 128 * 4


def test_apply_rejects_missing_vhat_inputs(L):
    from concord_amd import _lib as C
    p = C.UpdateParams(alpha=0.1, gf_trust_delta_sq=1.0, mantissa_bias=15)
    import ctypes
    buf = ctypes.create_string_buffer(64)
    s = C.DeviceScalars(ctypes.addressof(buf), ctypes.addressof(buf), None, None, None,
                        ctypes.addressof(buf), None)
    rc = L.concord_apply_adamw(buf, 8, buf, 8, None, 8, buf, buf, buf, buf, None, None, None,
                               None, 8, 2, 8, ctypes.byref(p), ctypes.byref(s),
                               C.GF_TRUST_REGION, None)
    assert rc == C.EINVAL and b"v_row" in L.concord_last_error()


def test_module_refuses_cpu_device():
    import concord_amd as ca
    with pytest.raises(RuntimeError, match="ROCm GPU"):
        ca.ConcordLinearPackedB(8, 4, device="cpu")


def test_wrappers_refuse_cpu_tensors():
    from concord_amd import packed_b as pb
    p = torch.zeros(4, 8, dtype=torch.int32)
    with pytest.raises(RuntimeError, match="ROCm device"):
        pb.materialize_packed_bf16(p, torch.zeros(4, dtype=torch.int8), torch.zeros(8, dtype=torch.int8),
                                   torch.empty(4, 8, dtype=torch.bfloat16))


@pytest.mark.parametrize("device", ["cpu", "meta"])
def test_products_refuse_tensors_of_other_devices(device):
    """No host address may reach a launch: the stream lookup of every product
    refuses the device, as torch.cuda.current_stream does."""
    from concord_amd import _lib as C, packed_b as pb
    x, dy = (torch.empty(16, k, dtype=torch.bfloat16, device=device) for k in (24, 8))
    W = torch.empty(8, 24, dtype=torch.bfloat16, device=device)
    packed = (torch.empty(8, 24, dtype=torch.int32, device=device), torch.empty(8, dtype=torch.int8, device=device),
              torch.empty(24, dtype=torch.int8, device=device), 15)
    for call in (lambda: C.stream_of(torch.device(device)), lambda: C.stream_of(device),
                 lambda: pb._gemm_fwd(x, *packed, None, None), lambda: pb._gemm_dgrad(dy, *packed, W),
                 lambda: pb._wgrad(dy, x), lambda: pb._bias_grad(dy)):
        with pytest.raises(ValueError, match="Expected a cuda device"):
            call()


def test_public_api_surface():
    """Names a user of concord/__init__.py:7-31 imports exist with the same meaning."""
    import concord_amd as ca
    for name in ["ConcordLinearPackedB", "compute_drift_cancel_C", "set_fixed_coh", "set_gate_gain",
                 "reset_reb_stats", "get_reb_stats", "S_SLOW_FACTOR", "V_SLOW_FACTOR",
                 "MANTISSA_BIAS"]:
        assert hasattr(ca, name), name
    assert ca.S_SLOW_FACTOR == ca.V_SLOW_FACTOR == 128 and ca.MANTISSA_BIAS == 15
    assert abs(ca.compute_drift_cancel_C(0.1, 0.001) - 0.018036072144288578) < 1e-15
    assert abs(ca.compute_drift_cancel_C(0.1, 0.001, mass_preserve=False) - 0.009081735620585268) < 1e-15
    ca.reset_reb_stats()
    assert ca.get_reb_stats()["calls"] == 0
    with pytest.raises(NotImplementedError):
        ca.set_coh_weighted_v(True)
    assert abs(ca.bias_correction_factor(0) - 1000.0) < 1e-6


def test_default_knobs_match_reference():
    """concord/test_baked_defaults.py:17-27 / concord/packed_b.py:1394-1443, read
    from the constructor's source defaults without touching a device."""
    import inspect

    import concord_amd.packed_b as pb
    src = inspect.getsource(pb.ConcordLinearPackedB.__init__)
    for frag in ["self.optimizer_kind = 'adamw'", "self._eps_value = 1e-10", "self.v_scale = 0.0",
                 "self.precond_p = 0.5", "self.gf_trust_delta_sq = 1.0", "self.step_cap = 10.0",
                 "self.alpha_v_fast = 0.001", "self.mass_preserve_v = True",
                 "self.track_rebalance = True", "self.adafactor_beta2 = 0.999",
                 "self._coh_pre = torch.ones_like"]:
        assert frag in src, frag
    assert pb._USE_FIXED_COH is True and pb._RATIO_COH is False


def _rg_records(sizes):
    import ctypes

    from concord_amd import _lib as C
    rec = (ctypes.c_int64 * (len(sizes) * C.RG_FIELDS))()
    for i, (N, K) in enumerate(sizes):
        r = i * C.RG_FIELDS
        for f in (C.RG_PACKED, C.RG_ROW_EXP, C.RG_COL_EXP, C.RG_ROW_MAX, C.RG_COL_MAX, C.RG_SEED):
            rec[r + f] = 0x10000 * (i + 1) + 16 * f
        rec[r + C.RG_LD] = K
        rec[r + C.RG_N] = N
        rec[r + C.RG_K] = K
        rec[r + C.RG_MAX_M] = 24000
        rec[r + C.RG_EXP_MAX] = 7
        rec[r + C.RG_EXP_MIN] = -8
    return rec


def test_rebalance_group_plan_layout(L):
    """The group plan (host only): records copied, per-layer scratch offsets
    (row ticks N + column ticks K + one flag per 256-row / 256-column decide
    block), prefix sums of decide blocks and of 16 x 256 shift tiles."""
    import ctypes

    from concord_amd import _lib as C
    sizes = [(300, 520), (1, 1), (1280, 5120), (257, 256)]
    n = len(sizes)
    rec = _rg_records(sizes)
    plen = n * C.RG_FIELDS + 2 * (n + 1)
    plan = (ctypes.c_int64 * plen)()
    words = ctypes.c_int64(-1)
    assert L.concord_rebalance_group_plan(rec, n, plan, plen, ctypes.byref(words)) == C.OK
    cd = lambda a, b: -(-a // b)  # noqa: E731
    scr, dp, tp = 0, [0], [0]
    for i, (N, K) in enumerate(sizes):
        r = i * C.RG_FIELDS
        for f in range(14):
            assert plan[r + f] == rec[r + f], (i, f)
        assert plan[r + 14] == scr
        nd = cd(N, 256) + cd(K, 256)
        scr += N + K + nd
        dp.append(dp[-1] + nd)
        tp.append(tp[-1] + cd(N, 16) * cd(K, 256))
    assert words.value == scr == 7254 + 257 + 256 + 3
    assert list(plan[n * C.RG_FIELDS:n * C.RG_FIELDS + n + 1]) == dp == [0, 5, 7, 32, 35]
    assert list(plan[n * C.RG_FIELDS + n + 1:]) == tp == [0, 57, 58, 1658, 1658 + 17]


def test_rebalance_group_rejects_bad_plans(L):
    import ctypes

    from concord_amd import _lib as C
    n = 2
    plen = n * C.RG_FIELDS + 2 * (n + 1)
    plan = (ctypes.c_int64 * plen)()
    words = ctypes.c_int64(0)
    rec = _rg_records([(10, 20), (0, 5)])
    assert L.concord_rebalance_group_plan(rec, n, plan, plen, ctypes.byref(words)) == C.EINVAL
    assert b"layer 1: bad size" in L.concord_last_error()
    rec = _rg_records([(10, 20), (4, 5)])
    rec[C.RG_FIELDS + C.RG_LD] = 4
    assert L.concord_rebalance_group_plan(rec, n, plan, plen, ctypes.byref(words)) == C.EINVAL
    assert b"leading dimension" in L.concord_last_error()
    rec = _rg_records([(10, 20), (4, 5)])
    rec[C.RG_SEED] = 0
    assert L.concord_rebalance_group_plan(rec, n, plan, plen, ctypes.byref(words)) == C.EINVAL
    assert b"layer 0: NULL" in L.concord_last_error()
    rec = _rg_records([(10, 20), (4, 5)])
    assert L.concord_rebalance_group_plan(rec, n, plan, plen - 1, ctypes.byref(words)) == C.EINVAL
    assert L.concord_rebalance_group_plan(rec, 0, plan, plen, ctypes.byref(words)) == C.EINVAL
    # the launch entry point checks its workspace before any GPU work
    ws = ctypes.create_string_buffer(16)
    assert L.concord_rebalance_group(plan, n, ws, 24000, None, ws, 16, 100, None) == C.EWORKSPACE
    assert L.concord_rebalance_group(plan, n, None, 24000, None, ws, 16, 4, None) == C.EINVAL


def test_calls_that_write_operands_get_a_workspace_of_their_own(L):
    """Padded copies of a ragged layer's operands and decoded weights go into the
    workspace: two such calls in flight (two streams, a graph beside eager
    calls) must not hold the same buffer."""
    from concord_amd import packed_b as pb
    for M, N, K in [(2048, 320, 36), (512, 65, 384), (4096, 1280, 1280)]:
        a, b = (pb._gemm_workspace("cpu", M, N, K, True) for _ in range(2))
        assert a.numel() == b.numel() >= L.concord_gemm_workspace_bytes(M, N, K)
        assert a.data_ptr() != b.data_ptr(), (M, N, K)
    # a cached bf16 weight and the weight gradient alone decode nothing: no room
    # for a decoded weight, and the device's buffer
    cached = pb._gemm_workspace("cpu", 4096, 1280, 1280, False)
    assert cached is pb._gemm_workspace("cpu", 4096, 1280, 1280, False)
    assert (L.concord_gemm_workspace_need(4096, 1280, 1280, 0, None) + 1280 * 1280 * 2
            <= L.concord_gemm_workspace_need(4096, 1280, 1280, 1, None))
    # nothing is copied: the zeroed buffer of the device, its tile counters in use
    for M, N, K in [(308, 1280, 2048), (3, 5, 7)]:
        assert pb._gemm_workspace("cpu", M, N, K, True) is pb._gemm_workspace("cpu", M, N, K, True)
    pb._GEMM_WORKSPACES.pop("cpu")


@pytest.mark.parametrize("M,N,K,copied", [
    (16384, 50257, 768, 50264 * 768 * 2),            # dy's copy would pass 2^30 bytes: the weight's alone, for the forward
    (16384, 768, 50257, 768 * 50264 * 2),            # x's likewise: the weight's, for the dgrad
    (1 << 20, 505, 8, (1 << 20) * 512 * 2 + 512 * 8 * 2),   # dy's copy ends 14 bytes short of them
    (16384, 65, 384, 16384 * 72 * 2 + 72 * 384 * 2),   # x has whole chunks
    (2048, 320, 36, 2048 * 40 * 2 + 320 * 40 * 2),     # dy has
    (4, 33, 31, 4 * 32 * 2 + 4 * 40 * 2),              # too few rows and terms for the forward and the dgrad
])
def test_workspace_holds_the_copies_that_are_made(L, M, N, K, copied):
    """The room of a ragged layer's padded copies: none for an operand that is
    used as it is, nor for one that the fast kernels could not address."""
    N8, K8 = -(-N // 8) * 8, -(-K // 8) * 8
    # the split-K partials of the layer and of its padded twin bound the rest
    rest = max(L.concord_gemm_workspace_need(M, n, k, 0, None) for n in (N8, N8 - 4, N) for k in (K8, K8 - 4, K)
               if n % 8 == 0 and k % 8 == 0)
    need = L.concord_gemm_workspace_bytes(M, N, K)
    assert copied <= need <= copied + rest + 4 * 256


def test_lds_dma_waits_for_m0():
    """An LDS-DMA reads its LDS address from M0 and needs a wait state after the
    scalar write of it; the compiler adds none inside inline asm."""
    import glob
    csrc = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "concord_amd", "csrc")
    found = 0
    for path in glob.glob(os.path.join(csrc, "*")):
        for text in re.findall(r'asm volatile\("([^"]*)"', open(path).read()):
            lines = [l.strip() for l in text.replace("\\t", "").split("\\n")]
            for i, l in enumerate(lines):
                if re.search(r"\blds$", l):
                    found += 1
                    before = lines[:i]
                    assert before and before[-1].startswith("s_nop"), (os.path.basename(path), lines)
                    assert re.match(r"s_\w+ m0,", before[-2]), (os.path.basename(path), lines)
    assert found >= 3
