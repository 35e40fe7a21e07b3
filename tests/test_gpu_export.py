"""The grouped export launch against one materialise call per layer."""

import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shapes", [[(1, 1)], [(3, 7), (129, 264), (1280, 1280), (1, 8200)],
                                    [(5 + i, 8 * i + 3) for i in range(30)]])   # more than one launch's items
def test_grouped_export_matches_layers(shapes):
    import concord_amd as ca
    torch.manual_seed(len(shapes))
    layers = [ca.ConcordLinearPackedB(k, n, bias=i % 3 != 2, device="cuda") for i, (n, k) in enumerate(shapes)]
    for m in layers:
        if m.bias is not None:
            m.bias.data.normal_()
    names = [str(i) for i in range(len(layers))]
    sd = ca.consolidated_state_dict(layers, names)
    assert list(sd) == [f"{n}.{x}" for n, m in zip(names, layers)
                        for x in (["weight", "bias"] if m.bias is not None else ["weight"])]
    for n, m in zip(names, layers):
        assert torch.equal(sd[n + ".weight"], m.consolidated_weight())
        if m.bias is not None:
            assert torch.equal(sd[n + ".bias"], m.bias.detach())
            assert sd[n + ".bias"].data_ptr() != m.bias.data_ptr()


def test_group_items_with_pitch_and_odd_copies():
    import concord_amd as ca
    from concord_amd import _lib as C
    torch.manual_seed(0)
    m = ca.ConcordLinearPackedB(72, 40, bias=False, device="cuda")
    ref = m.consolidated_weight()
    wide = torch.full((40, 81), 7.0, dtype=torch.bfloat16, device="cuda")   # an odd output pitch
    src = torch.randint(0, 255, (1003,), dtype=torch.uint8, device="cuda")
    dst = torch.zeros(1010, dtype=torch.uint8, device="cuda")
    f = [m.packed_w.data_ptr(), m.packed_w.stride(0), m.row_exp.data_ptr(), m.col_exp.data_ptr(), 40, 72,
         wide.data_ptr(), 81, m.MANTISSA_BIAS,
         0, 0, src.data_ptr() + 1, 0, 1001, 1, dst.data_ptr() + 3, 0, 0]
    C.check(C.lib().concord_materialize_group((ctypes.c_int64 * 18)(*f), 2, 1, C.stream_of(m.packed_w.device)), "group")
    assert torch.equal(wide[:, :72], ref) and torch.all(wide[:, 72:] == 7.0)
    assert torch.equal(dst[3:1004], src[1:1002]) and int(dst[:3].sum()) == 0 and int(dst[1004:].sum()) == 0
