"""The bits of the Muon drive: its split counts order the fp32 sums of fifteen
products that round to bf16 in turn, so a change of plan changes the result."""
import hashlib

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

# sha256 of the drive of 1e-3 RandomState(n + k).randn(n, k), as the drive gave
# it before its products ran on the LDS-DMA kernels: split and unsplit
# symmetric products, both orientations, widths that are multiples of 8, of 4
# and of neither
DIGESTS = [(8, 8, "a04f39a04e02f1ef"), (64, 72, "b8f30520027959cf"), (136, 200, "8c2e2a221a71fa8e"),
           (320, 1280, "28af7884bd9c4d99"), (640, 640, "a086b210ccd8e30c"), (1280, 5120, "b6836f3ab3c8ec12"),
           (2560, 640, "c08887a5e3379db8"), (65, 384, "c587d300544f034f"), (1001, 645, "ee92edecb39a93c1"),
           (100, 100, "048564d12e1ccaa3"), (1284, 1284, "faee22d840381ed5"), (129, 72, "74c22aa7a3e13864"),
           (2050, 645, "207080f57e165ef5")]


@pytest.mark.parametrize("N,K,digest", DIGESTS)
def test_muon_drive_bits(N, K, digest):
    import concord_amd as ca
    g = torch.from_numpy((1e-3 * np.random.RandomState(N + K).randn(N, K)).astype(np.float32)).to(torch.bfloat16)
    o = ca.muon_ns5(g.cuda()).cpu().view(torch.int16).numpy()
    assert hashlib.sha256(o.tobytes()).hexdigest()[:16] == digest
