"""GPU: the output projection whose K-chunk sums are added by the conversion in front of the FFN gives, bit for bit, what the projection
and the FFN give as two calls (there the sums are added by a launch of their own, in the same order)."""
import numpy as np
import pytest

from test_matmul_plan import plan

pytestmark = pytest.mark.gpu
T = {"q8_0": 8, "q4_k": 12, "q5_k": 13, "q6_k": 14, "mxfp4": 39}


@pytest.mark.parametrize("rows", [4, 53, 200])
@pytest.mark.parametrize("out_type,gu_type,hidden,ins,half,pad", [
    ("q8_0", "q8_0", 1536, 1536, 3584, 0), ("q4_k", "q4_k", 4096, 4096, 2048, 0), ("q6_k", "q5_k", 768, 5120, 1024, 4),
    ("q4_k", "q4_k", 8448, 512, 1024, 0), ("q4_k", "mxfp4", 1024, 4096, 512, 0), ("mxfp4", "q8_0", 1024, 6144, 1024, 8)])
def test_two_calls_or_one(hip, rows, out_type, gu_type, hidden, ins, half, pad):
    import torch
    from tensorsharp_amd import QuantizedWeight, synth
    dev = torch.device("cuda")
    g = torch.Generator().manual_seed(rows + hidden)
    weight = lambda t, n, k, seed: QuantizedWeight(synth.random_weight(T[t], n, k, dev, seed=seed), T[t], k, n)
    out, gu, down = weight(out_type, hidden, ins, 1), weight(gu_type, 2 * half, hidden, 2), weight("q8_0", hidden, half, 3)
    wide = torch.randn((rows, hidden + pad), generator=g).cuda()
    attention, norm = torch.randn((rows, ins), generator=g).cuda(), (1 + 0.1 * torch.randn(hidden, generator=g)).cuda()
    one, two = wide.clone(), wide.clone()
    hip.UseCurrentStream()
    for _ in range(2):                                                       # (the second pass finds used scratch)
        one.copy_(wide), two.copy_(wide)
        hip.FusedOutProjFFN(one[:, :hidden], attention, out, norm, 1e-6, gu, down, half)
        hip.FusedMatMulQuantAdd(two[:, :hidden], attention, out)
        between = two.clone()
        hip.FusedFFNSwiGLUQuant(two[:, :hidden], two[:, :hidden], norm, 1e-6, gu, down, half)
        torch.cuda.synchronize()
        assert torch.equal(one, two) and not torch.equal(between, wide) and not torch.equal(two, between)


def test_the_shapes_leave_sums():
    # chunks, or the register kernel's second pass, of every projection above (else the two calls would not differ at all)
    assert all(plan(T[t], m, h, k, 1)[3] > 0 for t, h, k in (("q8_0", 1536, 1536), ("q4_k", 4096, 4096), ("q6_k", 768, 5120)) for m in (4, 53, 200))
