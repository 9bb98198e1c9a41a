"""GPU: the output projection whose K-chunk sums are added by the conversion in front of the FFN gives, bit for bit, what the projection
and the FFN give as two calls (there the sums are added by a launch of their own, in the same order; rows beyond 2048 add the squares of
their norm in another order, in 64 bits, whose last bit the 32-bit scale of these rows does not see).

test_outproj_ffn_launches.py: which of these shapes leave the sums to the conversion.
"""
import pytest

pytestmark = pytest.mark.gpu
T = {"q4_0": 2, "q5_0": 6, "q8_0": 8, "q4_k": 12, "q5_k": 13, "q6_k": 14, "iq4_nl": 20, "mxfp4": 39}
ROWS = [4, 20, 53, 200, 333]
# output projection, gate / up, hidden, attention width, FFN half width, columns between the residual's rows
SHAPES = [("q8_0", "q8_0", 1536, 1536, 3584, 0), ("q4_k", "q4_k", 4096, 4096, 14336, 0), ("q4_k", "q5_k", 2048, 5120, 8192, 4),
          ("q6_k", "iq4_nl", 768, 5120, 4096, 8), ("q6_k", "q4_0", 1024, 4096, 6144, 0), ("q4_k", "q4_k", 2304, 2304, 8192, 12),
          ("mxfp4", "q8_0", 1024, 6144, 4096, 8), ("q8_0", "q6_k", 2048, 2048, 6144, 0), ("q4_k", "q4_k", 1024, 1536, 14336, 0),
          ("q8_0", "q5_k", 2304, 2304, 6144, 0), ("q8_0", "q5_0", 2304, 2304, 6144, 4)]
# the sums lie where the conversion writes; rows that do not fit its registers; activations in block-scaled pairs, which it does not form
REFUSED = [("q4_k", "q4_k", 4096, 4096, 2048, 0), ("q4_k", "q4_k", 8448, 512, 8192, 0), ("q4_k", "mxfp4", 1024, 4096, 4096, 0)]


@pytest.mark.parametrize("rows", ROWS)
@pytest.mark.parametrize("out_type,gu_type,hidden,ins,half,pad", SHAPES + REFUSED)
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
