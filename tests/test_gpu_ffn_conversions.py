"""GPU: the conversions that form the gated activations of an FFN or an expert stage, in the activation orders and row lengths that the
other tests do not meet.

The FFN is compared with its parts (the gated rows formed by torch, then the added product).  Bar: the two differ by the rounding of the
fp32 gates, which moves an fp16 operand by one place at most: 2^-11 of each activation, so at most 2^-11 of a result row's terms, against 1e-3
of the row's norm.  The expert stage: the bar of test_gpu_moe.py."""
import numpy as np
import pytest

import inputs
from test_gpu_moe import run_gpu
from test_matmul_plan import TILES, plan

pytestmark = pytest.mark.gpu
TYPES = {"f16": 1, "q5_0": 6, "q4_k": 12, "q5_k": 13}


@pytest.mark.parametrize("down,rows,hidden,half", [("q4_k", 2000, 2560, 4096), ("q4_k", 2000, 2560, 9728), ("q5_k", 200, 512, 1024),
                                                   ("q5_k", 200, 512, 9216), ("q5_0", 200, 512, 9216), ("f16", 5, 512, 768)])
def test_ffn_and_its_parts(hip, down, rows, hidden, half):
    import torch
    from tensorsharp_amd import QuantizedWeight, synth
    dev, t = torch.device("cuda"), TYPES[down]
    g = torch.Generator().manual_seed(rows + half)
    gu = QuantizedWeight(synth.random_weight(8, 2 * half, hidden, dev, seed=1), 8, hidden, 2 * half)
    if down == "f16":
        raw = (torch.randn((hidden, half), generator=g) * 0.02).half().cuda().view(torch.uint8).reshape(-1)
    else:
        raw = synth.random_weight(t, hidden, half, dev, seed=2)
        assert plan(t, rows, hidden, half, 1)[0] == TILES
    dn = QuantizedWeight(raw, t, half, hidden)
    x, norm = torch.randn((rows, hidden), generator=g).cuda(), (1 + 0.1 * torch.randn(hidden, generator=g)).cuda()
    one, parts, product = x.clone(), x.clone(), torch.zeros_like(x)
    hip.UseCurrentStream()
    hip.FusedFFNSwiGLUQuant(one, one, norm, 1e-6, gu, dn, half)
    gates = torch.empty((rows, 2 * half), device=dev)
    hip.FusedRmsNormMatMulQuant(gates, parts, norm, 1e-6, gu)
    act = torch.nn.functional.silu(gates[:, :half]) * gates[:, half:]
    hip.FusedMatMulQuantAdd(parts, act, dn)
    hip.FusedMatMulQuantAdd(product, act, dn)
    torch.cuda.synchronize()
    bar = 1e-3 * product.norm(dim=1, keepdim=True)
    assert torch.isfinite(one).all() and (product.abs().amax(dim=1) > 0).all()
    assert ((one - parts).abs() <= bar).all(), float(((one - parts).abs() / bar).max())


def test_expert_stage_with_long_q5_k_rows(hip, oracle):
    # more than 160 tokens per expert (128-row tiles) and F > 8192: the gating conversion of 1024 threads in the nibble-pair order
    import torch
    from tensorsharp_amd import synth
    t, (E, H, F, T, k), rng = TYPES["q5_k"], (2, 256, 8448, 330, 1), np.random.default_rng(79)
    gu = synth.random_weight(t, E * 2 * F, H, torch.device("cuda"), seed=1, sigma=0.03).cpu().numpy()
    dn = synth.random_weight(t, E * H, F, torch.device("cuda"), seed=2, sigma=0.03).cpu().numpy()
    gb, db = [(rng.standard_normal((E, n)) * 0.1).astype(np.float32) for n in (2 * F, H)]
    hidden = rng.standard_normal((T, H)).astype(np.float32)
    ids, wts = oracle.moe_route(rng.standard_normal((T, E)).astype(np.float32), k)
    ref = oracle.moe_forward(t, gu, gb, dn, db, E, H, F, hidden, ids, wts)
    got = run_gpu(hip, t, gu, gb, dn, db, E, H, F, hidden, ids, wts)
    assert inputs.row_l2_err(got, ref) <= 1e-3, inputs.row_l2_err(got, ref)
