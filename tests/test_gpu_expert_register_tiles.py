"""GPU parity: expert tiles of 32 rows on the register-resident kernels by tile tables, where their edges are - first rows of a tile that are
no multiple of 32, partial and empty tiles, runs of units that cross into another expert, K in two chunks, and members of two types (their
launches have fewer tiles than the scratch was sized for).  test_register_kernel_launches.py says which kernels these stages launch.

Bar: the expert stage's of test_gpu_moe.py, the expert sets' of test_gpu_expert_sets.py."""
import numpy as np
import pytest

import inputs
from test_gpu_expert_sets import run, set_tol
from test_gpu_moe import run_gpu

pytestmark = pytest.mark.gpu
TYPES = {"q4_0": 2, "q8_0": 8, "q4_k": 12, "q5_k": 13, "q6_k": 14}
# format, experts, hidden, FFN, tokens, experts per token
STAGES = [("q5_k", 8, 2304, 1024, 40, 2), ("q6_k", 8, 2304, 1024, 40, 2), ("q8_0", 8, 2304, 1024, 40, 2), ("q4_k", 3, 4096, 512, 20, 2),
          ("q8_0", 3, 4096, 512, 20, 2), ("q6_k", 8, 1024, 2560, 40, 2), ("q8_0", 8, 1024, 2560, 40, 2), ("q4_k", 8, 4352, 1024, 40, 2),
          ("q6_k", 8, 4352, 1024, 40, 2), ("q4_0", 8, 4352, 1024, 40, 2)]


@pytest.mark.parametrize("name,E,H,F,T,k", STAGES)
def test_expert_stage(hip, oracle, name, E, H, F, T, k):
    import torch
    from tensorsharp_amd import synth
    t, rng = TYPES[name], np.random.default_rng(H + F)
    gu = synth.random_weight(t, E * 2 * F, H, torch.device("cuda"), seed=1, sigma=0.03).cpu().numpy()
    dn = synth.random_weight(t, E * H, F, torch.device("cuda"), seed=2, sigma=0.03).cpu().numpy()
    gb, db = [(rng.standard_normal((E, n)) * 0.1).astype(np.float32) for n in (2 * F, H)]
    hidden = rng.standard_normal((T, H)).astype(np.float32)
    logits = rng.standard_normal((T, E)).astype(np.float32)
    logits[:, 1] += 2.0                 # expert 1 takes most tokens (two row tiles in the larger stages)
    if E > k + 1:
        logits[:, E - 1] -= 50.0        # the last expert takes none
    ids, wts = oracle.moe_route(logits, k)
    ref = oracle.moe_forward(t, gu, gb, dn, db, E, H, F, hidden, ids, wts)
    for _ in range(2):                  # (the second pass finds used scratch)
        got = run_gpu(hip, t, gu, gb, dn, db, E, H, F, hidden, ids, wts)
        assert inputs.row_l2_err(got, ref) <= 1e-3, inputs.row_l2_err(got, ref)


@pytest.mark.parametrize("routed,shared,n,M", [("q6_k", "q4_0", 4, 20), ("q4_0", "q6_k", 2, 33)])
def test_members_of_two_types(hip, oracle, routed, shared, n, M):
    import torch
    from tensorsharp_amd import QuantizedWeight, synth
    H, I, rng = 4352, 2304, np.random.default_rng(n + M)

    def member(name, seed):
        raw = lambda rows, k, s: (TYPES[name], synth.random_weight(TYPES[name], rows, k, torch.device("cuda"), seed=s, sigma=0.03).cpu().numpy(), rows, k)
        return dict(gate=raw(I, H, seed), up=raw(I, H, seed + 1), down=raw(H, I, seed + 2))
    ex, sh = [member(routed, 10 * e) for e in range(n)], member(shared, 1000)
    w = rng.uniform(0.05, 0.6, n).astype(np.float32)
    x, base = [rng.standard_normal((M, H)).astype(np.float32) for _ in range(2)]
    ref, parts = oracle.expert_set(x, ex + [sh], list(w) + [0.7], base)
    dev = lambda d: QuantizedWeight(torch.from_numpy(d[1].reshape(-1)).cuda(), d[0], d[3], d[2])
    get = lambda key: [dev(e[key]) for e in ex]
    fn = lambda r, i: hip.MoEExpertsSwiGLUResidual(r, i, get("gate"), get("up"), get("down"), w, shared=[dev(sh[q]) for q in ("gate", "up", "down")],
                                                   shared_scalar=0.7)
    got = run(hip, True, fn, base.copy(), x)[0]
    assert np.all(np.abs(got - ref) <= set_tol(oracle, parts, list(w) + [0.7])), float(np.max(np.abs(got - ref) / set_tol(oracle, parts, list(w) + [0.7])))
