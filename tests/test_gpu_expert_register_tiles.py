"""GPU parity: expert tiles of 32 rows on the register-resident kernels by tile tables: K in two chunks and members of two types (their
launches have fewer tiles than the scratch was sized for, and share the results' rows).

Bar: the expert sets' of test_gpu_expert_sets.py."""
import numpy as np
import pytest

from test_gpu_expert_sets import run, set_tol

pytestmark = pytest.mark.gpu
TYPES = {"q4_0": 2, "q6_k": 14}


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
