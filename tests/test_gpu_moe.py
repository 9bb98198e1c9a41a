"""GPU parity: MoE routing and the GPT-OSS expert stage through the C ABI against the oracle
(restating GptOssModel.cs:699-934).  Bar for the expert stage: max_j |y - ref| / ||ref row||_2 <= 1e-3."""
import numpy as np
import pytest

import inputs
from oracle.oracle import Q8_0, Q4_K, MXFP4

pytestmark = pytest.mark.gpu
T_ = {"q8_0": Q8_0, "q4_k": Q4_K, "mxfp4": MXFP4}


def test_route_matches_reference_semantics(hip, oracle):
    import torch
    rng = np.random.default_rng(61)
    T, E, k = 300, 32, 4
    logits = rng.standard_normal((T, E)).astype(np.float32)
    logits[3, 5] = logits[3, 9] = logits[3].max() + 1          # tie: first index wins
    logits[7, :] = 0.25                                         # all equal: 0,1,2,3
    wts, ids = hip.MoERoute(torch.from_numpy(logits).cuda(), k)
    torch.cuda.synchronize()
    ref_ids, ref_w = oracle.moe_route(logits, k)
    assert np.array_equal(ids.cpu().numpy(), ref_ids)
    np.testing.assert_allclose(wts.cpu().numpy(), ref_w, rtol=2e-6, atol=1e-7)
    for E2, k2 in ((8, 8), (130, 6), (64, 1)):
        lg = rng.standard_normal((17, E2)).astype(np.float32)
        w2, i2 = hip.MoERoute(torch.from_numpy(lg).cuda(), k2)
        ri, rw = oracle.moe_route(lg, k2)
        assert np.array_equal(i2.cpu().numpy(), ri)
        np.testing.assert_allclose(w2.cpu().numpy(), rw, rtol=2e-6, atol=1e-7)


@pytest.mark.parametrize("E,k", [(1, 1), (2, 2), (17, 16), (33, 4), (63, 5), (64, 16), (65, 4), (200, 8)])
def test_route_of_few_many_tied_and_infinite_logits(hip, oracle, E, k):
    """Up to 64 experts a lane of the token's wavefront holds a logit, beyond it reads them anew: ties across lanes and halves
    of the wavefront, rows with fewer finite logits than selections, infinities.  Ids exact; weights: one division and one
    exponential apart, as above."""
    import torch
    rng = np.random.default_rng(E * 31 + k)
    lg = np.round(rng.standard_normal((40, E)) * 2).astype(np.float32) / 2      # many ties
    lg[5, :] = -1.5
    lg[6, 1:] = -np.inf
    lg[7, : E // 2] = -np.inf
    lg[8, E - 1] = 40.0
    w, i = hip.MoERoute(torch.from_numpy(lg).cuda(), k)
    ri, rw = oracle.moe_route(lg, k)
    assert np.array_equal(i.cpu().numpy(), ri)
    np.testing.assert_allclose(w.cpu().numpy(), rw, rtol=2e-6, atol=1e-7)


def make_experts(oracle, t, E, H, F, rng, sigma=0.05):
    gu = oracle.quantize(t, (rng.standard_normal(E * 2 * F * H) * sigma).astype(np.float32))
    dn = oracle.quantize(t, (rng.standard_normal(E * H * F) * sigma).astype(np.float32))
    gb = (rng.standard_normal((E, 2 * F)) * 0.1).astype(np.float32)
    db = (rng.standard_normal((E, H)) * 0.1).astype(np.float32)
    return gu, gb, dn, db


def run_gpu(hip, t, gu, gb, dn, db, E, H, F, hidden, ids, wts):
    import torch
    c = lambda a: None if a is None else torch.from_numpy(np.ascontiguousarray(a)).cuda()
    out = hip.MoEExpertsGptOssForward(c(hidden), c(ids.astype(np.int32)), c(wts), c(gu), c(gb), c(dn), c(db), t, E, H, F)
    torch.cuda.synchronize()
    return out.cpu().numpy()


@pytest.mark.parametrize("name", ["mxfp4", "q8_0", "q4_k"])
@pytest.mark.parametrize("T,k", [(1, 4), (2, 4), (3, 4), (37, 2), (150, 4)])
def test_expert_stage_small_dims(hip, oracle, name, T, k):
    rng = np.random.default_rng(63 + T)
    E, H, F = 8, 512, 768
    t = T_[name]
    gu, gb, dn, db = make_experts(oracle, t, E, H, F, rng)
    hidden = rng.standard_normal((T, H)).astype(np.float32)
    ids, wts = oracle.moe_route(rng.standard_normal((T, E)).astype(np.float32), k)
    ref = oracle.moe_forward(t, gu, gb, dn, db, E, H, F, hidden, ids, wts)
    got = run_gpu(hip, t, gu, gb, dn, db, E, H, F, hidden, ids, wts)
    assert inputs.row_l2_err(got, ref) <= 1e-3, (name, T, inputs.row_l2_err(got, ref))
    # without biases
    ref2 = oracle.moe_forward(t, gu, None, dn, None, E, H, F, hidden, ids, wts)
    got2 = run_gpu(hip, t, gu, None, dn, None, E, H, F, hidden, ids, wts)
    assert inputs.row_l2_err(got2, ref2) <= 1e-3


@pytest.mark.parametrize("name", ["q4_0", "q4_1", "q5_0", "q5_1", "iq4_nl", "q5_k", "q6_k"])
@pytest.mark.parametrize("T", [1, 2])
def test_decode_stage_every_other_gemv_format(hip, oracle, name, T):
    """One or two tokens of experts in the block formats that have a GEMV kernel but no early expert records: the gate_up
    launch (expert ids read on the device, paired store) and the down launches read their problem fields where they need
    them.  Random valid blocks; reference = the oracle's expert stage over the bit-exact dequantized weights."""
    import torch
    from oracle.oracle import MORE_TYPES
    from tensorsharp_amd import synth
    t = MORE_TYPES[name]
    rng = np.random.default_rng(77 + T)
    E, H, F, k = 6, 512, 768, 4
    cpu = torch.device("cpu")
    gu = synth.random_weight(t, E * 2 * F, H, cpu, seed=21, sigma=0.05).numpy()
    dn = synth.random_weight(t, E * H, F, cpu, seed=22, sigma=0.05).numpy()
    gb = (rng.standard_normal((E, 2 * F)) * 0.1).astype(np.float32)
    db = (rng.standard_normal((E, H)) * 0.1).astype(np.float32)
    hidden = rng.standard_normal((T, H)).astype(np.float32)
    ids, wts = oracle.moe_route(rng.standard_normal((T, E)).astype(np.float32), k)
    ref = oracle.moe_forward(t, gu, gb, dn, db, E, H, F, hidden, ids, wts)
    got = run_gpu(hip, t, gu, gb, dn, db, E, H, F, hidden, ids, wts)
    assert inputs.row_l2_err(got, ref) <= 1e-3, (name, T, inputs.row_l2_err(got, ref))


@pytest.mark.parametrize("name", ["mxfp4", "q4_k"])
def test_expert_tiles_of_128_rows(hip, oracle, name):
    # more than 160 rows per expert on average: the grouped GEMM runs 128-row tiles instead of 32-row ones (MXFP4: with a
    # hidden size past the 3072 that the 48-row block-scaled units take)
    rng = np.random.default_rng(71)
    E, H, F, T, k = 4, 3328 if name == "mxfp4" else 256, 256, 400, 2
    t = T_[name]
    gu, gb, dn, db = make_experts(oracle, t, E, H, F, rng)
    hidden = rng.standard_normal((T, H)).astype(np.float32)
    ids, wts = oracle.moe_route(rng.standard_normal((T, E)).astype(np.float32), k)
    ref = oracle.moe_forward(t, gu, gb, dn, db, E, H, F, hidden, ids, wts)
    got = run_gpu(hip, t, gu, gb, dn, db, E, H, F, hidden, ids, wts)
    assert inputs.row_l2_err(got, ref) <= 1e-3, (name, inputs.row_l2_err(got, ref))


@pytest.mark.parametrize("name", ["mxfp4", "q4_k", "q8_0"])
def test_intermediate_rows_longer_than_one_conversion_pass(hip, oracle, name):
    # F > 8192: the SwiGLU-forming conversion of the down projection's activations runs its 1024-thread form; more than
    # 160 tokens per expert, so MXFP4 too stays on fp16 operands (128-row tiles)
    rng = np.random.default_rng(77)
    E, H, F, T, k = 2, 256, 8448, 330, 1
    t = T_[name]
    gu, gb, dn, db = make_experts(oracle, t, E, H, F, rng, sigma=0.03)
    hidden = rng.standard_normal((T, H)).astype(np.float32)
    ids, wts = oracle.moe_route(rng.standard_normal((T, E)).astype(np.float32), k)
    ref = oracle.moe_forward(t, gu, gb, dn, db, E, H, F, hidden, ids, wts)
    got = run_gpu(hip, t, gu, gb, dn, db, E, H, F, hidden, ids, wts)
    assert inputs.row_l2_err(got, ref) <= 1e-3, (name, inputs.row_l2_err(got, ref))


@pytest.mark.parametrize("T", [1, 2])
def test_top_1_routing(hip, oracle, T):
    rng = np.random.default_rng(73)
    E, H, F = 8, 512, 768
    gu, gb, dn, db = make_experts(oracle, MXFP4, E, H, F, rng)
    hidden = rng.standard_normal((T, H)).astype(np.float32)
    ids, wts = oracle.moe_route(rng.standard_normal((T, E)).astype(np.float32), 1)
    ref = oracle.moe_forward(MXFP4, gu, gb, dn, db, E, H, F, hidden, ids, wts)
    got = run_gpu(hip, MXFP4, gu, gb, dn, db, E, H, F, hidden, ids, wts)
    assert inputs.row_l2_err(got, ref) <= 1e-3, inputs.row_l2_err(got, ref)


@pytest.mark.parametrize("T", [1, 40])
def test_down_bias_at_an_address_that_is_not_16_byte_aligned(hip, oracle, T):
    # the weighted sum over a token's experts reads rows, bias and output as 16-byte vectors only when all are aligned
    import torch
    rng = np.random.default_rng(75)
    E, H, F, k = 8, 512, 768, 4
    gu, gb, dn, db = make_experts(oracle, MXFP4, E, H, F, rng)
    hidden = rng.standard_normal((T, H)).astype(np.float32)
    ids, wts = oracle.moe_route(rng.standard_normal((T, E)).astype(np.float32), k)
    ref = oracle.moe_forward(MXFP4, gu, gb, dn, db, E, H, F, hidden, ids, wts)
    c = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    buf = torch.zeros(E * H + 4, dtype=torch.float32, device="cuda")
    buf[1:1 + E * H] = c(db).reshape(-1)
    out = hip.MoEExpertsGptOssForward(c(hidden), c(ids.astype(np.int32)), c(wts), c(gu), c(gb), c(dn), buf[1:1 + E * H].view(E, H),
                                      MXFP4, E, H, F)
    torch.cuda.synchronize()
    assert inputs.row_l2_err(out.cpu().numpy(), ref) <= 1e-3


def test_unbalanced_and_empty_experts(hip, oracle):
    rng = np.random.default_rng(65)
    E, H, F, T, k = 16, 256, 256, 200, 2
    gu, gb, dn, db = make_experts(oracle, MXFP4, E, H, F, rng)
    hidden = rng.standard_normal((T, H)).astype(np.float32)
    ids = np.zeros((T, k), dtype=np.int32)
    ids[:, 0] = 3                       # one expert takes every token, most experts stay empty
    ids[:, 1] = np.where(np.arange(T) % 7 == 0, 15, 9)
    wts = rng.random((T, k)).astype(np.float32)
    ref = oracle.moe_forward(MXFP4, gu, gb, dn, db, E, H, F, hidden, ids, wts)
    got = run_gpu(hip, MXFP4, gu, gb, dn, db, E, H, F, hidden, ids, wts)
    assert inputs.row_l2_err(got, ref) <= 1e-3


# MXFP4 experts whose gate_up rows are 1025 .. 3072 long form bias + SwiGLU in the gate_up GEMM's epilogue and write the
# down projection's block-scaled activations from there: row lengths at both ends of that range and of both k-tile
# counts per wavefront, F / 32 even and odd (an odd count leaves half a k-tile of padding), experts with more than 32
# tokens (two row tiles), partly filled tiles and empty experts, with and without biases.  More than 20 tokens per expert
# on average (the first two cases and the last) run in 48-row units, the others in 32-row units.
@pytest.mark.parametrize("E,H,F,T,k", [(4, 1088, 160, 70, 2), (4, 2048, 256, 130, 2), (8, 2880, 96, 40, 4),
                                       (4, 3072, 512, 9, 2), (4, 1536, 2880, 40, 2), (2, 3072, 1024, 60, 2)])
def test_gate_up_epilogue_writes_down_activations(hip, oracle, E, H, F, T, k):
    rng = np.random.default_rng(1000 + H + F)
    gu, gb, dn, db = make_experts(oracle, MXFP4, E, H, F, rng, sigma=0.03)
    hidden = rng.standard_normal((T, H)).astype(np.float32)
    logits = rng.standard_normal((T, E)).astype(np.float32)
    logits[:, 1] += 2.0                 # expert 1 takes most tokens
    logits[:, E - 1] -= 50.0            # the last expert takes none
    ids, wts = oracle.moe_route(logits, k)
    ref = oracle.moe_forward(MXFP4, gu, gb, dn, db, E, H, F, hidden, ids, wts)
    got = run_gpu(hip, MXFP4, gu, gb, dn, db, E, H, F, hidden, ids, wts)
    assert inputs.row_l2_err(got, ref) <= 1e-3, inputs.row_l2_err(got, ref)
    ref2 = oracle.moe_forward(MXFP4, gu, None, dn, None, E, H, F, hidden, ids, wts)
    got2 = run_gpu(hip, MXFP4, gu, None, dn, None, E, H, F, hidden, ids, wts)
    assert inputs.row_l2_err(got2, ref2) <= 1e-3, inputs.row_l2_err(got2, ref2)


@pytest.mark.parametrize("H,F", [(32, 672), (64, 96), (224, 64)])
def test_narrow_mxfp4_stages_stay_on_fp16_operands(hip, oracle, H, F):
    """Rows of a few dozen outputs: the MX fp6 pairs of the block-scaled path leave every activation with an error of up to
    2^-10 of its block's largest magnitude, which against the norm of a 32-wide result row comes to 1e-3 (a sweep case
    measured 1.24e-3 at H = 32); stages narrower than 256 (H) / 128 (F) therefore run on fp16 operands.  Same bar as every
    matmul: row-L2 <= 1e-3."""
    rng = np.random.default_rng(2000 + H)
    E, T, k = 4, 200, 2
    gu, _, dn, _ = make_experts(oracle, MXFP4, E, H, F, rng)
    hidden = rng.standard_normal((T, H)).astype(np.float32)
    ids, wts = oracle.moe_route(rng.standard_normal((T, E)).astype(np.float32), k)
    ref = oracle.moe_forward(MXFP4, gu, None, dn, None, E, H, F, hidden, ids, wts)
    got = run_gpu(hip, MXFP4, gu, None, dn, None, E, H, F, hidden, ids, wts)
    assert inputs.row_l2_err(got, ref) <= 1e-3, inputs.row_l2_err(got, ref)


@pytest.fixture(scope="module")
def cfg4_weights(oracle):
    E, H, F = 32, 2880, 2880
    gu = np.concatenate([oracle.quantize(MXFP4, inputs.weights("cfg4.gate_up", 2 * F * H, seed=e)) for e in range(E)])
    dn = np.concatenate([oracle.quantize(MXFP4, inputs.weights("cfg4.down", H * F, seed=e)) for e in range(E)])
    return gu, dn


@pytest.mark.parametrize("T", [1, 256])
def test_config4_mxfp4_moe(hip, oracle, cfg4_weights, T):
    """32 experts, top-4, hidden 2880, gate_up 5760x2880, down 2880x2880, T = 1 and 256.
    Expert e's weights are the seeded N(0, 0.02) values (seed e) quantized as the reference quantizes them; expert 0 is
    the tensor whose reference bytes are pinned by the digests sha_cfg4.*.  Every token (T = 1) or 64 tokens (T = 256)
    are checked against the oracle."""
    import torch
    E, H, F, k = 32, 2880, 2880, 4
    gu, dn = cfg4_weights
    rng = np.random.default_rng(67)
    hidden = rng.standard_normal((T, H)).astype(np.float32)
    ids = np.stack([rng.permutation(E)[:k] for _ in range(T)]).astype(np.int32)   # uniform without replacement
    lg = rng.standard_normal((T, k)).astype(np.float32)
    wts = np.exp(lg - lg.max(1, keepdims=True))
    wts = (wts / wts.sum(1, keepdims=True)).astype(np.float32)
    c = lambda a: torch.from_numpy(a).cuda()
    out = hip.MoEExpertsGptOssForward(c(hidden), c(ids), c(wts), c(gu), None, c(dn), None, MXFP4, E, H, F)
    torch.cuda.synchronize()
    got = out.cpu().numpy()
    rows = [0] if T == 1 else sorted(set([0, 1, 31, 32, 100, 255]) | set(int(v) for v in rng.choice(T, 64, replace=False)))[:70]
    ref = oracle.moe_forward(MXFP4, gu, None, dn, None, E, H, F, hidden[rows], ids[rows], wts[rows])
    for i, r in enumerate(rows):
        e = inputs.row_l2_err(got[r:r + 1], ref[i:i + 1])
        assert e <= 1e-3, (T, r, e)
    assert np.all(np.isfinite(got))
