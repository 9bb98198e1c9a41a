"""GPU parity: whole-layer decode (TSHip_TransformerLayerDecode / ModelDecode, device and host forms) against the oracle's restatement
of the bridge's layer graph (ggml_ops_transformer.cpp:379-470) on the same weights, token by token with a growing KV cache.

Bar: ||hidden - ref||_2 <= 3e-3 ||ref||_2 per token (four chained matmuls with fp16 operands, each held to 1e-3 of its
own row norm elsewhere) and the same for the K / V rows written."""
import os

import numpy as np
import pytest

from oracle.oracle import Q8_0, Q4_K, MXFP4, Q6_K

pytestmark = pytest.mark.gpu
GOLD = os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden", "layer.npz")


def rel(a, b):
    return float(np.linalg.norm(a.astype(np.float64) - b) / max(np.linalg.norm(b), 1e-30))


def to_device_layer(layer, torch, QuantizedWeight, dims):
    c = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    d = {k: (None if layer[k] is None else c(layer[k])) for k in ("attn_norm", "q_norm", "k_norm", "ffn_norm")}
    for k, (ne0, ne1) in dims.items():
        d[k] = QuantizedWeight(c(layer[k][1]), layer[k][0], ne0, ne1)
    return d


def make_layer(oracle, rng, hidden, heads, kv_heads, head_dim, inter, types, qk_norm=True):
    q_dim, k_dim = heads * head_dim, kv_heads * head_dim
    w = lambda t, n, k: (t, oracle.quantize(t, (rng.standard_normal(n * k) * 0.04).astype(np.float32)))
    layer = {"attn_norm": rng.uniform(0.5, 1.5, hidden).astype(np.float32), "ffn_norm": rng.uniform(0.5, 1.5, hidden).astype(np.float32),
             "q_norm": rng.uniform(0.5, 1.5, head_dim).astype(np.float32) if qk_norm else None,
             "k_norm": rng.uniform(0.5, 1.5, head_dim).astype(np.float32) if qk_norm else None,
             "qkv": w(types[0], q_dim + 2 * k_dim, hidden), "o": w(types[1], hidden, q_dim),
             "gate_up": w(types[2], 2 * inter, hidden), "down": w(types[3], hidden, inter), "intermediate": inter}
    dims = {"qkv": (hidden, q_dim + 2 * k_dim), "o": (q_dim, hidden), "gate_up": (hidden, 2 * inter), "down": (inter, hidden)}
    return layer, dims


@pytest.mark.parametrize("types,rope_mode,qk_norm", [((Q4_K, Q4_K, Q4_K, Q4_K), 2, True), ((Q8_0, Q8_0, Q8_0, Q8_0), 0, False),
                                                      ((MXFP4, MXFP4, MXFP4, MXFP4), 2, True)])
def test_layer_decode_tokens_in_sequence(hip, oracle, types, rope_mode, qk_norm):
    import torch
    from tensorsharp_amd import QuantizedWeight
    rng = np.random.default_rng(101 + rope_mode)
    hidden, heads, kv_heads, head_dim, inter, max_seq = 512, 8, 2, 64, 768 if types[0] != Q4_K else 1024, 600
    layer, dims = make_layer(oracle, rng, hidden, heads, kv_heads, head_dim, inter, types, qk_norm)
    dev = to_device_layer(layer, torch, QuantizedWeight, dims)
    kc = np.zeros((kv_heads, max_seq, head_dim), dtype=np.float32)
    vc = np.zeros_like(kc)
    # a long prefix already in the caches (several attention splits), then four new tokens
    prefix = 517
    kc[:, :prefix] = rng.standard_normal((kv_heads, prefix, head_dim)).astype(np.float32)
    vc[:, :prefix] = rng.standard_normal((kv_heads, prefix, head_dim)).astype(np.float32)
    kd, vd = torch.from_numpy(kc.copy()).cuda(), torch.from_numpy(vc.copy()).cuda()
    for pos in range(prefix, prefix + 4):
        h = rng.standard_normal(hidden).astype(np.float32)
        hd = torch.from_numpy(h.copy()).cuda()
        oracle.layer_decode(h, layer, kc, vc, heads, kv_heads, head_dim, pos, 1e-6, 10000.0, 1.0, rope_mode)
        hip.TransformerLayerDecode(hd, dev["attn_norm"], dev["qkv"], dev["q_norm"], dev["k_norm"], dev["o"], dev["ffn_norm"],
                                   dev["gate_up"], dev["down"], kd, vd, heads, kv_heads, head_dim, pos, 1e-6, 10000.0, 1.0, rope_mode)
        torch.cuda.synchronize()
        assert rel(hd.cpu().numpy(), h) <= 3e-3, (pos, rel(hd.cpu().numpy(), h))
        assert rel(kd.cpu().numpy()[:, pos], kc[:, pos]) <= 3e-3 and rel(vd.cpu().numpy()[:, pos], vc[:, pos]) <= 3e-3
    assert np.array_equal(kd.cpu().numpy()[:, :prefix], kc[:, :prefix])              # older rows untouched


def test_first_token_and_the_reference_graph_known_answer(hip, oracle):
    # the three tokens of the fixture computed by the reference's ggml CPU graph (coarse: int8 activations there)
    import torch
    from tensorsharp_amd import QuantizedWeight
    g = np.load(GOLD)
    L = dict(hidden=256, heads=4, kv_heads=2, head_dim=64, inter=512, max_seq=16)
    layer = {"attn_norm": g["layer_attn_norm"], "q_norm": g["layer_q_norm"], "k_norm": g["layer_k_norm"], "ffn_norm": g["layer_ffn_norm"],
             "qkv": (Q8_0, g["layer_qkv"]), "o": (Q8_0, g["layer_o"]), "gate_up": (Q4_K, g["layer_gate_up"]),
             "down": (Q4_K, g["layer_down"]), "intermediate": L["inter"]}
    dims = {"qkv": (256, 512), "o": (256, 256), "gate_up": (256, 1024), "down": (512, 256)}
    dev = to_device_layer(layer, torch, QuantizedWeight, dims)
    kd = torch.zeros((2, 16, 64), dtype=torch.float32, device="cuda")
    vd = torch.zeros_like(kd)
    kc, vc = np.zeros((2, 16, 64), np.float32), np.zeros((2, 16, 64), np.float32)
    for pos in range(3):
        hd = torch.from_numpy(g["layer_hidden_in"][pos].copy()).cuda()
        h = g["layer_hidden_in"][pos].copy()
        oracle.layer_decode(h, layer, kc, vc, 4, 2, 64, pos, 1e-6, 10000.0, 1.0, 2)
        hip.TransformerLayerDecode(hd, dev["attn_norm"], dev["qkv"], dev["q_norm"], dev["k_norm"], dev["o"], dev["ffn_norm"],
                                   dev["gate_up"], dev["down"], kd, vd, 4, 2, 64, pos, 1e-6, 10000.0, 1.0, 2)
        torch.cuda.synchronize()
        got = hd.cpu().numpy()
        assert rel(got, h) <= 3e-3, pos
        assert rel(got, g["layer_hidden_out"][pos]) <= 2e-2, pos


def test_model_decode_equals_layers_in_sequence_and_mixed_formats(hip, oracle):
    # two layers through the model entry point; down projections in Q6_K
    import torch
    from tensorsharp_amd import QuantizedWeight, synth
    rng = np.random.default_rng(107)
    hidden, heads, kv_heads, head_dim, inter, max_seq = 512, 4, 4, 128, 1024, 8
    layers, devs, caches = [], [], []
    for li in range(2):
        layer, dims = make_layer(oracle, rng, hidden, heads, kv_heads, head_dim, inter, (Q4_K, Q4_K, Q4_K, Q4_K))
        gt = torch.Generator()
        gt.manual_seed(li)
        layer["down"] = (Q6_K, synth.quantize_q6_k_simple(torch.randn((hidden, inter), generator=gt) * 0.04).numpy())
        layers.append(layer)
        d = to_device_layer(layer, torch, QuantizedWeight, dims)
        d["k_cache"] = torch.zeros((kv_heads, max_seq, head_dim), dtype=torch.float32, device="cuda")
        d["v_cache"] = torch.zeros_like(d["k_cache"])
        devs.append(d)
        caches.append((np.zeros((kv_heads, max_seq, head_dim), np.float32), np.zeros((kv_heads, max_seq, head_dim), np.float32)))
    for pos in range(2):
        h = rng.standard_normal(hidden).astype(np.float32)
        hd = torch.from_numpy(h.copy()).cuda()
        for layer, (kc, vc) in zip(layers, caches):
            oracle.layer_decode(h, layer, kc, vc, heads, kv_heads, head_dim, pos, 1e-5, 1e6, 1.0, 2)
        hip.TransformerModelDecode(hd, devs, heads, kv_heads, head_dim, pos, 1e-5, 1e6, 1.0, 2)
        torch.cuda.synchronize()
        assert rel(hd.cpu().numpy(), h) <= 5e-3, (pos, rel(hd.cpu().numpy(), h))


def test_layer_decode_argument_errors(hip, oracle):
    import torch
    from tensorsharp_amd import QuantizedWeight
    rng = np.random.default_rng(109)
    layer, dims = make_layer(oracle, rng, 256, 4, 2, 64, 256, (Q8_0, Q8_0, Q8_0, Q8_0))
    dev = to_device_layer(layer, torch, QuantizedWeight, dims)
    kd = torch.zeros((2, 4, 64), dtype=torch.float32, device="cuda")
    vd = torch.zeros_like(kd)
    h = torch.zeros(256, dtype=torch.float32, device="cuda")
    call = lambda **kw: hip.TransformerLayerDecode(h, dev["attn_norm"], dev["qkv"], dev["q_norm"], dev["k_norm"], dev["o"], dev["ffn_norm"],
                                                   dev["gate_up"], dev["down"], kd, vd, kw.get("heads", 4), 2, 64, kw.get("pos", 0), 1e-6,
                                                   10000.0, 1.0, kw.get("mode", 2))
    with pytest.raises(RuntimeError, match="position outside the KV cache"):
        call(pos=4)
    with pytest.raises(RuntimeError, match="dims don't match"):
        call(heads=8)
    with pytest.raises(RuntimeError, match="rope mode"):
        call(mode=8)
    call()


@pytest.mark.parametrize("heads,kv_heads,head_dim,rope_mode,prefix", [(8, 1, 80, 0, 130), (8, 2, 256, 2, 63), (16, 2, 96, 2, 2100),
                                                                      (6, 3, 192, 0, 0), (32, 4, 128, 2, 700)])
def test_head_shapes_groupings_and_split_counts(hip, oracle, heads, kv_heads, head_dim, rope_mode, prefix):
    # every head width the attention kernel is built for, 1 / 2 / 4 / 8 query heads per workgroup, one to many splits
    import torch
    from tensorsharp_amd import QuantizedWeight
    rng = np.random.default_rng(heads * 1000 + head_dim)
    hidden, inter, max_seq = 256, 512, prefix + 3
    layer, dims = make_layer(oracle, rng, hidden, heads, kv_heads, head_dim, inter, (Q8_0, Q8_0, Q8_0, Q8_0), True)
    dev = to_device_layer(layer, torch, QuantizedWeight, dims)
    kc = np.zeros((kv_heads, max_seq, head_dim), dtype=np.float32)
    vc = np.zeros_like(kc)
    kc[:, :prefix] = rng.standard_normal((kv_heads, prefix, head_dim)).astype(np.float32)
    vc[:, :prefix] = rng.standard_normal((kv_heads, prefix, head_dim)).astype(np.float32)
    kd, vd = torch.from_numpy(kc.copy()).cuda(), torch.from_numpy(vc.copy()).cuda()
    for pos in range(prefix, prefix + 3):
        h = rng.standard_normal(hidden).astype(np.float32)
        hd = torch.from_numpy(h.copy()).cuda()
        oracle.layer_decode(h, layer, kc, vc, heads, kv_heads, head_dim, pos, 1e-6, 10000.0, 1.0, rope_mode)
        hip.TransformerLayerDecode(hd, dev["attn_norm"], dev["qkv"], dev["q_norm"], dev["k_norm"], dev["o"], dev["ffn_norm"],
                                   dev["gate_up"], dev["down"], kd, vd, heads, kv_heads, head_dim, pos, 1e-6, 10000.0, 1.0, rope_mode)
        torch.cuda.synchronize()
        assert rel(hd.cpu().numpy(), h) <= 3e-3, (pos, rel(hd.cpu().numpy(), h))
        assert rel(kd.cpu().numpy()[:, pos], kc[:, pos]) <= 1e-5 and rel(vd.cpu().numpy()[:, pos], vc[:, pos]) <= 1e-5


@pytest.mark.parametrize("head_dim,prefix", [(64, 1023), (256, 1023), (128, 8191)])
def test_split_merge_on_few_and_many_wavefronts(hip, oracle, head_dim, prefix):
    # the merge takes 4 wavefronts up to 16 splits and 16 beyond (positions 1023 -> 1024), and a second batch of rows from
    # 65 splits on (positions 8191 -> 8192)
    test_head_shapes_groupings_and_split_counts(hip, oracle, 2, 1, head_dim, 2, prefix)


@pytest.mark.parametrize("head_dim", [64, 80, 96, 128, 192, 256])
@pytest.mark.parametrize("group,kv_heads,prefix", [(1, 4, 70), (4, 8, 2100), (8, 8, 2100)])
def test_every_attention_instantiation(hip, oracle, head_dim, group, kv_heads, prefix):
    # the attention kernel is compiled per head width and per number of query heads a workgroup serves (1, 2, 4, 8); the
    # launcher serves 4 or 8 only when that still leaves 128 workgroups, i.e. with many KV heads and splits - shapes the
    # tests above do not reach
    import torch
    from tensorsharp_amd import QuantizedWeight
    heads = group * kv_heads
    rng = np.random.default_rng(head_dim * 10 + group)
    hidden, inter, max_seq = 256, 256, prefix + 2
    layer, dims = make_layer(oracle, rng, hidden, heads, kv_heads, head_dim, inter, (Q8_0, Q8_0, Q8_0, Q8_0), True)
    dev = to_device_layer(layer, torch, QuantizedWeight, dims)
    kc = np.zeros((kv_heads, max_seq, head_dim), dtype=np.float32)
    vc = np.zeros_like(kc)
    kc[:, :prefix] = rng.standard_normal((kv_heads, prefix, head_dim)).astype(np.float32)
    vc[:, :prefix] = rng.standard_normal((kv_heads, prefix, head_dim)).astype(np.float32)
    kd, vd = torch.from_numpy(kc.copy()).cuda(), torch.from_numpy(vc.copy()).cuda()
    for pos in range(prefix, prefix + 2):
        h = rng.standard_normal(hidden).astype(np.float32)
        hd = torch.from_numpy(h.copy()).cuda()
        oracle.layer_decode(h, layer, kc, vc, heads, kv_heads, head_dim, pos, 1e-6, 10000.0, 1.0, 2)
        hip.TransformerLayerDecode(hd, dev["attn_norm"], dev["qkv"], dev["q_norm"], dev["k_norm"], dev["o"], dev["ffn_norm"],
                                   dev["gate_up"], dev["down"], kd, vd, heads, kv_heads, head_dim, pos, 1e-6, 10000.0, 1.0, 2)
        torch.cuda.synchronize()
        assert rel(hd.cpu().numpy(), h) <= 3e-3, (pos, rel(hd.cpu().numpy(), h))
        assert rel(kd.cpu().numpy()[:, pos], kc[:, pos]) <= 1e-5 and rel(vd.cpu().numpy()[:, pos], vc[:, pos]) <= 1e-5


@pytest.mark.parametrize("head_dim", [64, 80, 96, 128, 192, 256])
@pytest.mark.parametrize("group,kv_heads,prefix", [(1, 4, 0), (2, 4, 63), (1, 4, 127), (2, 32, 511), (4, 8, 1100), (8, 8, 1100)])
def test_attention_rows_per_group_at_their_borders(hip, oracle, head_dim, group, kv_heads, prefix):
    """Two or four cache rows per group of lanes, 1 to 8 query heads per workgroup: one position, the last position of a
    single split and the first beyond it (64 -> 65, 128 -> 129), the border at one workgroup per CU (512 -> 513 for 32 KV
    heads).  Cache rows past the position hold NaN and must not be read into any result."""
    import torch
    from tensorsharp_amd import QuantizedWeight
    heads = group * kv_heads
    rng = np.random.default_rng(head_dim * 10 + group + prefix)
    hidden, inter, max_seq = 256, 256, prefix + 70
    layer, dims = make_layer(oracle, rng, hidden, heads, kv_heads, head_dim, inter, (Q8_0, Q8_0, Q8_0, Q8_0), True)
    dev = to_device_layer(layer, torch, QuantizedWeight, dims)
    kc = np.full((kv_heads, max_seq, head_dim), np.nan, dtype=np.float32)
    vc = np.full_like(kc, np.nan)
    kc[:, :prefix] = rng.standard_normal((kv_heads, prefix, head_dim)).astype(np.float32)
    vc[:, :prefix] = rng.standard_normal((kv_heads, prefix, head_dim)).astype(np.float32)
    kd, vd = torch.from_numpy(kc.copy()).cuda(), torch.from_numpy(vc.copy()).cuda()
    for pos in range(prefix, prefix + 2):
        h = rng.standard_normal(hidden).astype(np.float32)
        hd = torch.from_numpy(h.copy()).cuda()
        oracle.layer_decode(h, layer, kc, vc, heads, kv_heads, head_dim, pos, 1e-6, 10000.0, 1.0, 2)
        hip.TransformerLayerDecode(hd, dev["attn_norm"], dev["qkv"], dev["q_norm"], dev["k_norm"], dev["o"], dev["ffn_norm"],
                                   dev["gate_up"], dev["down"], kd, vd, heads, kv_heads, head_dim, pos, 1e-6, 10000.0, 1.0, 2)
        torch.cuda.synchronize()
        assert rel(hd.cpu().numpy(), h) <= 3e-3, (pos, rel(hd.cpu().numpy(), h))
        assert rel(kd.cpu().numpy()[:, pos], kc[:, pos]) <= 1e-5 and rel(vd.cpu().numpy()[:, pos], vc[:, pos]) <= 1e-5


@pytest.mark.parametrize("head_dim,group,kv_heads,prefix", [(128, 3, 8, 1600), (128, 5, 8, 1600), (128, 6, 8, 1407), (128, 7, 4, 6200),
                                                            (64, 7, 8, 1600), (80, 3, 8, 1600), (96, 5, 8, 1600), (192, 6, 8, 1600), (192, 3, 8, 1600), (256, 5, 8, 1600)])
def test_a_group_of_heads_that_leaves_places_of_its_workgroup_over(hip, oracle, head_dim, group, kv_heads, prefix):
    """3, 5, 6 and 7 query heads of a KV head in a workgroup of 4 or 8, once there are 184 workgroups (1408 -> 1409 positions
    with 8 KV heads); two and four cache rows per group of lanes."""
    test_attention_rows_per_group_at_their_borders(hip, oracle, head_dim, group, kv_heads, prefix)


def to_host_layer(layer, QuantizedWeight, dims):
    d = {k: (None if layer[k] is None else np.ascontiguousarray(layer[k])) for k in ("attn_norm", "q_norm", "k_norm", "ffn_norm")}
    for k, (ne0, ne1) in dims.items():
        d[k] = QuantizedWeight(np.ascontiguousarray(layer[k][1]), layer[k][0], ne0, ne1)
    return d


def test_host_pointer_layer_decode_keeps_the_kv_cache_on_the_device(hip, oracle):
    # the bridge's own argument list: host arrays throughout; the caches come back with SyncHostBuffer
    from tensorsharp_amd import QuantizedWeight
    rng = np.random.default_rng(113)
    hidden, heads, kv_heads, head_dim, inter, max_seq, prefix = 512, 8, 2, 64, 1024, 160, 150
    layer, dims = make_layer(oracle, rng, hidden, heads, kv_heads, head_dim, inter, (Q4_K, Q8_0, Q4_K, Q4_K))
    host = to_host_layer(layer, QuantizedWeight, dims)
    kc = np.zeros((kv_heads, max_seq, head_dim), dtype=np.float32)
    vc = np.zeros_like(kc)
    kc[:, :prefix] = rng.standard_normal((kv_heads, prefix, head_dim)).astype(np.float32)
    vc[:, :prefix] = rng.standard_normal((kv_heads, prefix, head_dim)).astype(np.float32)
    kh, vh = kc.copy(), vc.copy()
    step = lambda h, pos: hip.TransformerLayerDecode(h, host["attn_norm"], host["qkv"], host["q_norm"], host["k_norm"], host["o"],
                                                     host["ffn_norm"], host["gate_up"], host["down"], kh, vh, heads, kv_heads, head_dim,
                                                     pos, 1e-6, 10000.0, 1.0, 2)
    try:
        for pos in range(prefix, prefix + 3):
            h = rng.standard_normal(hidden).astype(np.float32)
            got = h.copy()
            oracle.layer_decode(h, layer, kc, vc, heads, kv_heads, head_dim, pos, 1e-6, 10000.0, 1.0, 2)
            step(got, pos)
            assert rel(got, h) <= 3e-3, (pos, rel(got, h))
        # the host arrays were not written by the calls; the device copies hold the three new rows
        assert not kh[:, prefix:].any() and not vh[:, prefix:].any()
        hip.SyncHostBuffer(kh)
        hip.SyncHostBuffer(vh)
        assert np.array_equal(kh[:, :prefix], kc[:, :prefix]) and not kh[:, prefix + 3:].any()
        assert rel(kh[:, prefix:prefix + 3], kc[:, prefix:prefix + 3]) <= 3e-3
        assert rel(vh[:, prefix:prefix + 3], vc[:, prefix:prefix + 3]) <= 3e-3
        # a caller that rewinds the cache on the host: invalidate, and the next call reads the host bytes again
        kh[:, prefix:] = 0
        vh[:, prefix:] = 0
        kc[:, prefix:] = 0
        vc[:, prefix:] = 0
        hip.InvalidateHostBuffer(kh.ctypes.data)
        hip.InvalidateHostBuffer(vh.ctypes.data)
        h = rng.standard_normal(hidden).astype(np.float32)
        got = h.copy()
        oracle.layer_decode(h, layer, kc, vc, heads, kv_heads, head_dim, prefix, 1e-6, 10000.0, 1.0, 2)
        step(got, prefix)
        assert rel(got, h) <= 3e-3
        with pytest.raises(RuntimeError, match="position outside the KV cache"):
            step(got, max_seq)
    finally:
        hip.ClearHostBufferCache()


def test_host_pointer_model_decode_equals_the_device_form(hip, oracle):
    import torch
    from tensorsharp_amd import QuantizedWeight
    rng = np.random.default_rng(127)
    hidden, heads, kv_heads, head_dim, inter, max_seq = 512, 4, 2, 128, 768, 6
    hosts, devs = [], []
    for li in range(3):
        layer, dims = make_layer(oracle, rng, hidden, heads, kv_heads, head_dim, inter, (Q8_0, Q8_0, Q8_0, Q8_0), qk_norm=False)
        hl = to_host_layer(layer, QuantizedWeight, dims)
        hl["k_cache"] = np.zeros((kv_heads, max_seq, head_dim), np.float32)
        hl["v_cache"] = np.zeros_like(hl["k_cache"])
        hosts.append(hl)
        d = to_device_layer(layer, torch, QuantizedWeight, dims)
        d["k_cache"] = torch.zeros((kv_heads, max_seq, head_dim), dtype=torch.float32, device="cuda")
        d["v_cache"] = torch.zeros_like(d["k_cache"])
        devs.append(d)
    try:
        for pos in range(3):
            h = rng.standard_normal(hidden).astype(np.float32)
            hd = torch.from_numpy(h.copy()).cuda()
            hip.TransformerModelDecode(h, hosts, heads, kv_heads, head_dim, pos, 1e-5, 1e6, 1.0, 0)
            hip.TransformerModelDecode(hd, devs, heads, kv_heads, head_dim, pos, 1e-5, 1e6, 1.0, 0)
            torch.cuda.synchronize()
            assert np.array_equal(h, hd.cpu().numpy()), pos          # same kernels, same launch shapes: same bits
        for hl, d in zip(hosts, devs):
            hip.SyncHostBuffer(hl["k_cache"])
            hip.SyncHostBuffer(hl["v_cache"])
            assert np.array_equal(hl["k_cache"], d["k_cache"].cpu().numpy()) and np.array_equal(hl["v_cache"], d["v_cache"].cpu().numpy())
    finally:
        hip.ClearHostBufferCache()


@pytest.mark.parametrize("prefix", [0, 5, 70, 517])
def test_unwritten_cache_rows_may_hold_nan(hip, oracle, prefix):
    """Cache rows at and beyond `position` are not part of the attention (ggml_flash_attn_ext skips masked positions): whatever
    their memory holds - NaN bits from an uninitialised allocation - must not reach the result.  One split (short prefix),
    a ragged last split and several splits."""
    import torch
    from tensorsharp_amd import QuantizedWeight
    rng = np.random.default_rng(777 + prefix)
    hidden, heads, kv_heads, head_dim, inter, max_seq = 256, 4, 2, 64, 512, 640
    layer, dims = make_layer(oracle, rng, hidden, heads, kv_heads, head_dim, inter, (Q8_0, Q8_0, Q8_0, Q8_0), True)
    dev = to_device_layer(layer, torch, QuantizedWeight, dims)
    kc = np.zeros((kv_heads, max_seq, head_dim), dtype=np.float32)
    vc = np.zeros_like(kc)
    kc[:, :prefix] = rng.standard_normal((kv_heads, prefix, head_dim)).astype(np.float32)
    vc[:, :prefix] = rng.standard_normal((kv_heads, prefix, head_dim)).astype(np.float32)
    kn, vn = kc.copy(), vc.copy()
    kn[:, prefix:] = np.nan
    vn[:, prefix:] = np.nan
    kd, vd = torch.from_numpy(kn).cuda(), torch.from_numpy(vn).cuda()
    for pos in range(prefix, prefix + 2):
        h = rng.standard_normal(hidden).astype(np.float32)
        hd = torch.from_numpy(h.copy()).cuda()
        oracle.layer_decode(h, layer, kc, vc, heads, kv_heads, head_dim, pos, 1e-6, 10000.0, 1.0, 2)
        hip.TransformerLayerDecode(hd, dev["attn_norm"], dev["qkv"], dev["q_norm"], dev["k_norm"], dev["o"], dev["ffn_norm"],
                                   dev["gate_up"], dev["down"], kd, vd, heads, kv_heads, head_dim, pos, 1e-6, 10000.0, 1.0, 2)
        torch.cuda.synchronize()
        got = hd.cpu().numpy()
        assert np.all(np.isfinite(got)), pos
        assert rel(got, h) <= 3e-3, (pos, rel(got, h))
    assert np.all(np.isnan(kd.cpu().numpy()[:, prefix + 2:]))              # rows past the written ones untouched


def test_layer_decode_replayed_from_a_hip_graph(hip, oracle):
    # After one call on a stream the layer call allocates nothing (its scratch is the stream's grow-only buffer) and
    # records no memset, so its six launches can be captured on that stream and replayed.  Every replay is checked
    # against the eager result, with eager work and synchronisations of the program's own between the replays.
    import torch
    from tensorsharp_amd import QuantizedWeight
    rng = np.random.default_rng(131)
    hidden, heads, kv_heads, head_dim, inter, max_seq = 512, 8, 2, 64, 1024, 256
    layer, dims = make_layer(oracle, rng, hidden, heads, kv_heads, head_dim, inter, (Q4_K, Q4_K, Q4_K, Q4_K))
    dev = to_device_layer(layer, torch, QuantizedWeight, dims)
    pos = 140
    k0 = torch.randn((kv_heads, max_seq, head_dim), device="cuda")
    v0 = torch.randn((kv_heads, max_seq, head_dim), device="cuda")
    h0 = torch.randn(hidden, device="cuda")
    hd, kd, vd = h0.clone(), k0.clone(), v0.clone()

    def call():
        hip.TransformerLayerDecode(hd, dev["attn_norm"], dev["qkv"], dev["q_norm"], dev["k_norm"], dev["o"], dev["ffn_norm"],
                                   dev["gate_up"], dev["down"], kd, vd, heads, kv_heads, head_dim, pos, 1e-6, 10000.0, 1.0, 2)

    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        call()                                   # eager: sizes this stream's scratch, gives the expected result
    side.synchronize()
    want_h, want_k, want_v = hd.clone(), kd[:, pos].clone(), vd[:, pos].clone()
    graph = torch.cuda.CUDAGraph()
    hd.copy_(h0)
    torch.cuda.synchronize()
    with torch.cuda.graph(graph, stream=side):
        call()
    for rep in range(4):
        hd.copy_(h0)
        kd.copy_(k0)
        vd.copy_(v0)
        # unrelated eager work of the same library on the default stream between replays
        y = torch.empty((1, hidden), device="cuda")
        hip.AddmmQuantDevice(y, h0.view(1, -1) * float(rep + 1), dev["o"].ptr, Q4_K, hidden, hidden, dev["o"].raw_bytes)
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(hd, want_h), rep
        assert torch.equal(kd[:, pos], want_k) and torch.equal(vd[:, pos], want_v), rep
