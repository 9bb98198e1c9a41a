"""GPU parity: every prefill kernel that serves plain Q4_K, Q8_0 and Q6_K products, each at a ragged shape that the library plans
for it - the plan (TSHip_MatmulPlanDevice) is asserted, so a shape that drifts to another kernel fails its test instead of
testing that one.

Bar: the matmul bar of test_gpu_gemm.py (fp16 operands, fp32 sums) on sampled rows - tile edges and seeded random ones - against
the fp64 product of the dequantized weights.
"""
import numpy as np
import pytest

from oracle.oracle import Q4_K, Q6_K, Q8_0
from test_gpu_gemm import check, sample_rows
from test_matmul_plan import REGISTERS, TILES, WIDE, plan

pytestmark = pytest.mark.gpu
T = {"q4_k": Q4_K, "q8_0": Q8_0, "q6_k": Q6_K}
SCALE = {"q4_k": (256, 144, 0), "q8_0": (32, 34, 0), "q6_k": (256, 210, 208)}      # block: weights, bytes, where its fp16 d is
SCRATCH = 64 << 20                                                              # of the entry point that allocates nothing


def operands(name, M, N, K):
    import torch
    from tensorsharp_amd import synth
    w = synth.random_weight(T[name], N, K, torch.device("cuda"), seed=M + N + K)
    x = np.random.default_rng(M + 3 * N + K).standard_normal((M, K)).astype(np.float32)
    return w, x, sample_rows(M, [0, 1, 31, 32, 63, 64, 95, 96, 127, 128, 255, 256, M - 2, M - 1], min(40, M), M)


def weight(name, w, N, K):
    from tensorsharp_amd import QuantizedWeight
    return QuantizedWeight(w, T[name], K, N)


# (format, kernel, rows per tile, K in chunks, rows, columns, K): M and N ragged in the last tile; K of Q8_0 an odd number of blocks
# (the last k-tile holds one) and, chunked, an odd number of k-tiles; every K has several granules
PLAIN = [
    ("q4_k", WIDE, 32, False, 521, 485, 768), ("q4_k", WIDE, 32, True, 45, 487, 2304), ("q4_k", WIDE, 64, False, 1348, 1287, 768),
    ("q4_k", WIDE, 64, True, 899, 551, 1280), ("q4_k", WIDE, 96, False, 1795, 2051, 768), ("q4_k", WIDE, 96, True, 907, 517, 2816),
    ("q4_k", WIDE, 128, False, 1834, 3115, 768), ("q4_k", WIDE, 128, True, 971, 513, 4096),
    ("q4_k", TILES, 256, False, 1537, 4965, 768), ("q4_k", TILES, 256, True, 1800, 2079, 5120),
    ("q8_0", WIDE, 32, False, 949, 1093, 1056), ("q8_0", WIDE, 32, True, 321, 387, 2080), ("q8_0", WIDE, 64, False, 1157, 1561, 800),
    ("q8_0", WIDE, 64, True, 806, 291, 2080), ("q8_0", WIDE, 96, False, 1809, 2127, 800), ("q8_0", WIDE, 96, True, 770, 777, 2080),
    ("q8_0", WIDE, 128, False, 1825, 3143, 1568), ("q8_0", WIDE, 128, True, 1350, 515, 2592),
    ("q8_0", TILES, 128, False, 1967, 2617, 800), ("q8_0", TILES, 128, True, 1634, 1033, 2080),
    ("q8_0", TILES, 256, False, 1544, 4913, 800), ("q8_0", TILES, 256, True, 1795, 2113, 4128),
    ("q6_k", WIDE, 32, False, 1025, 1219, 768), ("q6_k", WIDE, 32, True, 519, 711, 2304), ("q6_k", WIDE, 64, False, 1346, 1299, 768),
    ("q6_k", WIDE, 64, True, 578, 835, 2304), ("q6_k", WIDE, 96, False, 1798, 2079, 1024), ("q6_k", WIDE, 96, True, 785, 803, 2304),
    ("q6_k", WIDE, 128, True, 1168, 783, 2304), ("q6_k", TILES, 128, False, 1798, 2053, 768), ("q6_k", TILES, 128, True, 1563, 769, 2304),
    ("q4_k", REGISTERS, 32, True, 21, 1001, 4352), ("q8_0", REGISTERS, 32, True, 45, 1001, 2080), ("q6_k", REGISTERS, 32, True, 35, 1001, 2304),
    # workgroups whose run of 32-column units crosses into the next 32 rows
    ("q4_k", REGISTERS, 32, False, 60, 9001, 768), ("q8_0", REGISTERS, 32, False, 70, 4501, 1312), ("q6_k", REGISTERS, 32, False, 70, 4501, 1280),
]
ADDED = [
    ("q4_k", WIDE, 32, False, 1038, 783, 768), ("q4_k", WIDE, 32, True, 77, 487, 4352), ("q4_k", WIDE, 64, False, 1414, 1533, 768),
    ("q4_k", WIDE, 64, True, 897, 517, 1280), ("q4_k", WIDE, 96, False, 1795, 2051, 768), ("q4_k", WIDE, 96, True, 1794, 525, 1280),
    ("q4_k", WIDE, 128, False, 1834, 3115, 768), ("q4_k", WIDE, 128, True, 971, 513, 4096),
    ("q4_k", TILES, 256, False, 1928, 6157, 768), ("q4_k", TILES, 256, True, 1613, 2315, 2048),
    ("q8_0", WIDE, 32, False, 799, 2517, 1056), ("q8_0", WIDE, 32, True, 517, 487, 1056), ("q8_0", WIDE, 64, False, 1545, 2329, 1056),
    ("q8_0", WIDE, 64, True, 913, 549, 1056), ("q8_0", WIDE, 96, True, 1352, 769, 1056), ("q8_0", WIDE, 128, True, 1183, 1031, 1568),
    ("q8_0", TILES, 128, False, 1545, 2351, 800), ("q8_0", TILES, 128, True, 1634, 1033, 2080),
    ("q8_0", TILES, 256, False, 1544, 4913, 800), ("q8_0", TILES, 256, True, 1561, 2321, 2080),
    ("q6_k", WIDE, 32, False, 1620, 1015, 768), ("q6_k", WIDE, 32, True, 801, 941, 1024), ("q6_k", WIDE, 64, False, 1546, 2363, 1280),
    ("q6_k", WIDE, 64, True, 833, 1185, 768), ("q6_k", WIDE, 96, True, 785, 803, 2304), ("q6_k", WIDE, 128, True, 1168, 783, 2304),
    ("q6_k", TILES, 128, False, 1752, 1551, 768), ("q6_k", TILES, 128, True, 1563, 769, 2304),
    ("q4_k", REGISTERS, 32, False, 37, 1001, 768), ("q8_0", REGISTERS, 32, False, 45, 1001, 1056), ("q6_k", REGISTERS, 32, True, 35, 1001, 2304),
]
# a scratch of 64 MiB: some of the K chunks, or another kernel than the one planned without a bound
BOUNDED = [("q4_k", WIDE, WIDE, 1843, 499, 10240), ("q4_k", REGISTERS, WIDE, 2690, 85, 12032), ("q4_k", TILES, WIDE, 2445, 1025, 6144),
           ("q8_0", WIDE, WIDE, 2279, 499, 7936), ("q8_0", REGISTERS, WIDE, 1973, 105, 15360), ("q8_0", TILES, WIDE, 2573, 1149, 4096),
           ("q8_0", TILES, WIDE, 2820, 1571, 3840), ("q6_k", WIDE, TILES, 2053, 737, 9472), ("q6_k", REGISTERS, WIDE, 2315, 283, 11520),
           ("q6_k", TILES, WIDE, 2437, 757, 7936)]


@pytest.mark.parametrize("name,kernel,tile,chunked,M,N,K", PLAIN)
def test_product(hip, oracle, name, kernel, tile, chunked, M, N, K):
    import torch
    got = plan(T[name], M, N, K)
    assert got[:2] == (kernel, tile) and (got[2] > 1) == chunked, got
    w, x, rows = operands(name, M, N, K)
    xd = torch.from_numpy(x).cuda()
    y = hip.LinearForward(xd, weight(name, w, N, K)).cpu().numpy()
    check(y[rows], oracle.matmul_f64(T[name], w.cpu().numpy().reshape(-1), N, K, x[rows]), got)
    assert np.isfinite(y).all()
    # a scale outside the fp16 operands in the last block of the last column: that column is NaN, nothing else changes
    per, size, at = SCALE[name]
    bad = w.reshape(-1).view(torch.uint8).clone()
    end = ((N - 1) * (K // per) + K // per - 1) * size + at
    bad[end:end + 2] = torch.from_numpy(np.frombuffer(np.float16(1.0).tobytes(), np.uint8).copy()).cuda()
    z = hip.LinearForward(xd, weight(name, bad, N, K)).cpu().numpy()
    assert np.isnan(z[:, N - 1]).all()
    assert np.array_equal(z[:, :N - 1], y[:, :N - 1])


@pytest.mark.parametrize("name,kernel,tile,chunked,M,N,K", ADDED)
def test_product_added_to_a_residual(hip, oracle, name, kernel, tile, chunked, M, N, K):
    import torch
    got = plan(T[name], M, N, K, 1)
    assert got[:2] == (kernel, tile) and (got[2] > 1) == chunked, got
    w, x, rows = operands(name, M, N, K)
    residual = np.random.default_rng(N).standard_normal((M, N)).astype(np.float32)
    r = torch.from_numpy(residual).cuda()
    hip.UseCurrentStream()
    hip.FusedMatMulQuantAdd(r, torch.from_numpy(x).cuda(), weight(name, w, N, K))
    torch.cuda.synchronize()
    ref = oracle.matmul_f64(T[name], w.cpu().numpy().reshape(-1), N, K, x[rows])
    # (the product by itself: the residual would hide its error in the norm; one more fp32 rounding of the sum is 6e-8 of it)
    check(r.cpu().numpy()[rows].astype(np.float64) - residual[rows], ref, got)


@pytest.mark.parametrize("name,free,bounded,M,N,K", BOUNDED)
def test_product_with_a_bounded_scratch(hip, oracle, name, free, bounded, M, N, K):
    import torch
    got = plan(T[name], M, N, K, 0, SCRATCH)
    assert plan(T[name], M, N, K)[0] == free and plan(T[name], M, N, K)[3] > SCRATCH
    assert got[0] == bounded and got[3] <= SCRATCH, got
    w, x, rows = operands(name, M, N, K)
    y = torch.full((M, N), float("nan"), dtype=torch.float32, device="cuda")
    flat = w.reshape(-1).view(torch.uint8)
    hip.UseCurrentStream()
    hip.AddmmQuantDeviceNoAlloc(y, torch.from_numpy(x).cuda(), flat.data_ptr(), T[name], K, N, flat.numel())
    torch.cuda.synchronize()
    y = y.cpu().numpy()
    assert np.isfinite(y).all()
    check(y[rows], oracle.matmul_f64(T[name], w.cpu().numpy().reshape(-1), N, K, x[rows]), got)


@pytest.mark.parametrize("name,kernel,M,N,K", [("q8_0", WIDE, 321, 387, 2080), ("q8_0", TILES, 1634, 1033, 2080), ("q6_k", WIDE, 519, 711, 2304),
                                               ("q6_k", TILES, 1563, 769, 2304)])
def test_weight_view_that_begins_inside_a_16_byte_piece(hip, oracle, name, kernel, M, N, K):
    # a view from row 1 (rows of 2210 and 1890 bytes: it begins two bytes into a piece)
    import torch
    w, x, rows = operands(name, M, N + 1, K)
    per, size, _ = SCALE[name]
    view = w.reshape(-1).view(torch.uint8)[K // per * size:]
    assert view.data_ptr() % 16 == 2 and plan(T[name], M, N, K)[0] == kernel
    y = hip.LinearForward(torch.from_numpy(x).cuda(), weight(name, view, N, K)).cpu().numpy()
    check(y[rows], oracle.matmul_f64(T[name], view.cpu().numpy(), N, K, x[rows]), name)
