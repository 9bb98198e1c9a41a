"""GPU parity of the register-resident kernels (tiles of 16 columns and 16 or 32 rows, or of 32 columns; K dealt out to eight wavefronts
block by block) where their edges are: one row tile of 16 rows and the first of 32, a ragged last tile of columns, K whose blocks do not
divide by eight, fewer blocks than wavefronts, K in a full and a short chunk, and runs of units that cross into the next 32 rows or the
next chunk.  test_register_kernel_launches.py: every kernel of them is launched here.

Bar: the matmul bar of test_gpu_gemm.py (fp16 operands, fp32 sums) against the fp64 product of the dequantized weights.
"""
import numpy as np
import pytest

from test_gpu_gemm import check
from test_matmul_plan import REGISTERS, plan

pytestmark = pytest.mark.gpu
FORMATS = {"q4_0": (2, 32), "q4_1": (3, 32), "q5_0": (6, 32), "q5_1": (7, 32), "q8_0": (8, 32), "q4_k": (12, 256), "q5_k": (13, 256),
           "q6_k": (14, 256), "iq4_nl": (20, 32), "mxfp4": (39, 32)}
# rows, columns, K in units of 256 (formats of 32-weight blocks: 32 less, an odd number of blocks)
SHAPES = [(4, 64, 1), (16, 65, 3), (17, 4097, 9), (32, 79, 16), (33, 1041, 17), (16, 300, 18), (24, 4100, 23), (61, 1027, 33),
          (7, 129, 10), (12, 200, 16), (20, 70, 3), (40, 200, 8), (40, 200, 11), (5, 333, 7), (9, 1500, 12), (30, 640, 12), (9, 4100, 17),
          (16, 6200, 28), (40, 2100, 9), (70, 2100, 15), (40, 2100, 17)]


@pytest.mark.parametrize("name", sorted(FORMATS))
@pytest.mark.parametrize("M,N,blocks", SHAPES)
def test_product(hip, oracle, name, M, N, blocks):
    import torch
    from tensorsharp_amd import QuantizedWeight, synth
    t, per = FORMATS[name]
    K = 256 * blocks - (32 if per == 32 else 0)
    got = plan(t, M, N, K)
    if name not in ("q4_k", "q8_0", "q6_k") or M <= 16:                     # (the others may go to gemm_wide_kernel)
        assert got[:2] == (REGISTERS, 32), got
    w = synth.random_weight(t, N, K, torch.device("cuda"), seed=M + N + K)
    x = np.random.default_rng(M + 3 * N + K).standard_normal((M, K)).astype(np.float32)
    y = hip.LinearForward(torch.from_numpy(x).cuda(), QuantizedWeight(w, t, K, N)).cpu().numpy()
    check(y, oracle.matmul_f64(t, w.cpu().numpy().reshape(-1), N, K, x), got)


@pytest.mark.parametrize("name", ["q4_0", "q8_0", "q4_k", "q6_k"])
@pytest.mark.parametrize("M", [16, 32])
@pytest.mark.parametrize("where", [0, 8, -1])
def test_a_scale_out_of_range_marks_its_column_only(hip, oracle, name, M, where):
    # block `where` of column 37 (another lane group and wavefront each): every row of that column is NaN, nothing else changes
    import torch
    from tensorsharp_amd import QuantizedWeight, synth
    t, per = FORMATS[name]
    size, at, N, K = {"q4_0": (18, 0), "q8_0": (34, 0), "q4_k": (144, 0), "q6_k": (210, 208)}[name] + (83, 2304)
    w = synth.random_weight(t, N, K, torch.device("cuda"), seed=M)
    x = torch.randn((M, K), generator=torch.Generator().manual_seed(M)).cuda()
    y = hip.LinearForward(x, QuantizedWeight(w, t, K, N)).cpu().numpy()
    bad = w.reshape(-1).view(torch.uint8).clone()
    begin = (37 * (K // per) + where % (K // per)) * size + at
    bad[begin:begin + 2] = torch.from_numpy(np.frombuffer(np.float16(60.0).tobytes(), np.uint8).copy()).cuda()
    z = hip.LinearForward(x, QuantizedWeight(bad, t, K, N)).cpu().numpy()
    assert np.isfinite(y).all() and np.isnan(z[:, 37]).all()
    assert np.array_equal(np.delete(z, 37, 1), np.delete(y, 37, 1))


@pytest.mark.parametrize("M,N", [(4, 5760), (9, 2880), (16, 2880), (16, 5760), (30, 1440)])
@pytest.mark.parametrize("K", [2880, 1760])
@pytest.mark.parametrize("begin", [0, 1, 3])
def test_mxfp4_rows_that_begin_at_any_byte(hip, oracle, M, N, K, begin):
    # blocks of 17 bytes: the weight and its rows begin at any address; 2880 is the width of GPT-OSS (45 k-tiles, an odd number)
    import torch
    from tensorsharp_amd import QuantizedWeight, synth
    assert plan(39, M, N, K)[:3] == (REGISTERS, 32, 1)
    w = synth.random_weight(39, N, K, torch.device("cuda"), seed=M + N).reshape(-1)
    room = torch.zeros(w.numel() + 64, dtype=torch.uint8, device="cuda")
    view = room[16 + begin:16 + begin + w.numel()]
    view.copy_(w)
    assert view.data_ptr() % 4 == begin
    x = np.random.default_rng(M + N).standard_normal((M, K)).astype(np.float32)
    y = hip.LinearForward(torch.from_numpy(x).cuda(), QuantizedWeight(view, 39, K, N)).cpu().numpy()
    check(y, oracle.matmul_f64(39, w.cpu().numpy(), N, K, x), (M, N, K, begin))
