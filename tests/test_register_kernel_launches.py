"""Which register-resident kernels the shapes of the GPU tests launch: CPU tests on a HIP runtime without a device (see test_launches.py)."""
import re

import pytest

from test_gpu_expert_register_tiles import STAGES, TYPES
from test_gpu_register_kernel import FORMATS, SHAPES
from test_launches import stub  # noqa: F401

BYTES = {2: 18, 3: 20, 6: 22, 7: 24, 8: 34, 12: 144, 13: 176, 14: 210, 20: 18, 39: 17}
PRODUCT = """
for t, per, size, M, N_, K in cases:
    w, x, y = space(N_ * (K // per) * size), space(M * K * 4).view(np.float32), space(M * N_ * 4).view(np.float32)
    assert L.TSHip_AddmmQuantF32Device(view(y, M, N_), view(x, M, K), w.ctypes.data, t, K, N_, w.size), L.TSHip_GetLastError()
    out.append(log())
"""
STAGE = """
for t, per, size, E, H, F, T, k in cases:
    gu, dn, few = space(E * 2 * F * (H // per) * size), space(E * H * (F // per) * size), space(T * k * 4)
    x = space(T * H * 4).view(np.float32)
    assert L.TSHip_MoEExpertsGptOssForwardF32Device(view(x, T, H), view(x, T, H), few.ctypes.data, few.ctypes.data, k, gu.ctypes.data, None,
                                                    dn.ctypes.data, None, t, E, H, F, 1.702, 7.0), L.TSHip_GetLastError()
    out.append(log())
"""


def kernels(log):
    """(columns of a tile, k-tiles per wavefront, rows of a tile) of the register-resident kernels launched"""
    found = [re.search(r"gemm_slim(32)?_kernelINS0_.*?(?:Li(\d+))(?:ELi(\d+))?EEEvNS0_8GemmArgs", l[1]) for l in log if l[0] == "launch"]
    return [(32, int(m[2]), 32) if m[1] else (16, int(m[2]), 16 * int(m[3])) for m in found if m]


@pytest.mark.parametrize("name", sorted(FORMATS))
def test_every_kernel_is_launched(stub, name):  # noqa: F811
    t, per = FORMATS[name]
    cases = [(t, per, BYTES[t], M, N, 256 * blocks - (32 if per == 32 else 0)) for M, N, blocks in SHAPES]
    logs = stub(PRODUCT, cases=cases)
    seen = {k for log in logs for k in kernels(log)}
    if per == 256:
        expected = {(16, 4, 16), (16, 8, 16), (16, 8, 32), (32, 4, 32)} | ({(32, 8, 32)} if name == "q4_k" else set())
    else:
        # (two raw buffers of 32 rows fit LDS with four k-tiles of Q8_0, six of the formats above 18 bytes a block, eight of the others)
        wide = {"q8_0": (2, 4), "q4_1": (2, 4, 6), "q5_0": (2, 4, 6), "q5_1": (2, 4, 6)}.get(name, (2, 4, 6, 8))
        expected = {(16, k, 16) for k in (2, 4, 6, 8)} | {(16, k, 32) for k in (6, 8)} | {(32, k, 32) for k in wide}
    assert seen == expected, (sorted(seen - expected), sorted(expected - seen))
    # runs that cross into another K chunk, or other rows, on tiles of 16 columns
    crossing = set()
    for (_, _, _, M, N, K), log in zip(cases, logs):
        for columns, ktw, rows in kernels(log):
            chunks, tiles = -(-K // 64 // (8 * ktw)), -(-N // 16)
            if columns == 16 and -(-M // rows) * chunks * tiles > 256:
                crossing |= ({"chunk"} if chunks > 1 else set()) | ({"rows"} if M > rows else set())
    assert "chunk" in crossing and ("rows" in crossing or name in ("q4_k", "q8_0")), crossing


def test_expert_stages_launch_the_kernels_they_are_for(stub):  # noqa: F811
    cases = [(TYPES[n], 32 if n in ("q8_0", "q4_0") else 256, BYTES[TYPES[n]], E, H, F, T, k) for n, E, H, F, T, k in STAGES]
    seen = {n[0]: set() for n in STAGES}
    for n, log in zip(STAGES, stub(STAGE, cases=cases)):
        got = kernels(log)
        assert len(got) == 2, (n, log)
        seen[n[0]] |= set(got)
    for name in ("q4_k", "q5_k", "q6_k", "q8_0"):
        assert (16, 8, 32) in seen[name] and any(k[0] == 32 for k in seen[name])
    assert (16, 6, 32) in seen["q8_0"] & seen["q4_0"]


@pytest.mark.parametrize("name,M,N,K,columns", [
    ("q4_k", 40, 2340, 5120, 16), ("q4_k", 53, 2195, 5120, 16), ("q4_k", 24, 4096, 4096, 16), ("q8_0", 24, 4096, 2560, 16), ("q8_0", 108, 1024, 6080, 16),
    ("q4_k", 24, 14336, 4096, 32), ("q4_k", 29, 4096, 14336, 32), ("q6_k", 23, 5120, 6144, 32), ("mxfp4", 26, 4096, 14336, 32), ("q8_0", 21, 5120, 14848, 32)])
def test_the_faster_kernel_is_launched(stub, name, M, N, K, columns):  # noqa: F811
    """Calls that take 4 to 25 % longer on the other one."""
    t, per = FORMATS[name]
    (log,) = stub(PRODUCT, cases=[(t, per, BYTES[t], M, N, K)])
    assert [k[0] for k in kernels(log)] == [columns], log
