"""Which fused output projections and FFNs leave the projection's K-chunk sums to the conversion in front of the FFN: CPU tests on a HIP
runtime without a device (see test_launches.py)."""
import pytest

from test_gpu_outproj_ffn_sums import REFUSED, ROWS, SHAPES, T
from test_launches import launches, stub  # noqa: F401

BLOCKS = {"q4_0": (32, 18), "q5_0": (32, 22), "q8_0": (32, 34), "q4_k": (256, 144), "q5_k": (256, 176), "q6_k": (256, 210), "iq4_nl": (32, 18), "mxfp4": (32, 17)}
CALL = """
for rows, out_type, gu_type, hidden, ins, half, pad in cases:
    weight = lambda t, n, k: (types[t], k, n, n * (k // blocks[t][0]) * blocks[t][1])
    data = space(max(weight(out_type, hidden, ins)[3], weight(gu_type, 2 * half, hidden)[3], weight("q8_0", hidden, half)[3], 4 * hidden))
    r, x = space(4 * rows * (hidden + pad)).view(np.float32), space(4 * rows * ins).view(np.float32)
    p = C.c_void_p(data.ctypes.data)
    ok = L.TSHip_FusedOutProjFFNQuantF32Device(view(r, rows, hidden, hidden + pad), view(x, rows, ins), p, *weight(out_type, hidden, ins), p, hidden, 1e-6,
                                               p, *weight(gu_type, 2 * half, hidden), p, *weight("q8_0", hidden, half), half)
    assert ok, L.TSHip_GetLastError()
    out.append(log())
"""


def left(log):
    """threads of the conversion that adds chunk sums (the kernel's last template argument is 3), if one was launched"""
    got = [l for l in log if l[0] == "launch" and "convert_x_kernel" in l[1] and "Li3EEE" in l[1]]
    return [1024 if "Li1024ELi3EEE" in l[1] else 256 for l in got]


@pytest.mark.parametrize("shape", SHAPES)
def test_the_sums_are_left(stub, shape):  # noqa: F811
    for rows, log in zip(ROWS, stub(CALL, cases=[(rows, *shape) for rows in ROWS], types=T, blocks=BLOCKS)):
        if (rows, *shape[:2]) == (200, "q4_k", "q5_k"):                              # (seven chunks, more than the gate / up rows take)
            assert left(log) == []
        else:
            assert left(log) == [1024 if shape[2] > 2048 else 256], (rows, log)


@pytest.mark.parametrize("shape", REFUSED)
def test_the_sums_are_not_left(stub, shape):  # noqa: F811
    rows = [4, 200, 333] if shape[1] != "mxfp4" else [200, 333]             # (few rows of MXFP4: no pairs)
    for log in stub(CALL, cases=[(r, *shape) for r in rows], types=T, blocks=BLOCKS):
        assert left(log) == [], log
