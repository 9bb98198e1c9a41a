"""Which kernels a call launches, and what it does when one of them fails: the library on a HIP runtime without a device
(hip_stub.cpp, preloaded into a process of its own).  CPU tests; nothing is computed."""
import json
import os
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PRELUDE = """
import ctypes as C, json, sys
import numpy as np
sys.path.insert(0, {root!r})
from tensorsharp_amd import hip_native as N
stub = C.CDLL({stub!r})
stub.stub_log.restype = C.c_char_p
N._lib = L = C.CDLL(N.LIB_PATH)
for name, (res, args) in N.SIGNATURES.items():
    getattr(L, name).restype = res
    getattr(L, name).argtypes = args
def view(a, rows, cols, stride=None):
    s = cols if stride is None else stride
    return N.TensorView2D(a.ctypes.data, rows, cols, s, 1, ((rows - 1) * s + cols) * 4)
def space(nbytes):
    a = np.zeros(nbytes + 64, dtype=np.uint8)
    return a[-a.ctypes.data % 64:][:nbytes]
def log():
    text = stub.stub_log().decode()
    stub.stub_clear()
    return [l.split() for l in text.splitlines()]
out = []
"""


@pytest.fixture(scope="module")
def stub(tmp_path_factory):
    lib = str(tmp_path_factory.mktemp("stub") / "libhip_stub.so")
    subprocess.run(["g++", "-O1", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", "-Wno-deprecated-declarations",
                    os.path.join(ROOT, "tests", "hip_stub.cpp"), "-o", lib], check=True)

    def run(code, **values):
        text = PRELUDE.format(root=ROOT, stub=lib) + "".join(f"{k} = {v!r}\n" for k, v in values.items()) + code + "\nprint(json.dumps(out))"
        p = subprocess.run([sys.executable, "-c", text], env=dict(os.environ, LD_PRELOAD=lib), capture_output=True, text=True, timeout=300)
        assert p.returncode == 0, p.stderr[-2000:]
        return json.loads(p.stdout.splitlines()[-1])
    return run


def launches(log, name):
    return [l for l in log if l[0] == "launch" and name in l[1]]


HOST_LINEAR = """
x, w, y = np.zeros((M, K), np.float32), space(N_ * K // 256 * 144), np.zeros((M, N_), np.float32)
for n in fails:
    stub.stub_fail_launch(n)
    ok = L.TSHip_AddmmQuantF32(view(y, M, N_), view(x, M, K), w.ctypes.data, 12, K, N_, w.size)
    out.append([ok, log()])
"""


@pytest.mark.parametrize("M,N,K", [(32, 4096, 4096), (2, 512, 4096)])
def test_a_host_linear_that_fails_waits_for_what_it_launched(stub, M, N, K):
    """Kernels read and store the pinned staging memory themselves: after a failed launch the earlier ones have to have ended
    before the next call packs its activations there."""
    for n, (ok, log) in enumerate(stub(HOST_LINEAR, M=M, K=K, N_=N, fails=[0, 2, 1, 2])):
        if n == 0:
            assert ok == 1 and log[-1][0] == "wait"
            continue
        assert ok == 0 and any(l[0] == "failed" for l in log), log
        assert log[-1][0] == "wait", log


@pytest.mark.parametrize("M,N,K,copies", [(64, 4096, 4096, 0), (65, 4096, 4096, 1), (380, 4096, 4096, 1), (400, 4096, 4096, 2), (600, 4096, 4096, 2),
                                          (700, 4096, 256, 0), (800, 4096, 256, 2), (2, 4096, 4096, 1)])
def test_which_way_a_host_linear_takes_over_the_link(stub, M, N, K, copies):
    """Up to 1 MiB of activations are read from pinned memory (not by a GEMV); results are stored to it while both take up to 12 MiB."""
    ((ok, log),) = stub(HOST_LINEAR, M=M, K=K, N_=N, fails=[0])
    assert ok == 1 and sum(l[0] == "copy" for l in log) == copies, log


GEMV_LINEAR = """
for t, per, size, rows, k, norm, add in cases:
    w, x, y = space(rows * (k // per) * size), np.zeros((1, k + 16), np.float32), np.zeros((1, rows), np.float32)
    xv = N.TensorView2D(x.ctypes.data + -x.ctypes.data % 16, 1, k, k, 1, k * 4)
    if norm:
        nw = space(4 * k)
        ok = L.TSHip_FusedRmsNormMatMulQuantF32Device(view(y, 1, rows), xv, nw.ctypes.data, k, 1e-6, w.ctypes.data, t, k, rows, w.size)
    elif add:
        ok = L.TSHip_FusedMatMulQuantAddF32Device(view(y, 1, rows), xv, w.ctypes.data, t, k, rows, w.size)
    else:
        ok = L.TSHip_AddmmQuantF32Device(view(y, 1, rows), xv, w.ctypes.data, t, k, rows, w.size)
    assert ok, L.TSHip_GetLastError()
    out.append(log())
"""
BLOCKS = {"q8_0": (8, 32, 34), "mxfp4": (39, 32, 17), "q4_0": (2, 32, 18), "q4_1": (3, 32, 20), "q5_0": (6, 32, 22), "q5_1": (7, 32, 24), "iq4_nl": (20, 32, 18)}
LONGEST = {"q8_0": 35840}           # of the formats of 80 LDS bytes per block: 65024


@pytest.mark.parametrize("name", BLOCKS)
def test_the_longest_rows_of_a_split_launch_fit_into_lds(stub, name):
    k = LONGEST.get(name, 65024)
    cases = [(*BLOCKS[name], 40, k, norm, 0) for norm in (0, 1)]
    for log in stub(GEMV_LINEAR, cases=cases):
        (split,) = launches(log, "gemv_split_kernel")
        assert int(split[6]) <= 160 * 1024


@pytest.mark.parametrize("name,rows,steps,added", [("q4_1", 1024, 8, 0), ("q4_1", 1024, 9, 1), ("mxfp4", 600, 8, 0), ("q4_0", 2048, 9, 1), ("q8_0", 1024, 6, 1),
                                                    ("q5_0", 1024, 7, 1)])
def test_cheap_blocks_are_split_a_step_later_where_a_residual_is_added(stub, name, rows, steps, added):
    plain, norm, add = stub(GEMV_LINEAR, cases=[(*BLOCKS[name], rows, 512 * steps, n, a) for n, a in ((0, 0), (1, 0), (0, 1))])
    assert len(launches(plain, "gemv_split_kernel")) == len(launches(norm, "gemv_split_kernel")) == 1
    assert len(launches(add, "gemv_split_kernel")) == added


@pytest.mark.parametrize("name,rows,steps,split", [
    ("q8_0", 1024, 6, 1), ("q8_0", 1024, 5, 0), ("q8_0", 2048, 7, 1), ("q8_0", 2048, 6, 0), ("q8_0", 4096, 10, 1), ("q8_0", 4096, 9, 0),
    ("q8_0", 6144, 30, 1), ("q8_0", 6144, 28, 0), ("q8_0", 7172, 42, 0),
    ("q4_0", 1024, 8, 1), ("q4_0", 1024, 7, 0), ("q4_1", 1745, 9, 1), ("q4_1", 1745, 8, 0), ("mxfp4", 1318, 8, 0), ("mxfp4", 3072, 10, 1),
    ("q5_0", 1024, 7, 1), ("iq4_nl", 2048, 8, 1), ("q5_1", 5120, 15, 0),
])
def test_rows_are_split_where_that_was_measured_faster(stub, name, rows, steps, split):
    for norm, add in ((0, 0), (1, 0), (0, 1)):
        if add and (name, rows, steps) == ("q4_0", 1024, 8):
            continue                                                # (above)
        (log,) = stub(GEMV_LINEAR, cases=[(*BLOCKS[name], rows, 512 * steps, norm, add)])
        assert len(launches(log, "gemv_split_kernel")) == split and len(launches(log, "gemv")) == 1, log


LAYER = """
for heads, kv, d, position in cases:
    h, cap = 256, position + 1
    q, n = heads * d, kv * d
    f = lambda m: space(4 * m).ctypes.data_as(C.c_void_p)
    w = lambda rows, k: (space(rows * k // 32 * 34).ctypes.data_as(C.c_void_p), 8, k, rows, rows * k // 32 * 34)
    cache = space(4 * kv * cap * d)
    ok = L.TSHip_TransformerLayerDecodeDevice(f(h), h, f(h), *w(q + 2 * n, h), None, None, d, *w(h, q), f(h), *w(512, h), *w(h, 256),
                                              cache.ctypes.data, cache.ctypes.data, heads, kv, cap, position, 1e-6, 1e4, 1.0, 256, 2)
    assert ok, L.TSHip_GetLastError()
    out.append(log())
"""


@pytest.mark.parametrize("heads,kv,head_dim,position,places,chunks", [
    (40, 8, 128, 6000, 8, 1), (28, 4, 128, 8191, 8, 1), (24, 8, 128, 4000, 4, 1), (12, 2, 192, 32000, 8, 1),       # the rows of a KV head loaded once
    (40, 8, 128, 1000, 1, 5), (24, 4, 256, 2047, 2, 3),                                                            # too few workgroups for that
    (40, 8, 128, 1407, 1, 5), (40, 8, 128, 1408, 8, 1),
    (32, 8, 128, 4000, 4, 1), (64, 8, 128, 4000, 8, 1), (48, 4, 128, 8000, 4, 3), (8, 8, 128, 8000, 1, 1),
])
def test_query_heads_per_attention_workgroup(stub, heads, kv, head_dim, position, places, chunks):
    (log,) = stub(LAYER, cases=[(heads, kv, head_dim, position)])
    (attention,) = launches(log, "attn_decode_kernel")
    assert f"attn_decode_kernelILi{head_dim // 16}ELi{places}E" in attention[1] and int(attention[4]) == chunks, attention


@pytest.mark.parametrize("heads,kv,position,rows", [(32, 32, 2559, 2), (32, 32, 2560, 4), (16, 16, 2048, 2), (32, 8, 2048, 4), (32, 8, 2047, 2),
                                                    (8, 2, 4095, 2), (8, 2, 4096, 4), (32, 32, 63, 2), (32, 32, 64, 4), (32, 32, 128, 2)])
def test_cache_rows_per_group_of_lanes(stub, heads, kv, position, rows):
    (log,) = stub(LAYER, cases=[(heads, kv, 64, position)])
    (attention,) = launches(log, "attn_decode_kernel")
    assert f"ELi{rows}EEEvP" in attention[1], attention


SCRATCH = """
def blocks(rows, k): return space(rows * k // 32 * 34)
x, r, nw = np.zeros((M, H), np.float32), np.zeros((M, H), np.float32), space(4 * H)
plan = (C.c_int64 * 4)()
def workspace(rows, n, k, add):
    assert L.TSHip_MatmulPlanDevice(8, rows, k, n, add, 0, plan)
    return plan[3]
gu, dn = blocks(2 * F, H), blocks(H, F)
x16 = N.TensorView2D(x.ctypes.data & ~15, M, H, H, 1, 4 * M * H)
r16 = N.TensorView2D(r.ctypes.data & ~15, M, H, H, 1, 4 * M * H)
assert L.TSHip_FusedFFNSwiGLUQuantF32Device(r16, x16, nw.ctypes.data, H, 1e-6, gu.ctypes.data, 8, H, 2 * F, gu.size, dn.ctypes.data, 8, F, H, dn.size, F)
out.append([log(), 8 * M * F + max(workspace(M, 2 * F, H, 0), workspace(M, H, F, 1))])
n = 3
w = (C.c_void_p * n)(*[gu.ctypes.data] * n)
d = (C.c_void_p * n)(*[dn.ctypes.data] * n)
up = (8, H, F, F * H // 32 * 34)
stream = C.c_void_p(1 << 20)                    # (a buffer of its own)
L.TSHip_SetStream(stream)
assert L.TSHip_MoEExpertsSwiGLUForwardF32Device(r16, x16, n, w, w, d, *up, *up, 8, F, H, dn.size, (C.c_float * n)(1, 1, 1)), L.TSHip_GetLastError()
out.append([log(), n * M * (8 * F + 4 * H + 2 * H + 2 * F)])
"""


def test_scratch_of_gated_rows_is_not_reserved_where_the_conversion_forms_them(stub):
    """[gate | up], the results and the converted activations, but no M x F floats of gated rows."""
    M, H, F = 64, 1024, 1024
    for log, need in stub(SCRATCH, M=M, H=H, F=F):
        (got,) = [int(l[1]) for l in log if l[0] == "malloc"]
        assert need <= got / 1.25 < need + 4 * M * F, (got / 1.25, need)


TILE_SCRATCH = """
w = space(max(H, F) * max(H, F) // 32 * 34)
x, r = space(4 * M * H).view(np.float32), space(4 * M * H).view(np.float32)
e, up, down = (C.c_void_p * n)(*[w.ctypes.data] * n), (8, H, F, F * H // 32 * 34), (8, F, H, F * H // 32 * 34)
assert L.TSHip_MoEExpertsSwiGLUForwardF32Device(view(r, M, H), view(x, M, H), n, e, e, e, *up, *up, *down, (C.c_float * n)(*[1] * n)), L.TSHip_GetLastError()
out.append(log())
"""


@pytest.mark.parametrize("n,M,H,F", [(2, 200, 4096, 512), (3, 300, 4096, 512), (2, 161, 512, 4096)])
def test_expert_sets_on_128_row_tiles_reserve_no_chunk_sums(stub, n, M, H, F):
    """Launches by tile tables run with whole K; the size of their scratch is asked for before the tables are there."""
    (log,) = stub(TILE_SCRATCH, n=n, M=M, H=H, F=F)
    (got,) = [int(l[1]) for l in log if l[0] == "malloc"]
    need = n * M * (8 * F + 4 * H + 2 * H + 2 * F)                          # (gate | up), the results, the converted rows of both
    assert need <= got / 1.25 < need + n * M * 64 + (1 << 16), (got / 1.25, need)


def test_only_stamped_launches_leave_the_split_kernel(stub):
    """While a timeline buffer is set, plain launches of few and long rows run unsplit; those with the RMSNorm are not stamped."""
    on = "assert L.TSHip_SetGemvTimeline(C.c_void_p(4096), 1 << 20)\n"
    cases = [(*BLOCKS["q8_0"], 512, 8192, norm, 0) for norm in (0, 1)]
    for plain, norm in (stub(GEMV_LINEAR, cases=cases), stub(on + GEMV_LINEAR, cases=cases)):
        assert len(launches(norm, "gemv_split_kernel")) == 1
    assert not launches(plain, "gemv_split_kernel")


TWO_TYPES = """
w, blocks = space(max(H, I) * max(H, I) // 32 * 34), {8: 34, 2: 18}
x, r = space(4 * M * H).view(np.float32), space(4 * M * H).view(np.float32)
shape = lambda t: (t, H, I, I * H // 32 * blocks[t], t, H, I, I * H // 32 * blocks[t], t, I, H, H * I // 32 * blocks[t])
e, p = (C.c_void_p * n)(*[w.ctypes.data] * n), C.c_void_p(w.ctypes.data)
assert L.TSHip_MoEExpertsSwiGLUResidualF32Device(view(r, M, H), view(x, M, H), n, e, e, e, *shape(8), (C.c_float * n)(*[1] * n), 1, p, p, p, *shape(2), 1.0), L.TSHip_GetLastError()
out.append(log())
"""


def test_sums_of_an_expert_set_of_two_types_are_added_for_the_rows_of_each(stub):
    """Gate, up and down projections of four routed Q8_0 experts and a shared Q4_0 one, K in chunks: the sums of one type's launch are
    added to its members' rows only, the others' rows are another launch's results."""
    n, M = 4, 20
    (log,) = stub(TWO_TYPES, n=n, M=M, H=8192, I=8192)
    assert [int(l[3]) for l in launches(log, "gemm_chunk_sum")] == 3 * [n * M, M], launches(log, "gemm_chunk_sum")
