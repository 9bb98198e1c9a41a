"""How products are planned (TSHip_MatmulPlanDevice): CPU tests, no GPU needed - the library assumes 256 CUs without one."""
import ctypes as C

import pytest

from tensorsharp_amd import hip_native as N

Q4_K, Q5_K, Q6_K, Q8_0, MXFP4, Q8_1, F32 = 12, 13, 14, 8, 39, 9, 0
GEMV, DENSE, REGISTERS, WIDE, TILES = 1, 2, 3, 4, 5


def plan(t, rows, n, k, accumulate=0, max_workspace=0):
    """(kernel, rows per tile, K chunks, workspace bytes)"""
    out = (C.c_int64 * 4)()
    N.check_result(N.lib().TSHip_MatmulPlanDevice(t, rows, k, n, accumulate, max_workspace, out), "plan")
    return tuple(out)


def converted_bytes(rows, k):
    """row scales and fp16 activations of a call, 256-byte granules"""
    al = lambda b: (b + 255) // 256 * 256
    return al(rows * ((k + 63) // 64 * 64) * 2 + al(rows * 4) + 256)


def test_kernels_by_rows_columns_and_type():
    for t in (Q4_K, Q5_K, Q6_K, Q8_0, MXFP4):
        for rows in (1, 2, 3):
            assert plan(t, rows, 4096, 4096) == (GEMV, 1, 1, 0)
        assert plan(t, 4, 63, 4096)[0] == DENSE and plan(t, 4, 64, 4096)[0] != DENSE
        assert plan(t, 4096, 4096, 1024)[0] in (WIDE, TILES)
    assert plan(F32, 100, 4096, 4096) == (DENSE, 1, 1, 0)
    assert plan(Q8_1, 100, 4096, 4096)[0] == DENSE


@pytest.mark.parametrize("t", [Q4_K, Q5_K, Q6_K, Q8_0, MXFP4])
@pytest.mark.parametrize("rows,n,k", [(4, 4096, 4096), (24, 14336, 4096), (200, 4096, 14336), (700, 1024, 2048), (2048, 21504, 5376)])
@pytest.mark.parametrize("accumulate", [0, 1])
def test_workspace_holds_the_converted_rows_and_the_chunk_sums(t, rows, n, k, accumulate):
    kernel, tile, chunks, ws = plan(t, rows, n, k, accumulate)
    sums = chunks * rows * n * 4 if chunks > 1 or (accumulate and kernel == REGISTERS) else 0     # the register kernel adds in a second pass
    assert ws >= converted_bytes(rows, k) + sums
    assert 1 <= chunks <= (k + 63) // 64 and tile in (32, 64, 96, 128, 256)


def test_argument_errors():
    out = (C.c_int64 * 4)()
    for args in ((Q4_K, 0, 4096, 4096), (Q4_K, 8, 4000, 4096), (Q4_K, 8, 4096, 0), (77, 8, 4096, 4096)):
        assert N.lib().TSHip_MatmulPlanDevice(*args, 0, 0, out) == 0
    assert N.lib().TSHip_MatmulPlanDevice(Q4_K, 8, 4096, 4096, 0, 0, None) == 0


@pytest.mark.parametrize("t,rows,n,k,m_step,n_step", [
    # activations beyond 2 GiB of fp16: 16128 rows at a time, and a rest whose 32-row units need their K-chunk sums
    (Q5_K, 16128 + 32, 64, 65536, 16128, 64), (MXFP4, 16128 + 9, 300, 65536, 16128, 300), (Q4_K, 16128 + 32, 300, 65536, 16128, 300),
    # weights beyond 2 GiB: 123136 columns at a time, and a rest of few tiles
    (Q8_0, 512, 123136 + 300, 16384, 512, 123136), (Q4_K, 700, 232960 + 70, 16384, 700, 232960), (Q6_K, 40, 159744 + 513, 16384, 40, 159744),
])
def test_workspace_holds_the_sums_of_every_slice(t, rows, n, k, m_step, n_step):
    have = plan(t, rows, n, k)[3] - converted_bytes(m_step, k)
    for m in {m_step, rows % m_step or m_step}:
        for cols in {n_step, n % n_step or n_step}:
            need = plan(t, m, cols, k)[3] - converted_bytes(m, k)
            assert have >= need, (m, cols, have, need)


@pytest.mark.parametrize("t,rows,n,k", [(Q6_K, 333, 4096, 14336), (Q4_K, 333, 4096, 14336), (Q8_0, 200, 4096, 14336), (Q4_K, 700, 4096, 14336),
                                        (Q4_K, 64, 4096, 14336), (Q8_0, 16, 4096, 14336), (Q6_K, 20, 9728, 9728)])
@pytest.mark.parametrize("accumulate", [0, 1])
def test_a_bounded_workspace_keeps_as_many_chunks_as_fit(t, rows, n, k, accumulate):
    conv, sums = converted_bytes(rows, k), rows * n * 4
    kernel, _, free, ws = plan(t, rows, n, k, accumulate)
    assert free >= 2 and ws >= conv + free * sums
    assert plan(t, rows, n, k, accumulate, ws) == plan(t, rows, n, k, accumulate)           # just enough
    last = free
    for fit in range(free - 1, -1, -1):
        got = plan(t, rows, n, k, accumulate, conv + fit * sums)
        assert got[3] <= conv + fit * sums and got[2] <= max(fit, 1) and got[2] <= last
        assert got[2] >= 2 or fit < 2 or got[0] != WIDE, (fit, got)        # some of the chunks, where the tiles take any number
        last = got[2]
    assert plan(t, rows, n, k, accumulate, 1)[2] == 1                       # (refused by the entry points: not even the conversions fit)


# measured us of a call, conversion included, weights from HBM: register-resident kernel, the best tiling of the wide kernel, 128- and
# 256-row tiles (None: not a candidate, or not measured)
# (of the kernels that the rule's constants were first fitted to: the register-resident kernel with whole rows of activations, the wide
# kernel of Q6_K before its loop was unrolled; both are faster now, the picks asserted here are those of that fit)
MEASURED = [
    (Q4_K, 8, 4096, 4096, 12.44, 16.28, None, None),
    (Q4_K, 24, 14336, 4096, 21.49, 22.75, 29.53, None),
    (Q4_K, 64, 4096, 4096, 17.41, 21.03, 28.53, 34.04),
    (Q4_K, 96, 4096, 4096, 30.29, 22.9, 29.82, 35.6),
    (Q4_K, 333, 4096, 14336, 115.11, 68.06, 75.84, 90.81),
    (Q4_K, 512, 14336, 4096, 115.92, 75.75, 82.23, 82.91),
    (Q4_K, 1024, 9728, 2560, 150.97, 85.79, 104.73, 68.69),
    (Q4_K, 2048, 21504, 5376, 1369.3, 563.49, 629.79, 474.88),
    (Q8_0, 4, 4096, 4096, 12.79, 18.09, None, None),
    (Q8_0, 8, 9728, 2560, 18.02, 18.44, None, None),
    (Q8_0, 8, 14336, 4096, 23.23, 23.96, None, None),
    (Q8_0, 64, 4096, 4096, 18.59, 22.1, 29.58, 36.76),
    (Q8_0, 128, 28672, 4096, 90.74, 60.0, 66.98, 76.55),
    (Q8_0, 400, 4096, 4096, 55.68, 39.17, 37.37, 44.49),
    (Q8_0, 512, 14336, 4096, 164.74, 80.42, 87.37, 88.92),
    (Q8_0, 2048, 21504, 5376, 1408.48, 599.65, 683.56, 522.59),
    (Q6_K, 8, 4096, 4096, 12.97, 23.46, None, None),
    (Q6_K, 32, 9728, 2560, 21.68, 25.89, 31.07, None),
    (Q6_K, 64, 4096, 4096, 19.18, 28.07, 35.66, None),
    (Q6_K, 128, 14336, 4096, 54.08, 47.4, 44.14, None),
    (Q6_K, 333, 4096, 14336, 140.48, 94.45, 100.25, None),
    (Q6_K, 512, 14336, 4096, 181.74, 108.19, 106.67, None),
    (Q6_K, 1024, 14336, 4096, 374.15, 210.59, 205.78, None),
    (Q6_K, 2048, 2560, 9728, 351.84, 200.81, 240.7, None),
    (Q6_K, 512, 4096, 4096, 62.72, 47.51, 45.06, None),
]


@pytest.mark.parametrize("t,rows,n,k,registers,wide,tiles128,tiles256", MEASURED)
def test_the_pick_is_the_measured_best_or_close(t, rows, n, k, registers, wide, tiles128, tiles256):
    # few rows that the wide kernel pads to 32, Q6_K on 128-row tiles again, long prompts on 256-row tiles: nothing more than 5 %
    # behind the fastest
    kernel, tile, _, _ = plan(t, rows, n, k)
    took = {REGISTERS: registers, WIDE: wide}[kernel] if kernel != TILES else {128: tiles128, 256: tiles256}[tile]
    assert took <= 1.05 * min(us for us in (registers, wide, tiles128, tiles256) if us is not None)


def test_adding_to_a_residual_counts_the_second_pass_of_the_register_kernel():
    # it writes its sums to the workspace and adds them in a second launch; the wide kernel adds in place
    picks = [(plan(Q4_K, m, n, 2304)[0], plan(Q4_K, m, n, 2304, 1)[0]) for m in range(17, 200) for n in (1024, 2048, 4096, 8192, 14336)]
    assert any(plain == REGISTERS and added == WIDE for plain, added in picks)
    assert not any(plain == WIDE and added == REGISTERS for plain, added in picks)


@pytest.mark.parametrize("t", [Q8_0, Q6_K])
@pytest.mark.parametrize("rows", [4, 8, 16])
def test_few_rows_stay_on_the_register_kernel(t, rows):
    for n, k in ((1024, 4096), (4096, 4096), (9728, 2560), (21504, 5376), (4096, 14336)):
        assert plan(t, rows, n, k)[0] == REGISTERS and plan(t, rows, n, k, 1)[0] == REGISTERS


@pytest.mark.parametrize("t,rows,n,k,accumulate", [(Q4_K, 140, 701, 256, 1), (Q4_K, 339, 391, 256, 1), (Q4_K, 58, 975, 256, 1),
                                                   (Q8_0, 120, 5801, 256, 0), (Q6_K, 24, 14336, 1024, 0)])
def test_short_rows_are_not_sent_to_128_row_tiles(t, rows, n, k, accumulate):
    # a single super-block of K: starting a 128-row tile takes longer than the product (Q4_K 140 x 701 x 256 added to a residual
    # 31.5 us, 12.6 on the register-resident kernel)
    assert plan(t, rows, n, k, accumulate)[0] == REGISTERS
