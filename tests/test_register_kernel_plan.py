"""Which of the two register-resident kernels a product of few rows is planned for, seen in its K chunks (the one of 16-column tiles holds
twice the K range of the other in most formats): CPU tests, the library assumes 256 CUs without a GPU."""
import pytest

from test_matmul_plan import Q4_K, Q5_K, Q6_K, Q8_0, REGISTERS, converted_bytes, plan

Q5_0 = 6


@pytest.mark.parametrize("t,rows,n,k,accumulate,chunks", [
    # 32-column tiles: with 16 columns the runs of units cross into another chunk and these took 10 to 30 % longer
    (Q6_K, 23, 5120, 6144, 0, 3), (Q6_K, 26, 5288, 5120, 0, 3), (Q6_K, 31, 5428, 5120, 1, 3), (Q6_K, 37, 2560, 4352, 0, 3), (Q8_0, 27, 2560, 14336, 1, 7),
    (Q8_0, 55, 1088, 14336, 0, 7), (Q8_0, 21, 5120, 14848, 0, 8), (Q5_K, 17, 5120, 5120, 1, 3), (Q5_K, 34, 4096, 5888, 0, 3), (Q5_0, 24, 6144, 11488, 0, 4),
    # 16-column tiles: one chunk, or fewer, and nothing to cross into
    (Q8_0, 24, 4096, 2560, 0, 1), (Q6_K, 24, 14336, 4096, 0, 1), (Q8_0, 8, 9728, 4096, 0, 1), (Q6_K, 16, 4096, 4096, 0, 1), (Q5_K, 48, 14336, 4096, 0, 1)])
def test_the_faster_kernel_is_planned(t, rows, n, k, accumulate, chunks):
    assert plan(t, rows, n, k, accumulate)[:3:2] == (REGISTERS, chunks)


@pytest.mark.parametrize("t,rows,n,k,fewer", [(Q6_K, 23, 5120, 6144, 2), (Q8_0, 21, 5120, 14848, 4), (Q5_K, 34, 4096, 5888, 2), (Q5_0, 24, 6144, 11488, 3)])
def test_a_scratch_limit_takes_the_kernel_whose_sums_fit(t, rows, n, k, fewer):
    free = plan(t, rows, n, k)
    fits = converted_bytes(rows, k) + fewer * rows * n * 4
    assert free[3] > fits
    tight = plan(t, rows, n, k, 0, fits)
    assert tight[3] <= fits and (tight[0], tight[2]) in ((REGISTERS, fewer), (4, tight[2]))
    if t in (Q5_K, Q5_0):                                                    # (no other kernel serves these rows)
        assert (tight[0], tight[2]) == (REGISTERS, fewer)
