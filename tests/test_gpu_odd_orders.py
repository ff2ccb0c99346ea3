"""A call whose rows end inside a wave's 256, or a block's 1024, is not far slower
than its aligned neighbour: the waves there work in the same steps as the
others. (They once took the launch with them.) The times are the context's own,
the best of several calls, and the limits leave room for the edge and for
noise: beside each test stands what the fault measured and what it measures now."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

LIMIT = 1.35


@pytest.fixture(scope="module")
def timed():
    from wgblas_amd import Context

    c = Context(0)
    c.set_timing(True)
    yield c
    c.close()


def _best(c, call):
    for _ in range(3):
        call()
    times = []
    for _ in range(12):
        call()
        times.append(c.last_time_ms())
    return min(times)


# 1.7 to 1.8 with the fault, 1.0 without
@pytest.mark.parametrize("uplo,odd,lda,even", [(1, 12000, 12000, 12032), (2, 16383, 16384, 16384),
                                               (2, 16382, 16384, 16384)])
def test_ssymv_at_orders_that_are_no_multiple_of_256(timed, uplo, odd, lda, even):
    c = timed
    A, x, y = c.empty(even * even, np.float32), c.empty(even, np.float32), c.empty(even, np.float32)
    try:
        for k, buf in enumerate((A, x, y)):
            c.fill_uniform(buf, -1, 1, 7 + k)
        at_odd = _best(c, lambda: c.ssymv(uplo, odd, 1.0, A, lda, x, 1, 0.0, y, 1))
        at_even = _best(c, lambda: c.ssymv(uplo, even, 1.0, A, even, x, 1, 0.0, y, 1))
        assert at_odd < LIMIT * at_even, (at_odd, at_even)
    finally:
        for buf in (A, x, y):
            buf.free()


# 0.92 and 0.80 with the fault, 0.61 and 0.53 without
@pytest.mark.parametrize("rows,lda,limit", [(901, 904, 0.75), (768, 768, 0.67)])
def test_dger_with_a_cut_row_chunk(timed, rows, lda, limit):
    c, n = timed, 30000
    A, x, y = c.empty(1024 * n, np.float64), c.empty(1024, np.float64), c.empty(n, np.float64)
    try:
        for k, buf in enumerate((A, x, y)):
            c.fill_uniform(buf, -1, 1, 17 + k)
        cut = _best(c, lambda: c.dger(rows, n, 1e-9, x, 1, y, 1, A, lda))
        whole = _best(c, lambda: c.dger(1024, n, 1e-9, x, 1, y, 1, A, 1024))
        assert cut < limit * whole, (cut, whole)
    finally:
        for buf in (A, x, y):
            buf.free()


# 1.94 with the fault, 1.0 without
@pytest.mark.parametrize("m,lda", [(8191, 8191), (8189, 8190)])
def test_dgemv_at_rows_that_are_no_multiple_of_4(timed, m, lda):
    c = timed
    A, x, y = c.empty(8192 * 8192, np.float64), c.empty(8192, np.float64), c.empty(8192, np.float64)
    try:
        for k, buf in enumerate((A, x, y)):
            c.fill_uniform(buf, -1, 1, 27 + k)
        odd = _best(c, lambda: c.dgemv(0, m, 8191, 1.0, A, lda, x, 1, 0.0, y, 1))
        even = _best(c, lambda: c.dgemv(0, 8192, 8192, 1.0, A, 8192, x, 1, 0.0, y, 1))
        assert odd < LIMIT * even, (odd, even)
    finally:
        for buf in (A, x, y):
            buf.free()
