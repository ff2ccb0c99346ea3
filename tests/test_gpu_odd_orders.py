"""A call whose rows end inside a wave's 256 is not far slower than its aligned
neighbour: the one wave that crosses the matrix's last row works in the same
steps as the others. (It once took the launch with it: the ratios below were
1.7 and more.) The times are the context's own, the best of several calls, and
the limit leaves room for the edge and for noise."""
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
