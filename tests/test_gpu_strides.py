"""A host matrix whose columns lie back to back is copied to and from the device in one
linear copy, one with a larger leading dimension column by column: both must give the
same bits, and the rows between the columns stay as they were."""
import ctypes

import numpy as np
import pytest

from test_oracle_cauchy import interlaced

pytestmark = pytest.mark.gpu
MARK = -7.25


@pytest.fixture(scope="module")
def ctx():
    torch = pytest.importorskip("torch")
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from hsspack_amd import hsdc
    c = hsdc.Context()
    yield c
    c.close()


def padded(a, pad):
    """a in the first rows of a column-major block with pad rows more."""
    p = np.full((a.shape[0] + pad, a.shape[1]), MARK, order="F")
    p[:a.shape[0]] = a
    return p


def p_(a):
    return a.ctypes.data_as(ctypes.POINTER(ctypes.c_double))


def i_(a):
    return a.ctypes.data_as(ctypes.POINTER(ctypes.c_int))


def call(ctx, entry, n, pad):
    """One call of the entry with leading dimensions n + pad; the block it wrote."""
    from hsspack_amd import hsdc
    L = hsdc.lib()
    rng = np.random.default_rng(n)
    d, f, u, v = interlaced(n, n + 7)
    b = padded(rng.uniform(0, 1, (n, n)), pad)
    t, ranks = np.zeros(2), np.zeros(2 * (2 * n + 4), np.int32)
    if entry == "cauchyhssmm":
        rc = L.hsdc_cauchyhssmm(ctx._h, p_(d), p_(f), p_(u), p_(v), n, 60, 1e-11, 128, p_(b), n + pad, p_(t), i_(ranks))
    elif entry == "dhssmm":
        a = padded(u[:, None] * v[None, :] / (d[:, None] - f[None, :]), pad)
        rc = L.hsdc_dhssmm(ctx._h, p_(a), n + pad, n, n, p_(b), n + pad, n, 1e-11, 0, 60, 100, p_(t), i_(ranks))
    else:  # stedc with COMPZ = 'V': Z := Z Q
        dd, ee = np.full(n, 2.0), np.ones(max(n - 1, 1))
        work, iwork = np.zeros(1), np.zeros(1, np.int32)
        args = (ctypes.c_char(b"V"), n, p_(dd), p_(ee), p_(b), n + pad)
        rc = L.hsdc_stedc(ctx._h, *args, p_(work), -1, i_(iwork), -1)
        assert rc == 0
        work, iwork = np.zeros(int(work[0])), np.zeros(int(iwork[0]), np.int32)
        rc = L.hsdc_stedc(ctx._h, *args, p_(work), len(work), i_(iwork), len(iwork))
    assert rc == 0
    return b


@pytest.mark.parametrize("entry", ["cauchyhssmm", "dhssmm", "stedc"])
@pytest.mark.parametrize("n", [2, 257, 1100])
def test_leading_dimension(ctx, entry, n):
    want = call(ctx, entry, n, 0)
    assert not np.array_equal(want, np.random.default_rng(n).uniform(0, 1, (n, n)))
    got = call(ctx, entry, n, 3)
    np.testing.assert_array_equal(got[:n], want)
    assert np.all(got[n:] == MARK)
