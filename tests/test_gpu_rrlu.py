"""The construction and product kernels at the edges of their splits: pivot steps with more
node rows than a wavefront searches by itself (256), the swap check's lanes per column, the
general Cauchy compression with its arrays in LDS and in global memory, the truncated SVDs
with R and V, R alone or neither in LDS and with exactly parallel columns, and the dense
merge product over more inner columns than its table holds (512).  Ranks equal the
oracle's; products are within rounding of the oracle's form or of the dense product."""
import numpy as np
import pytest

import oracle_py as O
from hsspack_amd.workloads import tridiag_cfg
from test_oracle_cauchy import interlaced
from test_oracle_dhssmm import fmm_matrix, node_ranks

pytestmark = pytest.mark.gpu
EPS = 2.0 ** -53


@pytest.fixture(scope="module")
def ctx():
    torch = pytest.importorskip("torch")
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from hsspack_amd import hsdc
    c = hsdc.Context()
    yield c
    c.close()


@pytest.mark.parametrize("K,ni", [(40, 8), (513, 256), (640, 300), (1024, 512), (1500, 64)])
def test_structured_rrlu_ranks_vs_oracle(ctx, K, ni):
    rng = np.random.default_rng(K)
    d = np.sort(rng.uniform(-1, 1, K))
    z = rng.standard_normal(K)
    z /= np.linalg.norm(z)
    v = O.mdlaed3_vectors(d, z, 1.1)
    H = O.hss_build(v["dlamda"], v["d"], v["z"], v["alpha"], v["difl"], v["difr"], ni, 1e-14)
    try:
        usz, vsz = O.hss_ranks(H)
        Hd = O.hss_dense(H)
    finally:
        O.hss_free(H)
    x = rng.standard_normal((67, K))
    y, ranks = ctx.hss_evc(v["dlamda"], v["d"], v["z"], v["alpha"], v["difl"], v["difr"], x, ni, 1e-14)
    ltr = usz.shape[0]
    assert ranks[0] != -1
    assert np.array_equal(ranks[: 2 * ltr:2][: ltr - 1], usz[: ltr - 1, 1])
    assert np.array_equal(ranks[1: 2 * ltr:2][: ltr - 1], vsz[: ltr - 1, 0])
    assert np.abs(y - x @ Hd).max() <= 1e-12 * np.abs(x).max() * K ** 0.5


@pytest.mark.parametrize("n,ni", [(97, 31), (1200, 400), (4200, 2100)])
def test_general_cauchy_lds_and_global(ctx, n, ni):
    """n = 4200 with leaves of 2100 needs more LDS than a workgroup has."""
    d, f, u, v = interlaced(n, n)
    b = np.random.default_rng(n).uniform(0, 1, (n, n))
    y, _, ranks = ctx.cauchyhssmm(d, f, u, v, b, ni, 1e-13, 128)
    assert ranks is not None
    H = O.cauchy2hss(d, f, u, v, ni, 1e-13)
    try:
        usz, vsz = O.hss_ranks(H)
    finally:
        O.hss_free(H)
    got = ranks.reshape(-1, 2)[:len(usz)]
    assert np.array_equal(got[:, 0], usz[:, 1]) and np.array_equal(got[:, 1], vsz[:, 0])
    ref = O.cauchy_dense_general(d, f, u, v) @ b
    # the truncation leaves at most about tol per entry of a block row of n entries
    assert np.abs(y - ref).max() <= 1e-13 * n * np.abs(ref).max()


@pytest.mark.parametrize("n,ni,right", [(330, 99, False), (420, 130, True), (500, 160, False)])
def test_truncated_svd_lds_tiers(ctx, n, ni, right):
    """Leaves of 99 (R and V in LDS), 130 (R) and 160 or more rows (neither)."""
    a = fmm_matrix(n, 5)
    b = np.random.default_rng(n).uniform(0, 1, (n, n))
    y, _, ranks = ctx.dhssmm(a, b, ni, 1e-11, right=right)
    assert ranks is not None
    H = O.mat2hss(a, ni, 1e-11)
    ou, ov = node_ranks(H)
    ltr = H.ltr
    Hd = O.hss_dense(H)
    O.hss_free(H)
    r = np.asarray(ranks)[:2 * ltr].reshape(-1, 2)
    assert np.array_equal(r[:-1, 0], ou) and np.array_equal(r[:-1, 1], ov)
    ref = b @ Hd if right else Hd @ b
    assert np.abs(y - ref).max() <= 1e-11 * np.abs(ref).max()


def test_parallel_columns_converge(ctx):
    """Blocks of exact rank one: powers of two, so that the columns are parallel to the last
    bit and the Jacobi sweeps drive one of each pair to underflow."""
    n = 128
    u = 2.0 ** np.random.default_rng(2).integers(-3, 4, n)
    a = np.outer(u, u[::-1])
    b = np.random.default_rng(3).uniform(0, 1, (n, 20))
    y, _, ranks = ctx.dhssmm(a, b, 16, 1e-10)
    assert ranks is not None and np.asarray(ranks).max() <= 1
    assert np.abs(y - a @ b).max() <= 1e-12 * np.abs(a @ b).max()


@pytest.mark.parametrize("n", [1090, 1411])
def test_dense_product_over_several_column_groups(ctx, n):
    d, e = tridiag_cfg(1, n, 8)
    ctx.set_params(hss_min_k=1 << 30)
    try:
        lam, z, info = ctx.stedc(d, e)
    finally:
        ctx.set_params(hss_min_k=1500)
    assert info == 0
    t = np.diag(d) + np.diag(e, 1) + np.diag(e, -1)
    assert np.abs(lam - np.linalg.eigvalsh(t)).max() <= 4 * n * EPS * np.abs(t).max()
    assert np.abs(z.T @ z - np.eye(n)).max() <= 1e-12
    assert np.abs(t @ z - z * lam).max() <= 1e-12 * np.abs(t).max()
