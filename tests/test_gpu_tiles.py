"""Kernels at the edges of their tiles: the column dots at every group width
and piece count (and past one pass), on four waves and ahead on three, the
sweeps and the downdate on both sides of 64 and 128 columns, the scan's
results and digits at odd sizes, the raw body's rows at every alignment."""
import numpy as np
import pytest

import oracle
from bmagwa_amd import synth

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def bmg():
    import bmagwa_amd
    bmagwa_amd.lib()
    return bmagwa_amd


def genotypes(n, p, seed):
    """p x n genotypes and their packed body."""
    rng = np.random.default_rng(seed)
    maf = rng.uniform(0.1, 0.5, size=(p, 1))
    G = (rng.random((p, n)) < maf).astype(np.uint8) + (rng.random((p, n)) < maf)
    code = np.zeros((p, (n + 3) // 4 * 4), np.uint8)
    code[:, :n] = np.array([0, 2, 3], np.uint8)[G]
    body = (code.reshape(p, -1, 4) << np.array([0, 2, 4, 6], np.uint8)).sum(2, dtype=np.uint8)
    return G, body.ravel()


CODED = {"A": [0., 1., 2.], "H": [0., 1., 0.], "D": [0., 1., 1.], "R": [0., 0., 1.]}


# 16 / 32 / 64 lanes a column, then 2, 3 and 5 pieces a lane, then two passes
@pytest.mark.parametrize("n", [37, 1024, 1025, 2049, 4097, 8193, 12289, 20481])
def test_column_dots(bmg, n):
    """X^T X of a model with terms of every coding: whole numbers, exact."""
    types = ("A", "H", "D", "R")
    G, body = genotypes(n, 12, n)
    y = np.random.default_rng(n).normal(size=n)
    ctx = bmg.Ctx(n, 12, body, y, types=types)
    m = bmg.Model(ctx, n_plus_nu=n + 1.0, nus2_plus_yy=1.0 + float(y @ y), inv_tau2_e0=0.0)
    X = [np.ones(n)]
    for j in range(11):
        m.add_term(j, j % 4, 3.0)
        X.append(np.array(CODED[types[j % 4]])[G[j]])
    X = np.array(X)
    xx = m.get()["xx"]
    assert np.array_equal(np.triu(xx), np.triu(X @ X.T))
    m.close()
    ctx.close()


# one group width each, and two passes
@pytest.mark.parametrize("n", [37, 1025, 4097, 20481])
def test_column_dots_of_a_pair(bmg, n):
    """Two columns a term: X^T X exact while terms are added, removed and
    added again (a Model forms each column's dots on all four waves)."""
    G, body = genotypes(n, 14, n + 1)
    y = np.random.default_rng(n).normal(size=n)
    ctx = bmg.Ctx(n, 14, body, y, types=("AH",))
    m = bmg.Model(ctx, n_plus_nu=n + 1.0, nus2_plus_yy=1.0 + float(y @ y), inv_tau2_e0=0.0)
    terms = []

    def check():
        X = np.array([np.ones(n)] + [np.array(CODED[c])[G[j]] for j in terms for c in "AH"])
        assert np.array_equal(np.triu(m.get()["xx"]), np.triu(X @ X.T))

    for j in range(10):
        m.add_term(j, 0, [3.0, 4.0])
        terms.append(j)
    check()
    for i in (7, 0, 3):
        m.remove_term(i)
        del terms[i]
    for j in range(10, 14):
        m.add_term(j, 0, [2.0, 5.0])
        terms.append(j)
    check()
    m.close()
    ctx.close()


# both sides of every group width and piece count, then two and three passes
@pytest.mark.parametrize("types", ["A", "AH"])
@pytest.mark.parametrize("n", [37, 1024, 1025, 2048, 2049, 4097, 8192, 8193, 12288, 12289, 20480, 20481, 40961])
def test_column_dots_formed_ahead(bmg, n, types):
    """A chain's moves of several SNPs, whose next columns' dots three waves
    form beside a sweep or a downdate (with the tree write and the row move
    that go with it): the dots are whole numbers, so moves and sizes are the
    oracle's and log-likelihoods agree to 1e-10, as for every trajectory."""
    p, n_iter = 48, 400
    G, body = genotypes(n, p, n)
    rng = np.random.default_rng(n)
    y = rng.normal(size=12) @ G[:12] + rng.normal(scale=3.0, size=n)
    cfg = synth.sampler_cfg(n, p, 12, types=types, seed=5, n_rao=50, n_rao_burnin=2, max_move_size=10,
                            p_move_size=0.1, adapt_p_move_size=0, do_n_iter=n_iter)
    s = oracle.Sampler(cfg, oracle.Data(n, p, body, y))
    s.init_flat()
    assert s.setup() == 0
    s.iterate(n_iter)
    want = s.trace()
    ctx = bmg.Ctx(n, p, body, y, types=(types,))
    b = bmg.Batch([ctx], [0], [cfg], dict(trace_every_iter=1))
    b.setup()
    b.run(n_iter)
    got = b.trace(0)
    for key in ("move", "jd", "ms", "size"):
        assert np.array_equal(got[key], want[key]), key
    assert np.allclose(got["loglik"], want["loglik"], rtol=1e-10, atol=0)
    # moves of several SNPs were accepted, so their columns are in the model
    assert ((got["move"] == 0) & (got["jd"] > 2)).any()
    b.close()
    ctx.close()


# a workgroup a SNP below 1,536 SNPs, then groups of eight, whole and ragged
@pytest.mark.parametrize("n,p,types", [(15, 60, "A"), (4097, 60, "R"), (1030, 1535, "AH"), (1030, 1536, "A"),
                                       (1030, 1537, "D"), (515, 1543, "AH")])
def test_xy_table(bmg, n, p, types):
    """The table of x.y that a chain's additions read: a wrong entry shows in
    the first model that holds its SNP.  The sums of either form are within
    n ulps of the oracle's; trajectories agree to 1e-10 as elsewhere."""
    n_iter = 300
    G, body = genotypes(n, p, n + p)
    rng = np.random.default_rng(p)
    y = rng.normal(size=10) @ G[p - 10:] + rng.normal(scale=2.0, size=n)
    cfg = synth.sampler_cfg(n, p, 10, types=types, seed=9, n_rao=50, n_rao_burnin=2, max_move_size=10, do_n_iter=n_iter)
    s = oracle.Sampler(cfg, oracle.Data(n, p, body, y))
    s.init_flat()
    assert s.setup() == 0
    s.iterate(n_iter)
    want = s.trace()
    ctx = bmg.Ctx(n, p, body, y, types=(types,))
    b = bmg.Batch([ctx], [0], [cfg], dict(trace_every_iter=1))
    b.setup()
    b.run(n_iter)
    got = b.trace(0)
    for key in ("move", "jd", "ms", "size"):
        assert np.array_equal(got[key], want[key]), key
    assert np.allclose(got["loglik"], want["loglik"], rtol=1e-10, atol=0)
    assert got["size"].max() > 0
    b.close()
    ctx.close()


# columns before the removal; the removed term; n - 1 columns follow it
@pytest.mark.parametrize("k,rm", [(2, 0), (9, 0), (9, 4), (9, 8), (64, 0), (65, 0), (66, 0), (66, 60), (129, 0),
                                  (130, 1), (130, 70), (135, 0), (135, 127), (135, 134)])
def test_downdate_and_sweeps(bmg, k, rm):
    """Factor, v and log-likelihood after a removal (and an addition after
    it) equal a fresh float64 factorisation.  Both are backward stable, so
    entries agree to a small multiple of 2^-52 times the condition number,
    here below 1e4: 1e-10 of the largest entry."""
    n = 700
    G, body = genotypes(n, k + 1, 11 * k + rm)
    rng = np.random.default_rng(k)
    y = rng.normal(size=n)
    d = rng.uniform(5.0, 50.0, size=k + 1)
    ctx = bmg.Ctx(n, k + 1, body, y)
    n_nu, nus2_yy = n + 1.0, 1.0 + float(y @ y)
    m = bmg.Model(ctx, n_plus_nu=n_nu, nus2_plus_yy=nus2_yy, inv_tau2_e0=0.0)
    for j in range(k):
        m.add_term(j, 0, d[j])
    order = list(range(k))

    def check():
        X = np.concatenate([np.ones((1, n)), G[order].astype(float)])
        dd = np.concatenate([[0.0], d[order]])
        U = np.linalg.cholesky(X @ X.T + np.diag(dd)).T
        v = np.linalg.solve(U.T, X @ y)
        s = m.get()
        assert np.allclose(np.triu(s["l"]), U, rtol=0, atol=1e-10 * np.abs(U).max())
        assert np.allclose(s["v"], v, rtol=0, atol=1e-10 * np.abs(v).max())
        ll = 0.5 * np.log(dd[1:]).sum() - np.log(np.diag(U)).sum() - 0.5 * n_nu * np.log(nus2_yy - v @ v)
        assert abs(s["loglik"] - ll) < 1e-10 * abs(ll)

    check()
    m.remove_term(rm)
    del order[rm]
    check()
    m.add_term(k, 0, d[k])
    order.append(k)
    check()
    m.compute_log_likelihood()
    check()
    m.close()
    ctx.close()


@pytest.mark.parametrize("n,p,nvec,digits,coding", [(5, 1, 1, 1, 0), (63, 3, 3, 5, 0), (513, 66, 2, 6, 1),
                                                    (1000, 131, 16, 1, 2), (2500, 1025, 3, 4, 3),
                                                    (17000, 259, 3, 5, 0)])
def test_scan_results_at_odd_sizes(bmg, n, p, nvec, digits, coding):
    """Residuals of whole numbers are represented exactly, so X^T R is exact
    (one and several individual tiles, every digit count)."""
    G, body = genotypes(n, p, n + p)
    rng = np.random.default_rng(p)
    R = rng.integers(-7, 8, size=(nvec, n)).astype(float)
    ctx = bmg.Ctx(n, p, body, np.zeros(n))
    X = np.array(CODED["AHDR"[coding]])[G]
    assert np.array_equal(ctx.scan_xtr(R, coding=coding, digits=digits), R @ X.T)
    ctx.close()


@pytest.mark.parametrize("n", [2, 5, 63, 64, 65, 66, 67, 68, 1021, 2047])
@pytest.mark.parametrize("p", [1, 3, 8])
def test_raw_body_rows(bmg, n, p):
    """Rows of every byte alignment arrive whole; moments are exact."""
    G, body = genotypes(n, p, 7 * n + p)
    ctx = bmg.Ctx(n, p, body, np.zeros(n))
    assert np.array_equal(ctx.read_body(), body)
    s = G.astype(np.int64).sum(1)
    assert np.array_equal(ctx.self_moments()[:, 0], s.astype(float))
    assert ctx.missing_count() == 0
    ctx.close()
