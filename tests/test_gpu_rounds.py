"""The FP64 IRLS round kernels (rows too long for the gene kernel): one gene and
chunk per wavefront up to 96 genes, 16-gene tiles above, against the oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.fixture(scope="module")
def dv():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import devil_amd
    devil_amd.lib()
    return devil_amd


def counts(r, X, G, dtype=np.int32):
    n, p = X.shape
    B = np.column_stack([r.normal(0.5, 0.5, G)] + [r.normal(0, 0.1, G) for _ in range(p - 1)])
    sf = np.exp(r.normal(0, 0.3, n))
    mu = sf * np.exp(np.clip(B @ X.T, -5, 5))
    return r.poisson(r.gamma(2.0, mu / 2.0)).astype(dtype), sf


def check(dv, orc, Y, X, sf, Yd=None):
    """Iteration counts equal, beta within 1e-8 relative (floor 1e-6): an FP64 sum
    over n <= 2e5 cells in any order is within n 2^-53 ~ 2e-11 of another."""
    print(f"[case] G={Y.shape[0]} n={Y.shape[1]} p={X.shape[1]} {Y.dtype}", flush=True)
    fit = dv.fit_devil(torch.as_tensor(Y, device="cuda") if Yd is None else Yd, X,
                       size_factors=sf, overdispersion=False)
    ref = orc.cpu_fit(Y.astype(np.float64), X, np.log(sf), od_mode=orc.OD_NONE, n_threads=8)
    np.testing.assert_array_equal(fit["iterations"]["beta_iters"].cpu().numpy(),
                                  ref["beta_iters"])
    b = fit["beta"].cpu().numpy()
    err = np.abs(b - ref["beta"]) / np.maximum(np.abs(ref["beta"]), 1e-6)
    assert np.all(np.isfinite(err)) and err.max() <= 1e-8, err.max()
    return b


@pytest.mark.parametrize("intercept", [True, False])
def test_equal_columns_of_different_products(dv, orc, intercept):
    """x_3 = x_1 x_2 of two continuous columns: the sums of x_0 x_3 and x_1 x_2
    share a column and differ in their last bits; two fits have the same bits."""
    r = np.random.default_rng(11)
    n = 52428 + 100  # 8 (p + 1) n bytes just above 2 MiB
    z = r.normal(size=(n, 2))
    X = np.column_stack([np.ones(n) if intercept else 0.5 + r.uniform(size=n), z,
                         z[:, 0] * z[:, 1]])
    Y, sf = counts(r, X, 30)
    a = check(dv, orc, Y, X, sf)
    b = check(dv, orc, Y, X, sf)
    np.testing.assert_array_equal(a, b)


@pytest.mark.parametrize("G,n,p,intercept,one_launch", [
    (1025, 43690, 5, 1, True), (1025, 21845, 5, 0, True), (1025, 21846, 5, 0, False),
    (1024, 37449, 6, 0, True), (1025, 18724, 6, 1, True), (1025, 18725, 6, 1, False),
    (1025, 8192, 10, 0, True), (1025, 8193, 10, 0, False), (5001, 9362, 6, 1, True),
    (5001, 9363, 6, 1, False), (20001, 64, 8, 1, True), (20001, 64, 7, 0, True),
    (5000, 64, 8, 0, True), (5001, 64, 8, 0, False), (5001, 2978, 10, 1, True),
    (5001, 2979, 10, 1, False), (20000, 64, 9, 1, True), (20001, 64, 9, 1, False)])
def test_rule_of_the_gene_kernel(dv, G, n, p, intercept, one_launch):
    """The gene kernel runs the whole IRLS in one launch, the rounds in more:
    both sides of each line of the rule."""
    print(f"[case] rule G={G} n={n} p={p} intercept={intercept}", flush=True)
    gen = torch.Generator(device="cuda").manual_seed(n)
    Y = torch.poisson(torch.full((G, n), 2.0, device="cuda"), generator=gen).to(torch.int32)
    X = np.random.default_rng(p).normal(size=(n, p))
    X[:, 0] = 1.0 if intercept else X[:, 0] + 3.0
    ctx = dv.context(0)
    ctx.set_timing(True)
    try:
        dv.fit_devil(Y, X, overdispersion=False, max_iter=3)
        launches = ctx.kernel_stats()["irls_fp64"][0]
    finally:
        ctx.set_timing(False)
    assert (launches == 1) == one_launch, launches


def test_graph_tail_of_the_round_kernels(dv, orc):
    """The FP64 rounds of a row too long for the gene kernel, replayed from a
    captured graph (DEVIL_TUNE_GRAPH) and launched one by one: the lists of up to
    64 genes have the same chunks whatever their length, so the results have the
    same bits.  The graph records two rounds a launch: fewer timed launches."""
    from devil_amd import _lib as L
    r = np.random.default_rng(13)
    n, p, G = 120000, 8, 40
    X = np.column_stack([np.ones(n), r.uniform(size=n) < 0.4] +
                        [r.normal(size=n) for _ in range(p - 2)]).astype(np.float64)
    Y, sf = counts(r, X, G)
    Y[0] = 0  # more iterations than the others
    Y[0, ::9000] = 1
    Yd = torch.as_tensor(Y, device="cuda")
    ctx = dv.context(0)
    beta, launches = {}, {}
    try:
        ctx.set_timing(True)
        for graph in (1, 0):
            ctx.set_tuning(L.TUNE_GRAPH, graph)
            beta[graph] = check(dv, orc, Y, X, sf, Yd)
            launches[graph] = ctx.kernel_stats()["irls_fp64"][0]
    finally:
        ctx.set_tuning(L.TUNE_GRAPH, 0)
        ctx.set_timing(False)
    assert launches[1] < launches[0], launches
    np.testing.assert_array_equal(beta[1], beta[0])


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("G", [40, 96, 97, 130])
def test_count_types_of_the_round_kernels(dv, orc, G, dtype):
    """float32 and float64 counts, rows of odd length in an array of longer rows
    (leading dimension n + 6, a view that starts at an odd element): one gene
    per wavefront up to 96 genes, tiles above."""
    r = np.random.default_rng(G)
    n = 52428 + 3
    X = np.column_stack([np.ones(n), r.uniform(size=n) < 0.5] +
                        [r.normal(size=n) for _ in range(2)]).astype(np.float64)
    Y, sf = counts(r, X, G, dtype)
    wide = torch.full((G, n + 6), -1.0, dtype=torch.as_tensor(Y).dtype, device="cuda")
    wide[:, 3:n + 3] = torch.as_tensor(Y, device="cuda")
    check(dv, orc, Y, X, sf, wide[:, 3:n + 3])


def distinct_columns(X):
    """Distinct non-zero columns among the design's and their products."""
    p = X.shape[1]
    cols = [X[:, a] for a in range(p)] + [X[:, a] * X[:, b] for a in range(p)
                                          for b in range(a, p)]
    return len({c.tobytes() for c in np.array(cols) + 0.0 if c.any()})


@pytest.mark.parametrize("columns", [2, 17, 18, 19])
@pytest.mark.parametrize("patients", [0, 3])
def test_last_column_tile_of_long_rows(dv, orc, columns, patients):
    """Tiles of long rows (more than 96 genes) whose last column tile holds two
    columns and is the only one (an intercept and a 0/1 condition), one, two
    (both summed by vector instructions) and three (a matrix tile)."""
    r = np.random.default_rng(columns)
    n = 87381 + 5 if columns == 2 else 40000
    b = (r.uniform(size=n) < 0.4).astype(float)
    lv = r.integers(0, 3, n)
    z = r.normal(size=(n, 4))
    X = np.column_stack({
        2: [np.ones(n), b],
        17: [z[:, 0], z[:, 1], z[:, 2], b, 1 - b],          # no column of ones
        18: [np.ones(n), lv == 1, lv == 2, z[:, 0], z[:, 1], z[:, 2]],
        19: [z[:, 0], z[:, 1], z[:, 2], b, 0.5 * (lv == 1)],
    }[columns]).astype(np.float64)
    assert distinct_columns(X) == columns
    p = X.shape[1]
    if 8 * (p + 1) * n <= 2 << 20:
        n = (2 << 20) // (8 * (p + 1)) + 9
        X = np.resize(X, (n, p))
        assert distinct_columns(X) == columns
    G = 130
    Y, sf = counts(r, X, G)
    lab = np.sort(r.integers(0, patients, n)) if patients else None
    ends = None if lab is None else np.cumsum(np.bincount(lab)).astype(np.int32)
    print(f"[case] columns={columns} p={p} n={n} patients={patients}", flush=True)
    fit = dv.fit_devil(torch.as_tensor(Y, device="cuda"), X, size_factors=sf, clusters=lab)
    ref = orc.cpu_fit(Y.astype(np.float64), X, np.log(sf), od_mode=orc.OD_MOM,
                      clusters_ends=ends, n_threads=8)
    np.testing.assert_array_equal(fit["iterations"]["beta_iters"].cpu(), ref["beta_iters"])
    for key, want in (("beta", "beta"), ("overdispersion", "theta"),
                      ("beta_sandwiches_null", "bread"), ("beta_sandwiches", "sandwich")):
        if fit[key] is None:
            continue
        x, y = fit[key].cpu().numpy().reshape(G, -1), np.asarray(ref[want]).reshape(G, -1)
        scale = np.maximum(np.abs(y).max(axis=1, keepdims=True), 1e-12)
        err = np.abs(x - y) / scale
        assert np.all(np.isfinite(err)) and err.max() <= 1e-8, (key, err.max())
