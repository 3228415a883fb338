"""The init and post-IRLS passes on the short cell ranges of fits with few
genes, and the t tail of test_de, against the oracle.

Bars: those of the FP64 path (test_gpu_parity.py), theta / bread / sandwich
within 1e-8 relative.  The t tail's continued fraction loses up to about
df * 2^-53 (its partial sums cancel to 1 / df of their terms), on both sides:
log p within 1e-12 + 4e-16 df."""
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


def close(a, b, what):
    a, b = np.asarray(a.cpu()), np.asarray(b)
    scale = np.abs(b).reshape(len(b), -1).max(1).reshape((-1,) + (1,) * (b.ndim - 1))
    err = np.abs(a - b) / np.maximum(scale, 1e-12)
    assert np.all(np.isfinite(err)) and err.max() <= 1e-8, f"{what}: {err.max():.2e}"


@pytest.mark.parametrize("G,sizes", [
    (16, None), (17, None), (1, None), (300, None),
    (16, [1, 15, 16, 17, 127, 128, 129, 2067]),  # patients shorter than a block and a range
    (40, [5, 2400, 95])])
def test_short_ranges(dv, orc, G, sizes):
    r = np.random.default_rng(G)
    n = 2500 if sizes is None else sum(sizes)
    X = np.column_stack([np.ones(n), r.uniform(size=n) < 0.5, r.normal(size=n)])
    B = np.column_stack([r.normal(1, 0.5, G), r.normal(0, 0.5, G), r.normal(0, 0.1, G)])
    sf = np.exp(r.normal(0, 0.3, n))
    mu = sf * np.exp(B @ X.T)
    Y = r.poisson(r.gamma(2.0, mu / 2.0)).astype(np.int32)
    lab = None if sizes is None else np.repeat(np.arange(len(sizes)), sizes)
    ends = None if sizes is None else np.cumsum(sizes).astype(np.int32)
    print(f"[case] G={G} n={n} patients={sizes}", flush=True)
    fit = dv.fit_devil(torch.as_tensor(Y, device="cuda"), X, size_factors=sf, clusters=lab)
    ref = orc.cpu_fit(Y.astype(np.float64), X, np.log(sf), od_mode=orc.OD_MOM,
                      clusters_ends=ends)
    np.testing.assert_array_equal(fit["iterations"]["beta_iters"].cpu(), ref["beta_iters"])
    close(fit["beta"], ref["beta"], "beta")
    close(fit["overdispersion"], ref["theta"], "theta")
    close(fit["beta_sandwiches_null"], ref["bread"], "bread")
    if sizes is not None:
        close(fit["beta_sandwiches"], ref["sandwich"], "sandwich")


@pytest.mark.parametrize("n", [3, 20, 500, 5000, 100000])
def test_t_tail(dv, orc, n):
    t = np.concatenate([np.exp(np.linspace(-12, 6, 600)), [0.0, 1.0, 1.8, 2.0]])
    G = len(t)
    one = np.ones((G, 1, 1))
    fit = dict(beta=t[:, None], beta_sandwiches_null=one, design_matrix=np.ones((n, 1)))
    lp = dv.test_de(fit, [1.0])["log_pval"]
    ref = orc.de_test(t[:, None], one, None, n, [1.0])["log_pval"]
    err = np.abs(lp - ref) / np.maximum(1.0, np.abs(ref))
    print(f"[case] t tail df={n - 2} worst {err.max():.2e}", flush=True)
    assert np.all(np.isfinite(err)) and err.max() <= 1e-12 + 4e-16 * n


@pytest.mark.parametrize("extra", [0, 1, 2, 3])
@pytest.mark.parametrize("patients", [0, 3])
def test_vector_columns(dv, orc, extra, patients):
    """Designs of 16 + extra distinct columns of products (and of two): a last
    tile of one or two columns is summed by vector instructions, in the IRLS
    rounds, the bread, the score sums and the HC0 meat."""
    r = np.random.default_rng(extra)
    G, n = 130, 45000
    # 1, b1..bk 0/1 columns, z: distinct columns 1 + k + k (k - 1) / 2 + 1 + k + 1
    if extra == 0:
        X = np.column_stack([np.ones(n), r.uniform(size=n) < 0.5])  # 2 columns
    elif extra == 1:  # 3 indicators of one factor (products zero), 4 covariates: 1+3+4+12+10
        lv = r.integers(0, 4, n)
        X = np.column_stack([np.ones(n), lv == 1] + [r.normal(size=n) for _ in range(4)])[:, :6]
        X[:, 5] = lv == 2  # 1 2 3 z1..z3: 18 columns
    elif extra == 2:
        X = np.column_stack([np.ones(n), r.uniform(size=n) < 0.5] +
                            [r.normal(size=n) for _ in range(6)])  # 33 columns or more
        X[:, 2] = (r.uniform(size=n) < 0.3) & (X[:, 1] == 0)
    else:
        X = r.normal(size=(n, 5)) + 0.2  # 20 columns, no intercept
    X = X.astype(np.float64)
    p = X.shape[1]
    B = np.column_stack([r.normal(0.7, 0.3, G)] + [r.normal(0, 0.1, G) for _ in range(p - 1)])
    sf = np.exp(r.normal(0, 0.3, n))
    mu = sf * np.exp(np.clip(B @ X.T, -4, 4))
    Y = r.poisson(r.gamma(2.0, mu / 2.0)).astype(np.int32)
    lab = np.sort(r.integers(0, patients, n)) if patients else None
    ends = None if lab is None else np.cumsum(np.bincount(lab)).astype(np.int32)
    print(f"[case] vector columns p={p} extra={extra} patients={patients}", flush=True)
    Yd = torch.as_tensor(Y, device="cuda")
    fit = dv.fit_devil(Yd, X, size_factors=sf, clusters=lab)
    ref = orc.cpu_fit(Y.astype(np.float64), X, np.log(sf), od_mode=orc.OD_MOM,
                      clusters_ends=ends, n_threads=8)
    np.testing.assert_array_equal(fit["iterations"]["beta_iters"].cpu(), ref["beta_iters"])
    close(fit["beta"], ref["beta"], "beta")
    close(fit["beta_sandwiches_null"], ref["bread"], "bread")
    if patients:
        close(fit["beta_sandwiches"], ref["sandwich"], "sandwich")
    else:
        b, th = fit["beta"].cpu().numpy(), fit["overdispersion"].cpu().numpy()
        sw = dv.compute_sandwich(X, Yd, b, th, sf)
        want = []
        for g in range(0, G, 13):
            h = orc.compute_hessian(b[g], th[g], Y[g].astype(float), X, sf)
            m = orc.meat_hc0(X, Y[g].astype(float), b[g], th[g], sf)
            want.append(h @ m @ h * n)
        close(sw[::13], np.array(want), "HC0")


@pytest.mark.parametrize("dtype", [np.int32, np.float32, np.float64])
def test_init_large_counts(dv, orc, dtype):
    """Counts on both sides of 2^14 in one block, and zeros: the init pass takes
    its short form only for whole blocks below."""
    r = np.random.default_rng(3)
    G, n = 40, 2100
    X = np.column_stack([np.ones(n), r.normal(size=n)])
    sf = np.exp(r.normal(0, 0.3, n))
    Y = r.poisson(sf * r.gamma(3.0, 2.0, (G, n))).astype(dtype)
    Y[:, ::97] = 16383
    Y[:, 50::97] = 16384
    Y[:5, 100::301] = 2_000_000
    print(f"[case] large counts {Y.dtype}", flush=True)
    fit = dv.fit_devil(torch.as_tensor(Y, device="cuda"), X, size_factors=sf, max_iter=3)
    ref = orc.cpu_fit(Y.astype(np.float64), X, np.log(sf), od_mode=orc.OD_MOM, max_iter=3)
    close(fit["beta"], ref["beta"], "beta")
    close(fit["overdispersion"], ref["theta"], "theta")


@pytest.mark.parametrize("n", [64, 67])
def test_exponential_table(dv, n):
    """exp over its range, by the MOM overdispersion of zero counts with an
    intercept: theta = n / (n - 1) (1 - 1 / mu), mu = exp(beta).  Table entries
    on both sides of a rounding edge (odd multiples of ln2 / 512) and far ones.
    Tolerance: sums of n equal terms and exp's two ulps, relative to 1 + 1 / mu."""
    from devil_amd import _lib as L
    ln2 = np.log(2.0)
    x = np.concatenate([ln2 / 512 * np.arange(1, 2048), np.linspace(5, 350, 500),
                        ln2 / 256 * np.array([255, 256, 257, 511, 512, 100000])])
    G, lib, ctx = len(x), L.lib(), L.context(0)
    Y = torch.zeros((G, n), dtype=torch.int32, device="cuda")
    one, off = (torch.full((n,), v, dtype=torch.float64, device="cuda") for v in (1.0, 0.0))
    th = torch.empty(G, dtype=torch.float64, device="cuda")
    b = torch.as_tensor(x, device="cuda")
    torch.cuda.synchronize()
    ctx.check(lib.devil_mom_dispersion(ctx.h, Y.data_ptr(), L.COUNTS_I32, G, n, n,
                                       one.data_ptr(), 1, b.data_ptr(), off.data_ptr(),
                                       th.data_ptr()))
    want = n / (n - 1) * -np.expm1(-x)
    err = np.abs(th.cpu().numpy() - want) / (1 + np.exp(-x))
    print(f"[case] exp table n={n}: {err.max():.2e}", flush=True)
    assert err.max() <= (n + 16) * 2.0**-53 * n / (n - 1)
