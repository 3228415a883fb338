"""The FP64 IRLS of one gene per workgroup (kernels_gene.hip) against the
oracle, at the edges of its thread strides, its workgroup sizes, its design
rule and its design widths, with and without an intercept.

Bars: those of the FP64 path (test_gpu_parity.py): identical iteration counts,
beta within 1e-8 relative (floor 1e-6): an FP64 sum over n <= 1e5 cells in any
order is within n * 2^-53 ~ 1e-11 of another, and the iteration contracts.
"""
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


def problem(G, n, p, intercept=True, dtype=np.int32, seed=0):
    r = np.random.default_rng(1000 + 17 * n + p + seed)
    first = np.ones(n) if intercept else 0.5 + r.uniform(size=n)
    X = np.column_stack([first] + [r.normal(size=n) for _ in range(p - 1)])
    if intercept and p >= 3:
        X[:, 1] = r.uniform(size=n) < 0.5
    B = np.column_stack([r.normal(0.5, 0.5, G)] + [r.normal(0, 0.1, G) for _ in range(p - 1)])
    sf = np.exp(r.normal(0, 0.3, n))
    size = np.exp(r.normal(0.5, 0.5, G))[:, None]
    mu = sf * np.exp(B @ X.T)
    Y = r.poisson(r.gamma(size, mu / size)).astype(dtype)
    return Y, X, sf


def check(dv, orc, Y, X, sf, **kw):
    print(f"[case] G={Y.shape[0]} n={Y.shape[1]} p={X.shape[1]} {Y.dtype} {kw}", flush=True)
    fit = dv.fit_devil(torch.as_tensor(Y, device="cuda"), X, size_factors=sf,
                       overdispersion=False, **kw)
    ref = orc.cpu_fit(Y.astype(np.float64), X, np.log(sf), od_mode=orc.OD_NONE, n_threads=8, **kw)
    np.testing.assert_array_equal(fit["iterations"]["beta_iters"].cpu().numpy(),
                                  ref["beta_iters"])
    b = fit["beta"].cpu().numpy()
    err = np.abs(b - ref["beta"]) / np.maximum(np.abs(ref["beta"]), 1e-6)
    assert np.all(np.isfinite(err)) and err.max() <= 1e-8, err.max()


@pytest.mark.parametrize("n", [40, 255, 256, 257, 511, 512, 513, 1023, 1281, 16384, 16385, 16897])
def test_cell_strides(dv, orc, n):
    check(dv, orc, *problem(20, n, 3))


@pytest.mark.parametrize("intercept", [True, False])
@pytest.mark.parametrize("p", range(1, 11))
def test_design_widths(dv, orc, p, intercept):
    check(dv, orc, *problem(24, 1500 + p, p, intercept))


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_count_types(dv, orc, dtype):
    check(dv, orc, *problem(24, 3001, 4, dtype=dtype))


@pytest.mark.parametrize("p", [2, 5, 10])
@pytest.mark.parametrize("over", [0, 1])
def test_both_sides_of_the_design_rule(dv, orc, p, over):
    """8 (p + 1) n bytes of design at and just above 2 MiB: the gene kernel
    and the round kernels."""
    check(dv, orc, *problem(40, (2 << 20) // (8 * (p + 1)) + over, p))


def test_iteration_limit(dv, orc):
    check(dv, orc, *problem(30, 700, 3), max_iter=1)
    check(dv, orc, *problem(30, 700, 3), max_iter=3)


def test_more_genes_than_workgroups(dv, orc):
    check(dv, orc, *problem(5000, 300, 2))


@pytest.mark.parametrize("p,intercept", [(2, True), (3, False), (6, True), (8, False), (10, True)])
@pytest.mark.parametrize("G", [1, 5, 96, 97, 200])
def test_round_kernels(dv, orc, G, p, intercept):
    """Rows too long for the gene kernel: one gene per wavefront up to 96
    active genes, 16-gene tiles above."""
    Y, X, sf = problem(G, (2 << 20) // (8 * (p + 1)) + 77, p, intercept)
    check(dv, orc, Y, X, sf)


def test_design_setup(dv, orc):
    """The design's QR and its equal columns, found on the device: all nine
    indicators of a factor beside an intercept are rank deficient; with eight of
    them (54 candidates, many equal or zero), with products among the columns
    and with nearly collinear columns the fit is the oracle's."""
    r = np.random.default_rng(5)
    n, G = 4000, 20
    lv = r.integers(0, 9, n)
    X = np.column_stack([np.ones(n)] + [lv == k for k in range(9)]).astype(float)
    Y = r.poisson(np.exp(0.5 + 0.1 * lv) * r.gamma(2.0, 0.5, (G, n))).astype(np.int32)
    sf = np.exp(r.normal(0, 0.2, n))
    with pytest.raises(Exception, match="rank deficient"):
        dv.fit_devil(torch.as_tensor(Y, device="cuda"), X, size_factors=sf)
    check(dv, orc, Y, np.ascontiguousarray(X[:, :9]), sf)
    g = (lv > 4).astype(float)
    h = (lv % 2).astype(float)
    Xd = np.column_stack([np.ones(n), g, h, g * h])
    check(dv, orc, Y, Xd, sf)
    z = r.normal(size=n)
    Xc = np.column_stack([np.ones(n), z, z + 1e-3 * r.normal(size=n)])
    fit = dv.fit_devil(torch.as_tensor(Y, device="cuda"), Xc, size_factors=sf,
                       overdispersion=False)
    ref = orc.cpu_fit(Y.astype(np.float64), Xc, np.log(sf), od_mode=orc.OD_NONE)
    # the condition number 2e3 enters the normal equations squared: 4e6 * 2^-53
    np.testing.assert_allclose(fit["beta"].cpu().numpy(), ref["beta"], rtol=1e-8, atol=1e-8)
