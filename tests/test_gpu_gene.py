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


# A workgroup holds two genes (p <= 5) only where the genes outnumber the
# workgroups: 1024 up to 16384 cells, 512 above.  Few cells keep the oracle
# quick; a workgroup's step is 256 (512) cells.
@pytest.mark.parametrize("intercept", [True, False])
@pytest.mark.parametrize("p", [1, 2, 3, 4, 5])
def test_two_genes_side_by_side(dv, orc, p, intercept):
    """Three full steps (the pipeline's two buffers end on the odd one) and a
    partial one."""
    check(dv, orc, *problem(1400, 3 * 256 + 37, p, intercept))


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("n", [200, 256, 512, 4 * 256 + 1])
def test_two_genes_steps_and_count_types(dv, orc, n, dtype):
    """No full step, whole steps only, an even number of steps and a remainder."""
    check(dv, orc, *problem(1100, n, 3, dtype=dtype))


@pytest.mark.parametrize("n,p,intercept", [(16385, 2, True), (16896, 5, False)])
def test_two_genes_in_wide_workgroups(dv, orc, n, p, intercept):
    """512 threads: more than 512 genes, 32 full steps and a remainder, and 33."""
    check(dv, orc, *problem(600, n, p, intercept))


@pytest.mark.parametrize("p", [2, 4])
def test_pairing_does_not_change_bits(dv, p):
    """Which genes share a workgroup depends on timing; a gene's result does not:
    two fits have the same bits, and a gene fitted in a launch of its own (one
    gene per workgroup) has them too."""
    Y, X, sf = problem(1500, 900, p, seed=3)
    Yd = torch.as_tensor(Y, device="cuda")
    fit = lambda y: dv.fit_devil(y, X, size_factors=sf, overdispersion=False,
                                 init_overdispersion=0.7, init_mode="rough")
    print(f"[case] pairing p={p}", flush=True)
    a, b, few = fit(Yd), fit(Yd), fit(Yd[:40])
    for x, y in ((a, b), (a, few)):
        m = y["beta"].shape[0]
        np.testing.assert_array_equal(x["beta"][:m].cpu().numpy(), y["beta"].cpu().numpy())
        np.testing.assert_array_equal(x["iterations"]["beta_iters"][:m].cpu().numpy(),
                                      y["iterations"]["beta_iters"].cpu().numpy())


@pytest.mark.parametrize("sign", [1, -1])
def test_one_step_from_zero_counts(dv, sign):
    """One iteration on zero counts with an intercept is a closed expression of w
    = exp(-beta - off): r = -1 / (1 + k w), A = k (sum r + n), step = sum r / (sum
    r + n) = -1 / (k w) whatever n is.  Offsets over both signs; bar: sum r is
    within n 2^-53 and the reciprocal within 2.2e-15, and sum r + n = n k w / (1 +
    k w) divides both by the cancellation k w / (1 + k w)."""
    from devil_amd import _lib as L
    n, k = 128, 2.0
    b = sign * np.linspace(0.0, 3.0, 700)
    G = len(b)
    Y = torch.zeros((G, n), dtype=torch.int32, device="cuda")
    one, off = (torch.full((n,), v, dtype=torch.float64, device="cuda") for v in (1.0, 0.0))
    beta = torch.as_tensor(b, device="cuda").clone()
    alpha = torch.full((G,), 1.0 / k, dtype=torch.float64, device="cuda")
    it, st = (torch.empty(G, dtype=torch.int32, device="cuda") for _ in range(2))
    ctx = dv.context(0)
    torch.cuda.synchronize()
    ctx.check(dv.lib().devil_beta_fit(ctx.h, Y.data_ptr(), L.COUNTS_I32, G, n, n,
                                      one.data_ptr(), 1, beta.data_ptr(), off.data_ptr(),
                                      alpha.data_ptr(), 1, 1e-3, L.PREC_FP64, it.data_ptr(),
                                      st.data_ptr()))
    step = beta.cpu().numpy() - b
    kw = k * np.exp(-b)
    err = np.abs(step * kw + 1.0)
    # w's error (2 units of 2^-53), the reciprocal's, sum r's and the division's,
    # over the cancellation; the rounding of beta + step against the step
    bar = (2.2e-15 + 12 * 2.0**-53) * (1 + kw) / kw + 4 * 2.0**-53 * (1 + np.abs(b) * kw)
    print(f"[case] one step from zero counts, sign {sign}: {(err / bar).max():.2f} of the bar",
          flush=True)
    assert np.all(err <= bar), (err / bar).max()
