"""The design set-up on the device (kernels_design.hip) at the edge of the
double range, and the outputs of a fit that fails."""
from fractions import Fraction

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


@pytest.mark.parametrize("cells", [(0,), (63, 700), (1999,)])
def test_overflowing_size_factor(dv, cells):
    """exp(offset) = inf in some cells: the mean size factor is infinite, so
    alpha0 = var / mean^2 = n (n s2 - s1^2) / ((n - 1) s1^2)
    (R/overdispersion.R:129-135).  The sums of integer counts are exact; seven
    roundings follow, each within 2^-53."""
    from devil_amd import _lib as L
    r = np.random.default_rng(7)
    G, n = 20, 2000
    Y = r.poisson(r.gamma(2.0, 1.5, (G, n))).astype(np.int32)
    off = r.normal(0, 0.3, n)
    off[list(cells)] = 800.0
    print(f"[case] overflowing size factors at {cells}", flush=True)
    Yd, offd = torch.as_tensor(Y, device="cuda"), torch.as_tensor(off, device="cuda")
    a = torch.empty(G, dtype=torch.float64, device="cuda")
    ctx = dv.context(0)
    torch.cuda.synchronize()
    ctx.check(dv.lib().devil_estimate_dispersion(ctx.h, Yd.data_ptr(), L.COUNTS_I32, G, n, n,
                                                 offd.data_ptr(), a.data_ptr()))
    for g in range(G):
        s1, s2 = int(Y[g].sum()), int((Y[g].astype(np.int64) ** 2).sum())
        want = float(Fraction(n * (n * s2 - s1 * s1), (n - 1) * s1 * s1))
        assert abs(a[g].item() - want) <= 8 * 2.0**-53 * want, (g, a[g].item(), want)


def test_failing_fit_leaves_outputs(dv):
    """A fit that runs out of device memory after its IRLS (the MLE's table of
    32 KB a gene does not fit) leaves the caller's device outputs as they were."""
    import ctypes as C
    from devil_amd import _lib as L
    G = torch.cuda.mem_get_info()[1] // 32768 + 500_000
    print(f"[case] failing fit of {G} genes", flush=True)
    lib = dv.lib()
    Y = torch.randint(0, 9, (G, 2), dtype=torch.int32, device="cuda")
    X, off = (torch.full((2,), v, dtype=torch.float64, device="cuda") for v in (1.0, 0.0))
    f = {k: torch.full((G,), -7.0, dtype=torch.float64, device="cuda")
         for k in ("beta", "theta", "bread")}
    i = {k: torch.full((G,), -7, dtype=torch.int32, device="cuda")
         for k in ("beta_iters", "theta_iters", "status")}
    prob = L.Problem(mem=L.MEM_DEVICE, counts=Y.data_ptr(), counts_dtype=L.COUNTS_I32,
                     counts_ld=2, X=X.data_ptr(), offset=off.data_ptr(), G=G, n=2, p=1,
                     init_mode=L.INIT_QR, od_mode=L.OD_MLE, max_iter=5, tolerance=1e-3,
                     precision=L.PREC_FP64)
    outs = L.Outputs(**{k: v.data_ptr() for k, v in {**f, **i}.items()})
    ctx = L.Context(0)
    torch.cuda.synchronize()
    rc = lib.devil_fit(ctx.h, C.byref(prob), C.byref(outs), 1)
    message = lib.devil_last_error(ctx.h)
    ctx.close()
    try:  # HIP keeps the allocation's error for the next launch check: torch's
        torch.full((1,), 1.0, device="cuda").add_(1.0)
    except RuntimeError:
        pass
    torch.cuda.synchronize()
    assert rc == 3 and b"hipMalloc" in message, (rc, message)
    for k, v in {**f, **i}.items():
        assert bool((v == -7).all()), k
