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
