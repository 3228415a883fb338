"""The work a user of devil_amd has it do, as cases that can be timed and checked.

A case is one pass through the public entry points of ``devil_amd``:

  fit       fit_devil followed by test_de (a differential-expression run)
  many      fit_devil_many over several independent problems
  sandwich  compute_sandwich (HC0, or clustered with patients)
  de        test_de of a kept fit (another contrast on the same fit)
  prep      calculate_sf and group_data (a count matrix made ready for a fit)

Designs and counts are drawn as in ``devil_amd.synth``: an intercept, a 0/1
condition or a three-level factor, standard normal covariates; negative
binomial counts with size factors LogNormal(0, 0.3) and one overdispersion per
gene.  ``exact`` gives the same results from plain torch / numpy in 64 bits.
"""
import math
from itertools import combinations_with_replacement

import numpy as np
import torch

import devil_amd

DEVICE = torch.device("cuda", 0)


def listed():
    return [
        # a gene panel looked at interactively: launches and host time count
        dict(name="panel", kind="fit", G=64, n=2000, p=2, counts="int32", od="MOM",
             precision="fp64", patients=0, host=False),
        # the two-group comparison of a small experiment
        dict(name="two_groups", kind="fit", G=2000, n=5000, p=2, counts="int32", od="MOM",
             precision="fp64", patients=0, host=False),
        # an R session's matrix: doubles in host memory, an odd number of cells
        dict(name="host_doubles", kind="fit", G=3000, n=4001, p=4, counts="float64", od="MOM",
             precision="fp64", patients=0, host=True),
        # sparse counts with the Cox-Reid likelihood overdispersion
        dict(name="mle", kind="fit", G=4000, n=20000, p=4, counts="int32", od="MLE",
             precision="fp64", patients=0, host=False),
        # a selection of genes over an atlas: a factor and covariates over 500000 cells
        dict(name="atlas_fp64", kind="fit", G=4000, n=500000, p=8, counts="int32", od="MOM",
             precision="fp64", patients=0, host=False),
        # the same over a whole transcriptome (40 GB of counts) in mixed precision
        dict(name="atlas_mixed", kind="fit", G=20000, n=500000, p=8, counts="int32", od="MOM",
             precision="mixed", patients=0, host=False),
        # a cohort of 40 patients, cluster-robust errors, rows of odd length
        dict(name="cohort_mixed", kind="fit", G=3000, n=310683, p=6, counts="int32", od="MOM",
             precision="mixed", patients=40, host=False),
        # a small cohort with float32 counts (an AnnData layer) in 64 bits
        dict(name="cohort_fp64", kind="fit", G=1500, n=30001, p=5, counts="float32", od="MOM",
             precision="fp64", patients=8, host=False),
        # one fit per cell type: uneven problems in one call
        dict(name="cell_types", kind="many", G=1000, problems=12, n_min=500, n_max=50000,
             counts="int32", od="MOM", precision="fp64"),
        # robust errors for a fit that was made without patients
        dict(name="sandwich_hc0", kind="sandwich", G=2000, n=20000, p=5, counts="int32",
             patients=0),
        # a further contrast on a kept clustered fit of a whole transcriptome
        dict(name="contrast", kind="de", G=20000, n=100000, p=4, patients=40),
        # size factors and grouping by patient before a fit
        dict(name="prepare_counts", kind="prep", G=2000, n=50000, counts="float32",
             method="normed_sum", patients=24),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["fit"] * 6 + ["many", "sandwich", "de", "prep"])
    if kind == "de":
        return dict(kind="de", G=_log_int(rng, 64, 30000), n=_log_int(rng, 500, 500000),
                    p=rng.randint(2, 10), patients=rng.choice([0, 12]))
    if kind == "many":
        return dict(kind="many", G=_log_int(rng, 200, 2000), problems=rng.randint(3, 16),
                    n_min=500, n_max=_log_int(rng, 2000, 40000),
                    counts=rng.choice(["int32", "float32"]), od="MOM", precision="fp64")
    n = _log_int(rng, 700, 400000)
    G = _log_int(rng, 16, max(64, min(20000, int(4e8) // n)))
    counts = rng.choice(["int32", "int32", "int32", "float32", "float64"])
    if kind == "prep":
        return dict(kind="prep", G=max(G, 500), n=min(n, 100000), counts=counts,
                    method=rng.choice(["normed_sum", "psinorm"]), patients=rng.randint(2, 40))
    if kind == "sandwich":
        return dict(kind="sandwich", G=G, n=n, p=rng.randint(2, 10), counts=counts,
                    patients=rng.choice([0, rng.randint(3, 24)]))
    # mixed precision is asked for over whole transcriptomes
    large = G >= 2000 and n >= 8000 and counts != "float64"
    precision = "mixed" if large and rng.random() < 0.7 else "fp64"
    return dict(kind="fit", G=G, n=n, p=rng.randint(2, 10), counts=counts,
                od="MLE" if precision == "fp64" and rng.random() < 0.3 else "MOM",
                precision=precision, patients=rng.choice([0, 0, rng.randint(3, 40)]),
                host=G * n < 3e7 and rng.random() < 0.25)


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _design(r, n, p):
    """[1, condition, covariates], or for p >= 8 [1, two level indicators, covariates]."""
    if p >= 8:
        lvl = r.integers(0, 3, n)
        cols = [np.ones(n), lvl == 1, lvl == 2] + [r.normal(size=n) for _ in range(p - 3)]
    else:
        cols = [np.ones(n), r.uniform(size=n) < 0.5] + [r.normal(size=n) for _ in range(p - 2)]
    return np.column_stack(cols).astype(np.float64)


def _patient_sizes(r, n, patients):
    cut = np.sort(r.choice(np.arange(1, n), patients - 1, replace=False))
    return np.diff(np.concatenate([[0], cut, [n]]))


def _counts(gen, X, sf, B, size, patient=None, dtype=torch.int32):
    """G x n negative binomial counts on the GPU, in gene chunks."""
    G, n = B.shape[0], X.shape[0]
    Y = torch.empty((G, n), dtype=dtype, device=DEVICE)
    Xf = torch.as_tensor(X, dtype=torch.float32, device=DEVICE)
    ls = torch.as_tensor(np.log(sf), dtype=torch.float32, device=DEVICE)
    step = max(1, int(2e8) // n)
    for g in range(0, G, step):
        b, a = B[g:g + step], size[g:g + step, None]
        lin = b @ Xf.T + ls
        if patient is not None:
            effect = torch.randn((b.shape[0], int(patient[-1]) + 1), generator=gen, device=DEVICE)
            lin += (0.3 * effect)[:, patient]
        rate = torch._standard_gamma(a.expand(-1, n).contiguous(), generator=gen)
        rate.div_(a).mul_(lin.exp_())
        Y[g:g + step] = torch.poisson(rate, generator=gen).to(dtype)
    return Y


def _problem(seed, G, n, p, counts, od="MOM", patients=0):
    """Design, size factors, patient labels and counts of one fit."""
    r = np.random.Generator(np.random.Philox(seed))
    gen = torch.Generator(device=DEVICE)
    gen.manual_seed(seed)
    X = _design(r, n, p)
    # sparse counts where the likelihood overdispersion is fitted
    mean, sd = (-1.5, 1.0) if od == "MLE" else (0.0, 1.0)
    levels = 2 if p >= 8 else 1
    B = torch.randn((G, p), generator=gen, device=DEVICE)
    scale = [sd] + [0.5] * levels + [0.1] * (p - 1 - levels)
    B = B * torch.tensor(scale, device=DEVICE)
    B[:, 0] = (B[:, 0] + mean).clamp(-4.0, 3.0)
    size = torch.randn(G, generator=gen, device=DEVICE).exp()
    sf = np.exp(r.normal(0, 0.3, n))
    label = patient = None
    if patients:
        label = np.repeat(np.arange(patients), _patient_sizes(r, n, patients))
        patient = torch.as_tensor(label, device=DEVICE)
    Y = _counts(gen, X, sf, B, size, patient, getattr(torch, counts))
    return dict(Y=Y, X=X, sf=sf, label=label, B=B, size=size)


def _contrast(p):
    c = np.zeros(p)
    c[1] = 1.0
    return c


def _many_shapes(case, seed):
    r = np.random.Generator(np.random.Philox(seed + 7))
    u = r.uniform(np.log(case["n_min"]), np.log(case["n_max"]), case["problems"])
    return [(int(round(math.exp(v))), 2 + j % 9) for j, v in enumerate(u)]


def prepare(case, seed):
    kind = case["kind"]
    if kind == "many":
        return dict(case=case, problems=[
            _problem(1000 * seed + j, case["G"], n, p, case["counts"], case["od"])
            for j, (n, p) in enumerate(_many_shapes(case, seed))])
    if kind == "de":
        G, n, p = case["G"], case["n"], case["p"]
        gen = torch.Generator(device=DEVICE)
        gen.manual_seed(seed)
        rand = lambda *s: torch.randn(*s, generator=gen, device=DEVICE, dtype=torch.float64)

        def cov():  # covariance matrices of the size a fit of n cells has
            W = rand(G, p, p + 4)
            return W @ W.transpose(1, 2) / ((p + 4) * float(n))

        # half of the genes unchanged, effects of up to ~10 standard errors in the others
        beta = rand(G, p) * (3.0 / math.sqrt(n))
        beta[: G // 2] *= 0.33
        fit = dict(beta=beta, beta_sandwiches_null=cov(),
                   beta_sandwiches=cov() if case["patients"] else None,
                   design_matrix=torch.ones((n, p), dtype=torch.float64, device=DEVICE))
        return dict(case=case, fit=fit)
    if kind == "prep":
        p = 3
        s = _problem(seed, case["G"], case["n"], p, case["counts"])
        r = np.random.Generator(np.random.Philox(seed + 3))
        s["label"] = r.integers(0, case["patients"], case["n"])
        return dict(case=case, **s)
    s = _problem(seed, case["G"], case["n"], case["p"], case["counts"], case.get("od", "MOM"),
                 case["patients"])
    if kind == "sandwich":
        s["theta"] = 1.0 / s["size"].double()
        s["beta"] = s["B"].double()
    elif case["host"]:
        s["Y"] = s["Y"].cpu().numpy()
    else:  # what a program on the GPU keeps there beside the counts
        s["Xd"] = torch.as_tensor(s["X"], device=DEVICE)
        s["sfd"] = torch.as_tensor(s["sf"], device=DEVICE)
    return dict(case=case, **s)


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
def _fit_outputs(fit):
    out = {k: fit[k] for k in ("beta", "overdispersion", "beta_sandwiches_null",
                               "beta_sandwiches", "status")}
    out["beta_iters"] = fit["iterations"]["beta_iters"]
    return out


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "many":
        fits = devil_amd.fit_devil_many(
            [dict(x=s["Y"], design_matrix=s["X"], size_factors=s["sf"])
             for s in state["problems"]],
            overdispersion=case["od"], precision=case["precision"])
        return [{k: f[k] for k in ("beta", "overdispersion", "beta_sandwiches_null")}
                for f in fits]
    if kind == "de":
        res = devil_amd.test_de(state["fit"], _contrast(case["p"]))
        return {k: res[k] for k in ("pval", "adj_pval", "lfc", "log_pval")}
    if kind == "prep":
        sf = devil_amd.calculate_sf(state["Y"], case["method"])
        grouped = devil_amd.group_data(state["Y"], state["X"], state["label"])
        return dict(sf=sf, counts=grouped["input_matrix"], design=grouped["design_matrix"],
                    clusters=grouped["clusters"])
    if kind == "sandwich":
        return devil_amd.compute_sandwich(state["X"], state["Y"], state["beta"], state["theta"],
                                          state["sf"], clusters=state["label"])
    fit = devil_amd.fit_devil(
        state["Y"], state["X"] if case["host"] else state["Xd"], clusters=state["label"],
        overdispersion=case["od"], size_factors=state["sf"] if case["host"] else state["sfd"],
        precision=case["precision"])
    res = devil_amd.test_de(fit, _contrast(case["p"]))
    return dict(_fit_outputs(fit), **{k: res[k] for k in ("pval", "adj_pval", "lfc", "log_pval")})


def work(case):
    """Counts and design read once, results written once; operations of the
    contractions over the cells, with eight IRLS rounds per gene."""
    kind = case["kind"]
    if kind == "many":
        parts = [work(dict(case, kind="fit", n=n, p=p, patients=0))
                 for n, p in _many_shapes(case, 1)]
        return {k: sum(w[k] for w in parts) for k in ("bytes", "flops")}
    G, n = case["G"], case["n"]
    if kind == "de":
        p, mats = case["p"], 2 if case["patients"] else 1
        return dict(bytes=8.0 * G * (p + mats * p * p + 4), flops=2.0 * G * mats * p * p)
    es = 8 if case["counts"] == "float64" else 4
    if kind == "prep":
        return dict(bytes=2.0 * es * G * n, flops=1.0 * G * n)
    p = case["p"]
    mats = 2 if case["patients"] else 1
    cols = p * (p + 1) // 2
    passes = 1 if kind == "sandwich" else 8
    return dict(bytes=1.0 * es * G * n + 8.0 * n * (p + 1) + 8.0 * G * (p + mats * p * p),
                flops=2.0 * G * n * passes * (2 * p + cols))


# ---------------------------------------------------------------------------
# the same in 64 bits, from the definitions
# ---------------------------------------------------------------------------
_BLOCK = 2048


def _padded(v):
    """v with zero rows up to a multiple of _BLOCK rows."""
    return torch.nn.functional.pad(v, (0, 0, 0, -v.shape[0] % _BLOCK))


def _over_cells(a, b):
    """a (genes x cells) times b (cells x columns), blocks of cells summed last."""
    a = torch.nn.functional.pad(a, (0, b.shape[0] - a.shape[1]))
    nb = b.shape[0] // _BLOCK
    return torch.bmm(a.view(-1, nb, _BLOCK).transpose(0, 1),
                     b.view(nb, _BLOCK, b.shape[1])).sum(0)


def _pairs(X):
    p = X.shape[1]
    ab = list(combinations_with_replacement(range(p), 2))
    return ab, _padded(torch.stack([X[:, a] * X[:, b] for a, b in ab], dim=1))


def _sym(cols, ab, p):
    A = cols.new_empty((cols.shape[0], p, p))
    for j, (a, b) in enumerate(ab):
        A[:, a, b] = cols[:, j]
        A[:, b, a] = cols[:, j]
    return A


def _exact_sandwich(y, mu, X, ab, K, theta, ends=None, hc0=False):
    n, p = X.shape
    den = 1.0 + theta[:, None] * mu
    H = _sym(_over_cells(((y * theta[:, None] + 1.0) * mu) / (den * den), K), ab, p)
    bread = torch.linalg.inv_ex(H)[0]
    if ends is None and not hc0:
        return bread, None
    r = (y - mu) / den
    if hc0:
        meat = _sym(_over_cells(r * r, K), ab, p) / n
    else:
        C = len(ends)
        starts = [0] + [int(e) for e in ends[:-1]]
        S = torch.stack([_over_cells(r[:, a:int(b)], _padded(X[a:int(b)]))
                         for a, b in zip(starts, ends)], dim=1)
        meat = S.transpose(1, 2) @ S * ((C / (C - 1.0) if C > 1 else 1.0) / n)
    return bread, (bread @ meat @ bread) * n


def _exact_fit(s, od, patients):
    X = torch.as_tensor(s["X"], device=DEVICE)
    sf = torch.as_tensor(s["sf"], device=DEVICE)
    off = torch.log(sf)
    n, p = X.shape
    ab, K = _pairs(X)
    Q, R = torch.linalg.qr(X)
    Q, Xb = _padded(Q), _padded(X)
    Y = s["Y"] if torch.is_tensor(s["Y"]) else torch.as_tensor(s["Y"], device=DEVICE)
    ends = None
    if patients:
        lab = s["label"]
        ends = np.concatenate([np.flatnonzero(lab[1:] != lab[:-1]) + 1, [n]])
    eps = float(np.float32(1e-3))
    G = Y.shape[0]
    out = dict(beta=torch.empty((G, p), dtype=torch.float64, device=DEVICE),
               overdispersion=torch.empty(G, dtype=torch.float64, device=DEVICE),
               beta_sandwiches_null=torch.empty((G, p, p), dtype=torch.float64, device=DEVICE),
               beta_sandwiches=None if ends is None else torch.empty(
                   (G, p, p), dtype=torch.float64, device=DEVICE))
    step = max(1, int(1.5e8) // n)
    for g in range(0, G, step):
        y = Y[g:g + step].double()
        m = y.mean(1)
        var = ((y - m[:, None]) ** 2).sum(1) / (n - 1)
        a0 = (var - m / sf.mean()) / (m * m)
        a0 = torch.where(torch.isnan(a0) | (a0 < 0), torch.full_like(a0, 0.01), a0)
        k = (1.0 / a0.float().double()).float().double()  # k is a float in the reference
        beta = torch.linalg.solve_triangular(R, _over_cells(torch.log1p(y / sf), Q).T, upper=True).T
        beta = beta.contiguous()
        act = torch.arange(y.shape[0], device=DEVICE)
        ya = y
        for _ in range(200):
            ka = k[act, None]
            w = torch.exp(-(beta[act] @ X.T) - off)
            mw = (ka + ya) / (1.0 + ka * w) * w
            A = _sym(_over_cells(mw, K), ab, p) * ka[:, :, None]
            d = torch.linalg.solve_ex(A, ka * _over_cells(mw - 1.0, Xb))[0]
            beta[act] += d
            big = d.abs()
            nan = torch.isnan(big).any(1)
            keep = nan | ~(torch.nan_to_num(big, nan=0.0).amax(1) < eps)
            keep &= ~torch.isnan(d[:, 0])
            if not bool(keep.all()):
                act, ya = act[keep], ya[keep]
            if act.numel() == 0:
                break
        del ya
        mu = sf * torch.exp(beta @ X.T)
        num, den = ((y - mu) ** 2 - mu).sum(1), (mu * mu).sum(1)
        th = torch.where(den > 0, (n / (n - p) * num / den).clamp(min=0.0), torch.zeros_like(den))
        out["beta"][g:g + step] = beta
        out["overdispersion"][g:g + step] = th
        if od == "MOM":
            b, sw = _exact_sandwich(y, mu, X, ab, K, th, ends)
            out["beta_sandwiches_null"][g:g + step] = b
            if sw is not None:
                out["beta_sandwiches"][g:g + step] = sw
    return out


def _log_t_tail(t, df):
    """log of 2 P(T_df > |t|) = log I_x(df/2, 1/2), x = df / (df + t^2), by the
    continued fraction (DLMF 8.17.22, modified Lentz) and, for log B(df/2, 1/2),
    the asymptotic series of the gamma quotient."""
    a, b = 0.5 * df, 0.5
    t = np.abs(t)
    x, y = df / (df + t * t), t * t / (df + t * t)
    lx, ly = -np.log1p(t * t / df), 2 * np.log(t) - math.log(df) - np.log1p(t * t / df)
    ia = 1.0 / a
    quot = 0.5 * math.log(a) - ia / 8 + ia**3 / 192 - ia**5 / 640 + 17 * ia**7 / 14336
    front = a * lx + b * ly - (0.5 * math.log(math.pi) - quot)

    def frac(a, b, x):
        c, d = np.ones_like(x), 1.0 / (1.0 - (a + b) * x / (a + 1.0))
        h = d.copy()
        for m in range(1, 20000):
            for q in (m * (b - m) * x / ((a - 1.0 + 2 * m) * (a + 2 * m)),
                      -(a + m) * (a + b + m) * x / ((a + 2 * m) * (a + 1.0 + 2 * m))):
                d = 1.0 / (1.0 + q * d)
                c = 1.0 + q / c
                h = h * d * c
            if np.all(np.abs(d * c - 1.0) < 1e-16):
                break
        return h

    out = np.empty_like(x)
    low = x < (a + 1.0) / (a + b + 2.0)
    if low.any():
        out[low] = front[low] + np.log(frac(a, b, x[low])) - math.log(a)
    if (~low).any():
        out[~low] = np.log1p(-np.exp(front[~low] + np.log(frac(b, a, y[~low])) - math.log(b)))
    return out


def _exact_de(beta, bread, sandwich, n):
    c = torch.as_tensor(_contrast(beta.shape[1]), device=DEVICE)
    l = beta @ c
    lps = [_log_t_tail((l.abs() / torch.sqrt(torch.einsum("a,gab,b->g", c, V, c))).cpu().numpy(),
                       n - 2.0) for V in (bread, sandwich) if V is not None]
    lp = np.maximum.reduce(lps)
    pv = np.exp(lp)
    order = np.argsort(-pv, kind="stable")
    m = len(pv)
    adj = np.empty(m)
    adj[order] = np.minimum(1.0, np.minimum.accumulate(m / np.arange(m, 0, -1.0) * pv[order]))
    return dict(pval=pv, adj_pval=adj, log_pval=lp,
                lfc=(l / math.log(2.0)).clamp(-10.0, 10.0).cpu().numpy())


def exact(case, seed):
    kind = case["kind"]
    if kind == "fit" and case["G"] * case["n"] > 2.5e9:
        return None  # minutes of work
    s = prepare(case, seed)
    if kind == "many":
        return [_exact_fit(q, case["od"], 0) for q in s["problems"]]
    if kind == "de":
        f = s["fit"]
        return _exact_de(f["beta"], f["beta_sandwiches_null"], f["beta_sandwiches"], case["n"])
    if kind == "prep":
        Y = s["Y"].double()
        if case["method"] == "normed_sum":
            v = Y.sum(0)
        else:
            v = torch.log1p(Y)
            v = v.mean(0) - v.amin(0)
        return dict(sf=v / torch.exp(torch.log(v).mean()), counts=None, design=None,
                    clusters=None)
    if kind == "sandwich":
        X = torch.as_tensor(s["X"], device=DEVICE)
        sf = torch.as_tensor(s["sf"], device=DEVICE)
        n, p = X.shape
        ab, K = _pairs(X)
        ends = None
        if case["patients"]:
            lab = s["label"]
            ends = np.concatenate([np.flatnonzero(lab[1:] != lab[:-1]) + 1, [n]])
        out = torch.empty((case["G"], p, p), dtype=torch.float64, device=DEVICE)
        step = max(1, int(1.5e8) // n)
        for g in range(0, case["G"], step):
            y = s["Y"][g:g + step].double()
            mu = sf * torch.exp(s["beta"][g:g + step] @ X.T)
            out[g:g + step] = _exact_sandwich(y, mu, X, ab, K, s["theta"][g:g + step], ends,
                                              hc0=ends is None)[1]
        return out
    f = _exact_fit(s, case["od"], case["patients"])
    if case["od"] == "MOM":
        de = _exact_de(f["beta"], f["beta_sandwiches_null"], f["beta_sandwiches"], case["n"])
    else:  # the likelihood's overdispersion is where its driver stops, not a closed value
        f.update(overdispersion=None, beta_sandwiches_null=None, beta_sandwiches=None)
        l = f["beta"] @ torch.as_tensor(_contrast(case["p"]), device=DEVICE)
        de = dict(pval=None, adj_pval=None, log_pval=None,
                  lfc=(l / math.log(2.0)).clamp(-10.0, 10.0).cpu().numpy())
    return dict(f, status=None, beta_iters=None, **de)
