"""The work whose speed this repository is measured by.

A case is a dict of plain values whose "kind" says which public entry points
it goes through:

* ``chains``: `Batch.run` on chains in their steady state (or, with
  ``burn_in``, on chains that still adapt and train their learned
  proposals), the sampler itself;
* ``load``: a dataset from its packed .bed body to a batch that is ready to
  iterate (`Ctx`, `Batch`, `setup`);
* ``scan``: X^T R of every SNP for residuals on the device;
* ``rb``: the Rao-Blackwellised inclusion probabilities of every SNP for a
  caller-held model, host vectors in and out;
* ``band``: X^T X of every SNP with its neighbours (LD);
* ``model``: a caller that keeps its own sampler and moves only the linear
  model to the device, one call per term.

`listed` holds one case per use, `draw` gives others of the same ranges,
`prepare` makes what a program holds before the call, `run` is one pass and
`exact` the same results in float64 from torch and numpy alone.
"""
import math

import numpy as np
import torch

import bmagwa_amd
from bmagwa_amd import synth

LD = (0.7, 0.95, 20, 100)       # AR(1) blocks: rho range, length range
DO_N_ITER = 200000              # sizes the chains' sample buffers


def listed():
    return [
        # The reference's own example: n = 1,000, p = 10,000, two covariates,
        # two chains, delayed rejection up to moves of 10.  The smallest runs
        # that people start, alone on the GPU.
        dict(name="chains_example", kind="chains", n=1000, p=10000, chains=2, causal=10, h2=0.3, types="A", m_e=2,
             dr=10, learned=0, burn_in=False, n_rao=500, iters=500, datasets=1, max_size=0),
        # A study with dominance effects: two columns per SNP.
        dict(name="chains_dominance", kind="chains", n=5000, p=100000, chains=8, causal=50, h2=0.4, types="AH", m_e=0,
             dr=0, learned=0, burn_in=False, n_rao=500, iters=500, datasets=1, max_size=100),
        # The benchmark: 16 chains with both learned proposals, burn-in over.
        dict(name="chains_16", kind="chains", n=10000, p=500000, chains=16, causal=100, h2=0.5, types="A", m_e=0,
             dr=0, learned=3, burn_in=False, n_rao=500, iters=500, datasets=1, max_size=200),
        # The same dataset with a chain on every compute unit.  (Models are
        # limited to 200 SNPs, as at the largest sizes: without a limit some
        # chains of some datasets outgrow the device's 256 columns.)
        dict(name="chains_256", kind="chains", n=10000, p=500000, chains=256, causal=100, h2=0.5, types="A", m_e=0,
             dr=0, learned=3, burn_in=False, n_rao=500, iters=500, datasets=1, max_size=200),
        # Several phenotypes, each measured on its own part of a pool of
        # individuals, in one batch.
        dict(name="chains_phenotypes", kind="chains", n=20000, p=100000, chains=64, causal=40, h2=0.4, types="A", m_e=0,
             dr=0, learned=0, burn_in=False, n_rao=500, iters=500, datasets=4, max_size=100),
        # Models of up to 200 SNPs: past the columns that fit the LDS.
        dict(name="chains_wide", kind="chains", n=20000, p=100000, chains=16, causal=200, h2=0.6, types="A", m_e=0,
             dr=0, learned=0, burn_in=False, n_rao=250, iters=250, datasets=1, max_size=200),
        # Burn-in: adaptation, labels and a training round of both networks
        # after every all-SNP scan.
        dict(name="chains_burn_in", kind="chains", n=10000, p=200000, chains=16, causal=60, h2=0.5, types="A", m_e=0,
             dr=0, learned=3, burn_in=True, n_rao=250, iters=250, datasets=1, max_size=150),
        # What every run begins with: the .bed body of a study to a batch
        # ready to iterate.
        dict(name="load", kind="load", n=10000, p=100000, chains=4, causal=50),
        # One genotype pass for three residual vectors at the benchmark size.
        dict(name="scan_wide", kind="scan", n=10000, p=500000, vectors=3, digits=5, coding=0),
        # One Rao-Blackwellised scan for a caller-held model of odd sizes.
        dict(name="rb", kind="rb", n=4973, p=99991, loci=40),
        # LD windows of 500 SNPs.
        dict(name="band", kind="band", n=10000, p=200000, width=500, coding_a=0, coding_b=0),
        # The latency of single model updates: a rejected and an accepted
        # move of a few terms on a model of 60.
        dict(name="model", kind="model", n=10000, p=20000, loci=60, removes=3, adds=3),
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["chains", "chains", "chains", "load", "scan", "rb", "band", "model"])
    n, p = _log_int(rng, 500, 20000), _log_int(rng, 5000, 500000)
    if kind == "chains":
        types = rng.choice(["A", "A", "A", "AH", "D"])
        n_rao = rng.choice([100, 250, 500])
        p = min(p, 4 * 10 ** 9 // n)
        causal = _log_int(rng, 5, min(n // 40, 50 if types == "AH" else 100))
        return dict(kind=kind, n=n, p=p, chains=_log_int(rng, 1, 64), causal=causal, h2=round(rng.uniform(0.2, 0.6), 3),
                    types=types, m_e=rng.choice([0, 0, 1, 3]), dr=rng.choice([0, 0, 6, 10]),
                    learned=rng.choice([0, 0, 3]) if types == "A" else 0, burn_in=False, n_rao=n_rao, iters=n_rao,
                    datasets=1, max_size=2 * causal)
    if kind == "load":
        return dict(kind=kind, n=n, p=min(p, 10 ** 9 // n), chains=_log_int(rng, 1, 16), causal=_log_int(rng, 5, 100))
    if kind == "scan":
        digits = rng.choice([4, 5])
        return dict(kind=kind, n=n, p=min(p, 5 * 10 ** 9 // n), vectors=rng.randint(1, 3), digits=digits,
                    coding=rng.choice([0, 0, 1, 2, 3]))
    if kind == "rb":
        return dict(kind=kind, n=n, p=min(p, 2 * 10 ** 9 // n), loci=_log_int(rng, 2, 120))
    if kind == "band":
        width = _log_int(rng, 8, 560)
        return dict(kind=kind, n=n, p=max(2000, min(p, 10 ** 12 // (n * width), 10 ** 8 // width)), width=width,
                    coding_a=rng.randint(0, 3), coding_b=rng.randint(0, 3))
    return dict(kind=kind, n=n, p=min(p, 10 ** 8 // n), loci=_log_int(rng, 5, 140), removes=rng.randint(0, 4),
                adds=rng.randint(1, 4))


# ------------------------------------------------------------- inputs -----
def _body(n, p, seed):
    """Packed .bed body (p x ceil(n / 4) bytes) of independent SNPs with
    MAF ~ U(0.02, 0.5), made on the GPU: codes 0, 2 and 3 stand for 0, 1 and
    2 minor alleles, the first individual of a byte in its lowest bits."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    stride = (n + 3) // 4
    out = torch.empty((p, stride), dtype=torch.uint8)
    maf = torch.rand(p, generator=gen, device="cuda") * 0.48 + 0.02
    cut = (maf * 256).round().to(torch.uint8)
    shift = torch.tensor([1, 4, 16, 64], dtype=torch.uint8, device="cuda")
    rows = max(1, min(p, (1 << 28) // (8 * stride)))
    for j in range(0, p, rows):
        c = cut[j:j + rows, None]
        u = torch.randint(0, 256, (2, len(c), 4 * stride), generator=gen, dtype=torch.uint8, device="cuda")
        g = (u[0] < c).to(torch.uint8) + (u[1] < c).to(torch.uint8)
        g[:, n:] = 0
        code = (g + (g > 0)).view(len(c), stride, 4)
        out[j:j + rows] = (code * shift).sum(-1, dtype=torch.uint8).cpu()
    return out.numpy()


def _values(body, n, coding):
    """Genotype values of packed rows (on the GPU) in float64."""
    b = torch.as_tensor(body).cuda()
    code = torch.stack([(b >> s) & 3 for s in (0, 2, 4, 6)], dim=-1).reshape(len(b), -1)[:, :n]
    table = torch.tensor([[0., 0., 1., 2.], [0., 0., 1., 0.], [0., 0., 1., 1.], [0., 0., 0., 1.]],
                         dtype=torch.float64, device="cuda")[coding]
    return table[code.long()]


def _phenotype(body, n, causal, seed):
    """y = X beta + e for `causal` random SNPs that explain half of it."""
    rng = np.random.default_rng(seed)
    snps = np.sort(rng.choice(len(body), size=min(causal, len(body)), replace=False))
    x = _values(body[snps], n, 0).cpu().numpy()
    g = rng.normal(size=len(snps)) @ x
    return g + rng.normal(scale=max(g.std(), 1e-3), size=n)


def _residuals(case, seed):
    rng = np.random.default_rng(seed + 1)
    return rng.normal(size=(case["vectors"], case["n"])) * rng.uniform(0.2, 5.0, size=(case["vectors"], 1))


def _sampler_cfgs(case, seed, n_of, burnin):
    return [synth.sampler_cfg(n_of[c], case["p"], case["causal"], types=case.get("types", "A"), seed=seed % 100003 + c,
                              chain=c, m_e=case.get("m_e", 0), delay_rejection=case.get("dr", 0),
                              n_rao=case.get("n_rao", 500), n_rao_burnin=burnin, do_n_iter=DO_N_ITER)
            for c in range(case["chains"])]


def _chain_data(case, seed):
    """The datasets of a chains case and the dataset of every chain."""
    n, p = case["n"], case["p"]
    types = (case["types"],)
    thresh, rho, _ = synth.snp_layout(p, (0.02, 0.5), LD, seed)
    pool = bmagwa_amd.Ctx(n, p, synth=(seed % (1 << 31), thresh, rho), types=types)
    rng = np.random.default_rng(seed)

    def decode(snps):
        return pool.decode(np.asarray(snps), 0)

    if case["datasets"] == 1:
        y, _, _ = synth.phenotype(decode, n, p, case["causal"], case["h2"], seed, dominance=types == ("AH",))
        pool.set_y(y)
        if case["m_e"]:
            pool.set_covariates(rng.normal(size=(n, case["m_e"])))
        return [pool], [0] * case["chains"]
    ctxs = []
    for k in range(case["datasets"]):
        m = int(round(n * 10 ** (-k / max(1, case["datasets"] - 1)))) - k
        sub = np.sort(rng.choice(n, size=m, replace=False)).astype(np.uint32)
        y, _, _ = synth.phenotype(lambda s: decode(s)[:, sub], m, p, case["causal"], case["h2"], seed + k)
        ctxs.append(bmagwa_amd.Ctx.subset(pool, sub, y, types=types))
    pool.close()
    return ctxs, [c % case["datasets"] for c in range(case["chains"])]


def _prepare_chains(case, seed):
    ctxs, chain_ctx = _chain_data(case, seed)
    n_rao = case["n_rao"]
    burnin = 10 ** 6 if case["burn_in"] else max(2, 2000 // n_rao)
    cfgs = _sampler_cfgs(case, seed, [ctxs[k].n for k in chain_ctx], burnin)
    # thinned loci kept per chain: DO_N_ITER / 10 samples of up to ~2.5 times
    # the expected model, less for many chains (they make fewer passes)
    samples = DO_N_ITER // 10
    loci = samples * (int(2.5 * case["causal"]) + 20) // max(1, case["chains"] // 16)
    batch = bmagwa_amd.Batch(ctxs, chain_ctx, cfgs,
                             dict(proposal=case["learned"], use_graph=1, trace_capacity=loci,
                                  max_model_size=case["max_size"], learn_every=n_rao))
    batch.setup()
    # into the steady state: past the burn-in's adaptation and its last
    # all-SNP scan (or, for a burn-in case, past the growth of the empty
    # model)
    batch.run(6 * n_rao if case["burn_in"] else (burnin + 1) * n_rao)
    return dict(batch=batch)


def _run_chains(case, state):
    b = state["batch"]
    b.run(case["iters"])
    st = [b.state(c) for c in range(b.n_chains)]
    ints = np.array([[int(s["size"]), int(s["n_accepted"]), int(s["n_iter"]), int(s["loci_len"])] for s in st], np.int64)
    loci = np.full((b.n_chains, 256), -1, np.int64)      # a device model has at most 256 columns
    for c in range(b.n_chains):
        j = b.loci(c)
        loci[c, :len(j)] = j
    out = dict(loci=loci, counts=ints,
               loglik=np.array([s["loglik"] for s in st]), sigma2=np.array([s["sigma2"] for s in st]),
               alpha=np.array([s["alpha"] for s in st]), move_size=np.array([s["p_move_size"] for s in st]))
    if case["burn_in"]:
        out["proposal"] = b.p_proposal(0)
        out["network"] = b.learn_params(0)
    else:
        out["pip"] = b.p_rao(0)
    return out


# ---------------------------------------------------------------- load ----
def _load_inputs(case, seed):
    body = _body(case["n"], case["p"], seed)
    return body, _phenotype(body, case["n"], case["causal"], seed)


def _run_load(case, state):
    ctx = bmagwa_amd.Ctx(case["n"], case["p"], state["body"], state["y"])
    batch = bmagwa_amd.Batch([ctx], [0] * case["chains"], state["cfgs"], dict(use_graph=1))
    batch.setup()
    s = ctx.stats()
    out = dict(moments=ctx.self_moments(), stats=np.array([s["yy"], s["var_y"], s["var_x"], s["mean_x"]]),
               loglik=np.array([batch.state(c)["loglik"] for c in range(case["chains"])]))
    batch.close()
    ctx.close()
    return out


def _exact_load(case, seed):
    n, p = case["n"], case["p"]
    body, y = _load_inputs(case, seed)
    sums = np.empty((p, 2))
    rows = max(1, (1 << 27) // n)
    for j in range(0, p, rows):
        x = _values(body[j:j + rows], n, 0)
        sums[j:j + rows, 0] = x.sum(1).cpu().numpy()
        sums[j:j + rows, 1] = (x * x).sum(1).cpu().numpy()
    s, q = sums[:, 0], sums[:, 1]
    css = q - s * s / n
    yy, sy = float(y @ y), float(y.sum())
    cfg = _sampler_cfgs(case, seed, [n] * case["chains"], 4)[0]
    var_y = (yy - sy * sy / n) / (n - 1)
    s2 = var_y * (1 - cfg["R2mode_sigma2"]) * (cfg["nu_sigma2"] + 2) / cfg["nu_sigma2"]
    d0 = cfg["inv_tau2_e_const_val"]
    ll = (-0.5 * math.log(n + d0)
          - 0.5 * (n + cfg["nu_sigma2"]) * math.log(cfg["nu_sigma2"] * s2 + yy - sy * sy / (n + d0)))
    return dict(moments=np.stack([s, css], 1), stats=np.array([yy, var_y, (css / (n - 1)).mean(), (s / n).mean()]),
                loglik=np.full(case["chains"], ll))


# ---------------------------------------------------------------- scan ----
def _prepare_scan(case, seed):
    n, p = case["n"], case["p"]
    ctx = bmagwa_amd.Ctx(n, p, _body(n, p, seed), np.zeros(n))
    r = torch.zeros((case["vectors"], ctx.n_pad()), dtype=torch.float64, device="cuda")
    r[:, :n] = torch.as_tensor(_residuals(case, seed))
    out = torch.empty((case["vectors"], p), dtype=torch.float64, device="cuda")
    return dict(ctx=ctx, r=r, out=out)


def _run_scan(case, state):
    state["ctx"].scan_xtr_dev(state["r"].data_ptr(), case["vectors"], state["out"].data_ptr(), coding=case["coding"],
                              digits=case["digits"])
    return state["out"]


def _exact_scan(case, seed):
    n, p = case["n"], case["p"]
    body = _body(n, p, seed)
    r = torch.as_tensor(_residuals(case, seed)).cuda()
    out = torch.empty((case["vectors"], p), dtype=torch.float64, device="cuda")
    rows = max(1, (1 << 28) // n)
    for j in range(0, p, rows):
        out[:, j:j + rows] = (_values(body[j:j + rows], n, case["coding"]) @ r.T).T
    return out


# ------------------------------------------------------------ rb, model ---
def _prior_cfg(case, seed):
    return synth.sampler_cfg(case["n"], case["p"], max(10, case["loci"]), seed=seed % 100003, use_individual_tau2=0)


def _terms(case, seed, count):
    """Distinct SNPs and the prior precisions of their effects."""
    rng = np.random.default_rng(seed + 2)
    return rng.choice(case["p"], size=count, replace=False), rng.uniform(20.0, 400.0, size=count)


def _prepare_rb(case, seed):
    n, p = case["n"], case["p"]
    body = _body(n, p, seed)
    ctx = bmagwa_amd.Ctx(n, p, body, _phenotype(body, n, case["loci"], seed))
    model = bmagwa_amd.Model(ctx, cfg=_prior_cfg(case, seed))
    for j, d in zip(*_terms(case, seed, case["loci"])):
        model.add_term(int(j), 0, d)
    model.sample_beta_sigma2()
    model.compute_pve()
    return dict(ctx=ctx, model=model, y_hat=model.beta()[2])


def _prepare_model(case, seed):
    n, p = case["n"], case["p"]
    body = _body(n, p, seed)
    ctx = bmagwa_amd.Ctx(n, p, body, _phenotype(body, n, case["loci"], seed))
    current, proposed = (bmagwa_amd.Model(ctx, cfg=_prior_cfg(case, seed)) for _ in range(2))
    snps, ds = _terms(case, seed, case["loci"] + case["adds"])
    for j, d in zip(snps[:case["loci"]], ds):
        current.add_term(int(j), 0, d)
    proposed.commit_from(current)
    return dict(ctx=ctx, current=current, proposed=proposed, snps=snps[case["loci"]:], ds=ds[case["loci"]:],
                removes=_removals(case))


def _removals(case):
    """Positions removed in turn, spread over the model as it shrinks."""
    k = case["loci"]
    return [min((i + 1) * k // (case["removes"] + 1), k - i - 1) for i in range(case["removes"]) if k - i > 0]


def _run_model(case, state):
    """One rejected move: removals, additions and the way back, then the
    factor of the current model from scratch."""
    cur, new = state["current"], state["proposed"]
    ll = []
    for i in state["removes"]:
        new.remove_term(i)
        ll.append(new.log_likelihood())
    for j, d in zip(state["snps"], state["ds"]):
        new.add_term(int(j), 0, d)
        ll.append(new.log_likelihood())
    new.rollback_from(cur)
    new.compute_log_likelihood()
    ll.append(new.log_likelihood())
    return np.array(ll)


def _exact_model(case, seed):
    n = case["n"]
    body = _body(n, case["p"], seed)
    y = _phenotype(body, n, case["loci"], seed)
    cfg = _prior_cfg(case, seed)
    snps, ds = _terms(case, seed, case["loci"] + case["adds"])
    x = np.concatenate([np.ones((1, n)), _values(body[snps], n, 0).cpu().numpy()])
    d = np.concatenate([[cfg["inv_tau2_e_const_val"]], ds])
    xx, xy, yy = x @ x.T, x @ y, float(y @ y)
    s2 = y.var(ddof=1) * (1 - cfg["R2mode_sigma2"]) * (cfg["nu_sigma2"] + 2) / cfg["nu_sigma2"]

    def loglik(cols):
        c = [0] + [1 + i for i in cols]
        low = np.linalg.cholesky(xx[np.ix_(c, c)] + np.diag(d[c]))
        v = np.linalg.solve(low, xy[c])
        return (0.5 * np.log(d[c[1:]]).sum() - np.log(np.diag(low)).sum()
                - 0.5 * (n + cfg["nu_sigma2"]) * math.log(cfg["nu_sigma2"] * s2 + yy - v @ v))

    cols = list(range(case["loci"]))
    ll = []
    for i in _removals(case):
        del cols[i]
        ll.append(loglik(cols))
    for k in range(case["adds"]):
        cols.append(case["loci"] + k)
        ll.append(loglik(cols))
    ll.append(loglik(list(range(case["loci"]))))
    return np.array(ll)


# ---------------------------------------------------------------- band ----
def _prepare_band(case, seed):
    n, p = case["n"], case["p"]
    ctx = bmagwa_amd.Ctx(n, p, _body(n, p, seed), np.zeros(n))
    out = torch.zeros((p, case["width"]), dtype=torch.int32, device="cuda")
    return dict(ctx=ctx, out=out)


def _run_band(case, state):
    state["ctx"].band_xtx_dev(case["width"], case["coding_a"], case["coding_b"], state["out"].data_ptr())
    return state["out"]


# ----------------------------------------------------------------- all ----
def prepare(case, seed):
    kind = case["kind"]
    if kind == "chains":
        state = _prepare_chains(case, seed)
    elif kind == "load":
        body, y = _load_inputs(case, seed)
        state = dict(body=body, y=y, cfgs=_sampler_cfgs(case, seed, [case["n"]] * case["chains"], 4))
        for cfg in state["cfgs"]:
            cfg["do_n_iter"] = 10000
    else:
        state = {"scan": _prepare_scan, "rb": _prepare_rb, "band": _prepare_band, "model": _prepare_model}[kind](
            case, seed)
    state["case"] = case
    return state


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "chains":
        return _run_chains(case, state)
    if kind == "load":
        return _run_load(case, state)
    if kind == "scan":
        return _run_scan(case, state)
    if kind == "rb":
        return state["model"].rb(state["y_hat"])
    if kind == "band":
        return _run_band(case, state)
    return _run_model(case, state)


def exact(case, seed):
    """In float64 without this package: X^T R, the moments and the empty
    model's likelihood of a loaded dataset, the likelihoods of a caller's
    model.  Chains are draws of a random stream, whose float results no
    other code gives; X^T X is whole numbers."""
    kind = case["kind"]
    if kind == "load":
        return _exact_load(case, seed)
    if kind == "scan":
        return _exact_scan(case, seed)
    if kind == "model":
        return _exact_model(case, seed)
    return None


def work(case):
    n, p = case["n"], case["p"]
    row = (n + 3) // 4
    kind = case["kind"]
    if kind == "chains":
        # the genotypes once for the all-SNP scan, the probabilities it
        # gives; per iteration an addition and a removal in a model of
        # `causal` SNPs: its dot products, solves and rotations
        cols = case["causal"] * (2 if case["types"] == "AH" else 1) + 1
        steps = case["iters"] * case["chains"]
        return dict(bytes=p * row + 16.0 * p * case["chains"] + steps * cols * row,
                    flops=2.0 * n * p * case["chains"] + steps * (4.0 * n * cols + 8.0 * cols * cols))
    if kind == "load":
        return dict(bytes=2.0 * p * row + 16.0 * p, flops=2.0 * n * p)
    if kind == "scan":
        return dict(bytes=p * row + 8.0 * case["vectors"] * (n + p),
                    flops=2.0 * n * p * case["vectors"] * case["digits"])
    if kind == "rb":
        return dict(bytes=p * row + 8.0 * (n + p), flops=2.0 * n * p)
    if kind == "band":
        w = case["width"]
        return dict(bytes=p * row + 4.0 * p * w, flops=2.0 * n * p * w)
    k = case["loci"]
    calls = case["removes"] + case["adds"]
    return dict(bytes=calls * 1.0 * k * row + 8.0 * k * k, flops=calls * (2.0 * n * k + 8.0 * k * k) + k ** 3 / 3)
