"""The work that users of this framework have it do, as cases that can be timed and compared.

A case is one call of a public entry point on inputs that a program has in hand: a whole
MCI.integrate (calibration, decorrelation, sampling, estimation, combine), a submission of batched
integrals, a run of the learned proposal's chain, or a stretch of its network's training.  The
chains of one seed are the same chains whenever they are run, so two versions of the framework can
be compared on the numbers they return.
"""
import math

import numpy as np
import torch

from mcintegratorplusplus_amd import MCI, BatchIntegrals, constants as K, mixture_workload
from mcintegratorplusplus_amd.learned import INDEP_FP32, MIXED_FP32, LearnedProposalSampler, mixture_target

NDECORR = 1000  # decorrelation steps where a case sets them (0: the automatic decorrelation)


def integral(name, walkers, steps, ndim, **how):
    """A whole integrate.  block: 1 stores every step (the default accumulator), more sums blocks.
    target: independent Gaussians of widths U(0.5, 2), the isotropic exp(-|x|^2), exp(-sum |x_i|), or a
    mixture of three Gaussians in a periodic box.  observe: x_i^2, and |x|^2, exp(-|x|^2/d) or 1[x_0 > 0]."""
    c = dict(name=name, kind="integral", walkers=walkers, steps=steps, ndim=ndim, streams="reference", move="all",
             coupling="shared", target="gauss", block=1, observe="x2", precision="f64", ndecorr=0)
    c.update(how)
    return c


def listed():
    return [
        # one walker with the reference's defaults: what a program written for the reference does
        # unchanged, and the smallest call (one lane: latency)
        integral("one walker, defaults", 1, 16384, 3, target="iso", coupling="independent"),
        # a quick estimate on one wave: launches, round trips and a step's latency
        integral("64 walkers, native", 64, 1280, 16, streams="native", move="single", block=20, observe="x2+sum", ndecorr=NDECORR),
        # the benchmark's workload
        integral("benchmark", 65536, 10240, 16, streams="native", move="single", block=160, observe="x2+sum", ndecorr=NDECORR),
        # the precision form: FP32 chain, 64 dimensions, the most walkers
        integral("fp32, d=64", 262144, 10240, 64, streams="native", move="single", block=160, observe="x2+exp",
                 precision="f32", ndecorr=NDECORR),
        # the benchmark's workload on the reference's random streams (reproducing its chains)
        integral("reference streams", 65536, 10240, 16, move="single", block=160, observe="x2+sum", ndecorr=NDECORR),
        # the default move beyond sixteen dimensions, odd sizes throughout
        integral("all-coordinate, d=50", 20011, 2560, 50, streams="native", block=40, ndecorr=NDECORR),
        # the reference's defaults for many walkers, as MPI ranks sharing their statistics ...
        integral("defaults, shared", 65536, 4096, 16),
        # ... and as independent integrators (the default coupling)
        integral("defaults, independent", 65536, 4096, 16, coupling="independent"),
        # a target and a domain outside the specialised kernels: the chain that runs any plugin
        integral("mixture in a box", 16384, 2048, 6, streams="native", target="mixture", block=32, observe="x2+ind", ndecorr=NDECORR),
        # many small integrals at once
        dict(name="batch of 4096", kind="batch", integrals=4096, nmc=100000, dmax=128),
        # the learned proposal: the chain that mixes in independence moves from the trained mixture
        dict(name="learned chain", kind="learned", mode="independence", walkers=65536, steps=10240, ndim=32, comps=8),
        # the training of its network (forward, backward, Adam)
        dict(name="training", kind="training", walkers=16384, iters=100, batch=4096, ndim=32, comps=8),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """Another case of the ranges that the listed ones stand for."""
    c = _drawn(rng)
    c.pop("name", None)
    return c


def _drawn(rng):
    kind = rng.choice(["defaults", "defaults", "native single", "native all", "fp32", "reference single", "generic", "batch", "learned", "training"])
    if kind == "defaults":
        return integral("", _log_int(rng, 1, 32768), rng.choice([512, 1024, 2048, 4096]), rng.randint(1, 24), target=rng.choice(["gauss", "gauss", "iso"]),
                        coupling=rng.choice(["shared", "independent"]))
    if kind in ("native single", "native all", "fp32"):
        single = kind != "native all"
        blocks, block = rng.choice([16, 32, 64]), _log_int(rng, 10, 160 if single else 80)
        return integral("", _log_int(rng, 64, 131072 if single else 50000), blocks * block, _log_int(rng, 2, 64), streams="native",
                        move="single" if single else "all", block=block, observe=rng.choice(["x2", "x2+sum", "x2+exp"]),
                        precision="f32" if kind == "fp32" else "f64", ndecorr=_log_int(rng, 100, 1000))
    if kind == "reference single":
        block = _log_int(rng, 10, 160)
        return integral("", _log_int(rng, 64, 65536), 64 * block, rng.choice([2, 4, 8, 16, 32, 64]), move="single", block=block,
                        observe=rng.choice(["x2", "x2+sum"]), ndecorr=_log_int(rng, 100, 1000))
    if kind == "generic":
        block = _log_int(rng, 8, 32)
        return integral("", _log_int(rng, 64, 16384), 64 * block, rng.randint(2, 10), streams=rng.choice(["native", "reference"]),
                        move=rng.choice(["all", "single"]), target=rng.choice(["mixture", "mixture", "exp"]), block=block,
                        observe=rng.choice(["x2", "x2+ind"]), ndecorr=_log_int(rng, 100, 1000))
    if kind == "batch":
        return dict(kind="batch", integrals=_log_int(rng, 64, 4096), nmc=_log_int(rng, 5000, 100000), dmax=rng.randint(8, 128))
    if kind == "learned":
        return dict(kind="learned", mode=rng.choice(["independence", "independence", "conditional"]), walkers=_log_int(rng, 4096, 65536),
                    steps=64 * _log_int(rng, 16, 80), ndim=rng.choice([8, 16, 24, 32]), comps=rng.randint(2, 8))
    return dict(kind="training", walkers=8192, iters=_log_int(rng, 20, 200), batch=rng.choice([1024, 2048, 4096]),
                ndim=rng.choice([8, 16, 32]), comps=rng.randint(2, 8))


BOX = 8.0  # the mixture's periodic box is [-8, 8]^d


def _widths(case, rng):
    return rng.uniform(0.5, 2.0, case["ndim"])


def _mixture(case, rng):
    """three isotropic components: weights, widths, means"""
    w = rng.dirichlet(np.full(3, 3.0))
    return w, rng.uniform(0.7, 1.5, 3), rng.normal(0.0, 2.0, (3, case["ndim"]))


def prepare(case, seed):
    rng = np.random.default_rng(seed)
    if case["kind"] == "batch":
        ndim, nmc, w, s, mu, _ = mixture_workload(n=case["integrals"], seed=seed, dmax=case["dmax"], nmc_range=(1e3, case["nmc"]))
        b = BatchIntegrals(ndim, nmc, w, s, mu)
        b.setSeed(seed)
        return case, b
    if case["kind"] in ("learned", "training"):
        s = LearnedProposalSampler(*mixture_target(d=case["ndim"], ncomp=case["comps"], seed=seed)[:3], case["walkers"])
        s.setSeed(seed)
        s.setTrainingPairs(0.0)
        s.setFixedInput(case.get("mode") == "independence")
        s.collect(8, 256)
        s.initFromSamples(60)
        return case, s
    d = case["ndim"]
    m = MCI(d, case["walkers"])
    m.setSeed(seed)
    m.setRandomMode(K.RNG_MT19937_64 if case["streams"] == "reference" else K.RNG_PHILOX)
    m.setPrecision(K.PREC_FP32 if case["precision"] == "f32" else K.PREC_FP64)
    m.setWalkerCoupling(K.COUPLING_SHARED if case["coupling"] == "shared" else K.COUPLING_INDEPENDENT)
    m.setTrialMove(K.SRRD_UNIFORM, 1 if case["move"] == "single" else 0, 1)
    if case["ndecorr"]:
        m.setNdecorrelationSteps(case["ndecorr"])
    if case["target"] == "gauss":
        m.addSamplingFunction(K.PDF_GAUSS_DIAG, 0.5 / _widths(case, rng) ** 2)
    elif case["target"] == "exp":
        m.addSamplingFunction(K.PDF_EXP_DIAG, 1.0 / _widths(case, rng))
    elif case["target"] == "iso":
        m.addSamplingFunction(K.PDF_GAUSS_ISO)
    else:
        w, s, mu = _mixture(case, rng)
        m.setIRange(-BOX, BOX)
        m.addSamplingFunction(K.PDF_GMM_ISO, np.concatenate([[3.0], w, s, mu.ravel()]))
    block = case["block"]
    if block == 1:  # addObservable's own defaults: every step kept, correlated errors
        for kind in _observables(case):
            m.addObservable(kind)
    else:
        for kind in _observables(case):
            m.addObservable(kind, (), block, 1, True, estimator=K.ESTIM_MJBLOCKER)
    return case, m


def _observables(case):
    return [{"x2": K.OBS_X2, "sum": K.OBS_X2_SUM, "exp": K.OBS_EXP_X2, "ind": K.OBS_INDICATOR}[o] for o in case["observe"].split("+")]


def _nobs(case):
    return case["ndim"] + len(case["observe"].split("+")) - 1


def run(state):
    case, h = state
    if case["kind"] == "integral":
        avg, err = h.integrate(case["steps"])
        return {"average": avg, "error": err}
    if case["kind"] == "batch":
        avg, err = h.run()
        return {"average": avg, "error": err}
    if case["kind"] == "learned":
        avg, err = h.run(INDEP_FP32 if case["mode"] == "independence" else MIXED_FP32, case["steps"], 64, 0.5)
        return {"average": avg, "error": err}
    first, last = h.train(case["iters"], case["batch"], 1e-3)
    return {"loss": np.array([first, last]), "weights": h.network().params()}


def work(case):
    """bytes: the walkers' positions and generators in and out, stored traces or block means out.
    flops: an integral's chain at the cost of its move, its test and its sums; no generator."""
    if case["kind"] == "batch":
        lo, hi = math.log(1e3), math.log(case["nmc"])
        steps = case["integrals"] * (case["nmc"] - 1e3) / (hi - lo)  # the mean of a log-uniform draw
        return {"bytes": steps / 512 * 16 * 8, "flops": 26.0 * steps}
    if case["kind"] == "learned":
        n, d, k = case["walkers"] * case["steps"], case["ndim"], case["comps"]
        net = 2 * (d * 128 + 128 * 128 + 128 * 8 * (1 + 2 * d)) if case["mode"] == "conditional" else 0
        return {"bytes": 8.0 * case["walkers"] * (d + 2 * 64), "flops": 0.5 * n * (2 * k * d * d + 8 * k * d + net) + 0.5 * n * 4 * k * d}
    if case["kind"] == "training":
        d = case["ndim"]
        par = d * 128 + 128 * 128 + 128 * 8 * (1 + 2 * d)
        return {"bytes": case["iters"] * (16.0 * par + 8.0 * case["batch"] * d), "flops": 6.0 * par * case["batch"] * case["iters"]}
    W, n, d, no = case["walkers"], case["steps"], case["ndim"], _nobs(case)
    rows = n if case["block"] == 1 else n // case["block"]
    gen = 2 * 2500 if case["streams"] == "reference" else 16
    per = 9 + no if case["move"] == "single" else 8 * d + no
    if case["target"] == "mixture":
        per += 3 * 3 * d
    total = n + (case["ndecorr"] or max(100, int(math.sqrt(40000 * d))))
    return {"bytes": W * (16.0 * d + gen + 8.0 * rows * no), "flops": 1.0 * per * W * total}


def tolerance(case):
    """Chains whose decisions are those of the same arithmetic differ only by the rounding of their
    block sums: 1e-15 of an average; a combined error moves by far less than 1e-6 unless a walker's
    blocking test falls the other way.  The learned chain decides in 32 bits on matrix-core sums:
    another order of those sums takes other decisions here and there, and the averages and error bars
    then agree as two runs do (an error bar of W walkers to about 1 / sqrt(2 W)).  The weights after
    some Adam steps on 16-bit gradients agree to a few parts in a thousand."""
    if case["kind"] == "learned":
        return {"rel": min(0.03, 4 / math.sqrt(case["walkers"])), "max": min(0.9, 12 / math.sqrt(case["walkers"]))}
    if case["kind"] == "training":
        return {"rel": 0.01, "max": 0.2}
    if case["kind"] == "batch":
        return {"rel": 1e-5, "max": 1e-3}
    return {"rel": 1e-6, "max": 1e-5}


# ---- the native chains again, in 64 bits with torch operations ------------------------------------

M32 = 0xFFFFFFFF


def _philox(c0, c1, c2, c3, seed):
    """Philox4x32-10 on int64 tensors (or numbers) holding 32-bit words"""
    k0, k1 = seed & M32, (seed >> 32) & M32
    for r in range(10):
        p0, p1 = c0 * 0xD2511F53, c2 * 0xCD9E8D57
        c0, c1, c2, c3 = ((p1 >> 32) & M32) ^ c1 ^ k0, p1 & M32, ((p0 >> 32) & M32) ^ c3 ^ k1, p0 & M32
        k0, k1 = (k0 + 0x9E3779B9) & M32, (k1 + 0xBB67AE85) & M32
    return c0, c1, c2, c3


def _chi2_q95(n):
    """0.95 quantiles of chi-squared with 1..n degrees of freedom, by bisection"""
    k = torch.arange(1, n + 1, dtype=torch.float64)
    lo, hi = torch.zeros(n, dtype=torch.float64), torch.full((n,), 200.0, dtype=torch.float64)
    for _ in range(80):
        mid = 0.5 * (lo + hi)
        below = torch.special.gammainc(k / 2, mid / 2) < 0.95
        lo, hi = torch.where(below, mid, lo), torch.where(below, hi, mid)
    return lo


def _blocking_error(y):
    """the automatic blocking of Jonsson (Phys. Rev. E 98, 043304) along the first axis of y [2^p][...]"""
    n, mean = y.shape[0], y.mean(0)
    p = n.bit_length() - 1
    var, m = [], []
    for k in range(p):
        c = y - mean
        v, g = (c * c).mean(0), (c[1:] * c[:-1]).sum(0) / c.shape[0]
        var.append(v)
        m.append(torch.where(v == 0, 0.0, (g / v) ** 2) * 2.0 ** (p - k))  # a constant series passes
        y = 0.5 * (y[0::2] + y[1::2])
    total = torch.cumsum(torch.stack(m[::-1]), 0)
    q = _chi2_q95(p).to(total.device).reshape(-1, *[1] * (total.dim() - 1))
    last = torch.where(total < q, torch.arange(1, p + 1, device=total.device).reshape(q.shape), 0).amax(0)  # kk + 1
    k = torch.clamp(p - last, max=p - 1)
    var = torch.stack(var).gather(0, k[None])[0]
    return mean, torch.sqrt(var / 2.0 ** (p - k))


def _replays(case):
    """The native chains with shared statistics and a fixed decorrelation.  The others have no value that
    plain operations give in reasonable time: the reference streams keep 312 words for each walker,
    a 32-bit or learned chain decides by its own rounding, and a single-coordinate move on a number
    of coordinates that is no power of two draws again now and then."""
    d = case.get("ndim", 0)
    if case["kind"] != "integral" or case["streams"] != "native" or case["precision"] != "f64" or not case["ndecorr"]:
        return False
    if case["move"] == "single" and (case["target"] != "gauss" or d & (d - 1)):
        return False
    width = (d + 2) // 2 if case["move"] == "all" else 1
    return case["target"] in ("gauss", "mixture") and (case["steps"] + 2 * NDECORR) * (1 + case["walkers"] * width / 1.5e5) < 3e4


def exact(case, seed):
    if not _replays(case):
        return None
    rng = np.random.default_rng(seed)
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    W, d, B = case["walkers"], case["ndim"], case["block"]
    single, mix = case["move"] == "single", case["target"] == "mixture"
    m = d.bit_length() - 1 if single else 0
    w = torch.arange(W, device=dev, dtype=torch.int64)
    T = lambda v: torch.tensor(v, device=dev, dtype=torch.float64)  # noqa: E731
    if mix:
        cw, cs, cmu = _mixture(case, rng)
        gc, gb, mu = T(np.log(cw) - d * np.log(cs)), T(0.5 / cs ** 2), T(cmu)

        def logp(x):
            r = torch.stack([((x - mu[k][:, None]) ** 2).sum(0) for k in range(3)])
            return torch.logsumexp(gc[:, None] - gb[:, None] * r, 0)
    else:
        a = T(0.5 / _widths(case, rng) ** 2)

        def logp(x):
            return -(x * x * a[:, None]).sum(0)
    x = torch.zeros((d, W), device=dev, dtype=torch.float64)
    lp = logp(x)
    nblk = 1 if single else (d + 2) // 2
    blk = torch.arange(nblk, device=dev, dtype=torch.int64)[:, None]
    t, words, s = 0, None, 0.05

    def step():
        nonlocal x, lp, t, words
        if t % 2 == 0 or words is None:
            words = _philox(blk + 0 * w, w + 0 * blk, torch.full((nblk, W), t // 2, device=dev, dtype=torch.int64), 0 * w, seed)
        odd = t % 2
        wa, wb = words[2 * odd], words[2 * odd + 1]  # main words 2 j and 2 j + 1 of the step
        shared = wa[0]
        low = _philox(torch.full((W,), 0x30000000, device=dev, dtype=torch.int64), w, torch.full_like(w, t), 0 * w, seed)[0]
        u = ((((shared << 32) | low) << m) >> 11 & ((1 << 53) - 1)).to(torch.float64) * 2.0 ** -53
        if single:
            j = (shared >> (32 - m)) if m else 0 * w
            r = (2 * wb[0] + 1 - (1 << 32)).to(torch.float64) * 2.0 ** -32
            xo = x.gather(0, j[None])[0]
            xn = xo + s * r
            aj = a[j]
            ratio = xn * xn * aj - xo * xo * aj
            acc = u <= torch.exp(-ratio)
            x = x.scatter(0, j[None], torch.where(acc, xn, xo)[None])
        else:
            v = torch.stack([wa, wb], 1).reshape(2 * nblk, W)[1:d + 1]
            xn = x + s * ((2 * v + 1 - (1 << 32)).to(torch.float64) * 2.0 ** -32)
            if mix:
                xn = torch.where(xn < -BOX, xn + 2 * BOX, xn)
                xn = torch.where(xn > BOX, xn - 2 * BOX, xn)
            ln = logp(xn)
            acc = u <= torch.exp(ln - lp)
            x, lp = torch.where(acc, xn, x), torch.where(acc, ln, lp)
        t += 1
        return acc

    # the shared step calibration: 50 % acceptance within 5 % five times running, at most 50 rounds
    hits = rounds = 0
    n = int(max(100.0, math.sqrt(40000.0 * d) / W))
    while hits < 5 and rounds < 50:
        got = torch.zeros(W, device=dev, dtype=torch.float64)
        for _ in range(n):
            got += step()
        rate = float((got / n).mean())
        hits = hits + 1 if abs(rate - 0.5) < 0.05 else 0
        s *= min(2.0, max(0.5, rate / 0.5))
        if mix:
            s = min(s, BOX)
        rounds += 1
    for _ in range(case["ndecorr"]):
        step()
    obs = case["observe"].split("+")
    blocks = []
    for _ in range(case["steps"] // B):
        acc = torch.zeros((_nobs(case), W), device=dev, dtype=torch.float64)
        for _ in range(B):
            step()
            q = x * x
            rows = [q]
            if "sum" in obs:
                rows.append(q.sum(0)[None])
            if "exp" in obs:
                rows.append(torch.exp(-q.sum(0) / d)[None])
            if "ind" in obs:
                rows.append((x[0] > 0).to(torch.float64)[None])
            acc += torch.cat(rows)
        blocks.append(acc / B)
    avg, err = _blocking_error(torch.stack(blocks))
    return {"average": avg.mean(1).cpu().numpy(), "error": (torch.sqrt((err * err).sum(1)) / W).cpu().numpy()}
