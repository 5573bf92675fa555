"""What the speed of this framework is measured on.

Twelve listed cases, and drawn ones of the same ranges, through the public
Python entry points (`Engine.run`, `Batch.run`, `model_isf` in
deac-cpp_amd/deac_amd.py): single reconstructions from the smoke-test size to
the long-grid workload, the reference command line's default population, the
detailed-balance and single-particle variants, the mixed-precision split loop,
seed batches at FP32 and FP64, an uneven batch over wavevectors at BF16x3, and
the evaluation of a stack of genomes.

Every run has a fixed number of generations (no stop threshold), so a pass
does the same work for every seed.  Inputs are synthetic imaginary-time
correlation functions of a few Gaussian peaks with seeded relative noise, as
in the repository's own benchmark.
"""
import math
import os
import sys

import numpy as np

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "deac-cpp_amd"))

import deac_amd as da  # noqa: E402

TEMPERATURE = 1.35
BETA = 1.0 / TEMPERATURE

# Every case has these; a listed or drawn case overrides what it is about.
DEFAULTS = dict(kind="engine", T=65, G=4096, P=8, N=1001, omega_max=512.0, rel_error=1e-4, model="standard",
                spectra="bfull", zero_temperature=False, renormalize=False, first_moment=False, third_moment=False,
                negative_first_moment=False, precision="fp64", instances=1, wavevectors=1)


def case(**over):
    return dict(DEFAULTS, **over)


def listed():
    return [
        # The smoke-test fixture's size: one short run, all latency and launches.
        case(name="smoke", T=4, G=16, N=200, omega_max=4.0, rel_error=5e-2, spectra="spfsf"),
        # The ordinary single run of a small data set (a laptop-size job of the reference).
        case(name="single_small", T=33, G=512, N=2001, omega_max=64.0, rel_error=1e-3),
        # One reconstruction at production resolution, small population: the plain path's headline.
        case(name="single_large", N=2001),
        # The same with the reference command line's default population of 512.
        case(name="default_population", P=512, N=101),
        # The bosonic detailed-balance build with its -1st-moment term, one seed.
        case(name="detailed_balance", P=32, N=201, spectra="bdsf", negative_first_moment=True),
        # A single-particle spectral function: renormalized every generation, both moments constrained.
        case(name="single_particle", G=2048, P=16, N=201, spectra="spfsf", renormalize=True, first_moment=True,
             third_moment=True),
        # The long-grid workload: many timeslices, long genome, hyperbolic kernel, exact.
        case(name="long_grid", T=257, G=16384, P=64, N=201, model="hyperbolic"),
        # The same with the contraction at FP32 (the split generation loop).
        case(name="long_grid_fp32", T=257, G=16384, P=64, N=601, model="hyperbolic", precision="fp32"),
        # 256 seeds of one problem in one launch, FP32 contraction: the batched headline.
        case(name="seed_batch_fp32", kind="batch", P=32, N=201, precision="fp32", instances=256),
        # The same bit for bit as 256 separate exact runs.
        case(name="seed_batch_fp64", kind="batch", P=32, N=201, instances=256),
        # A sweep over wavevectors: every one with its own grid, timeslices and model, 16 seeds each.
        case(name="uneven_batch", kind="uneven", P=16, N=101, precision="bf16x3", instances=192, wavevectors=12),
        # Scoring a stack of candidate spectra against the data.
        case(name="score_stack", kind="isf", N=1, instances=1024),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _generations(c, most, budget):
    """Generations that keep a drawn case within its listed one's work."""
    per = c["P"] * c["G"] * c["T"] * c["instances"]
    return max(20, min(most, int(budget / per)))


def draw(rng):
    kind = rng.choice(["small", "single", "population", "bdsf", "single_particle", "long", "long", "batch", "batch",
                       "uneven", "isf"])
    models = ["standard", "hyperbolic", "normalization"]
    if kind == "small":
        c = case(T=rng.randint(2, 40), G=_log_int(rng, 5, 700), P=rng.randint(4, 24), omega_max=64.0, rel_error=1e-2,
                 spectra=rng.choice(["spfsf", "bfull"]), zero_temperature=rng.random() < 0.2)
        c["N"] = rng.randint(100, 400)
    elif kind == "single":
        c = case(T=rng.randint(20, 130), G=_log_int(rng, 700, 6000), P=rng.randint(4, 48), model=rng.choice(models[::2]),
                 spectra=rng.choice(["bfull", "ffull"]), zero_temperature=rng.random() < 0.2)
        c["N"] = _generations(c, 1501, 2000 * 8 * 4096 * 65)
    elif kind == "population":
        c = case(T=rng.randint(17, 80), G=_log_int(rng, 500, 4096), P=_log_int(rng, 65, 512))
        c["N"] = _generations(c, 301, 100 * 512 * 4096 * 65)
    elif kind == "bdsf":
        c = case(T=rng.randint(17, 100), G=_log_int(rng, 500, 4200), P=rng.randint(5, 40), spectra="bdsf",
                 model=rng.choice(models[::2]), negative_first_moment=rng.random() < 0.5)
        c["N"] = _generations(c, 301, 200 * 32 * 4096 * 65)
    elif kind == "single_particle":
        c = case(T=rng.randint(17, 80), G=_log_int(rng, 300, 2500), P=rng.randint(5, 24), omega_max=128.0,
                 spectra=rng.choice(["spfsf", "spbsf"]), renormalize=True, first_moment=rng.random() < 0.5,
                 third_moment=rng.random() < 0.5)
        c["N"] = _generations(c, 301, 200 * 16 * 2048 * 65)
    elif kind == "long":
        precision = rng.choice(["fp64", "fp32", "bf16x3"])
        c = case(T=rng.randint(100, 260), G=_log_int(rng, 4000, 16384), P=rng.randint(24, 64), precision=precision,
                 model=rng.choice(models[:2]))
        c["N"] = _generations(c, 401, (200 if precision == "fp64" else 500) * 64 * 16384 * 257)
    elif kind == "batch":
        c = case(kind="batch", T=rng.randint(17, 120), G=_log_int(rng, 500, 4096), P=rng.randint(4, 64),
                 precision=rng.choice(["fp64", "fp32", "bf16x3"]), instances=_log_int(rng, 20, 512),
                 spectra=rng.choice(["bfull", "bfull", "bdsf"]))
        c["instances"] = max(1, min(c["instances"], 256 * 32 // c["P"]))
        c["N"] = _generations(c, 151, 150 * 256 * 32 * 4096 * 65)
    elif kind == "uneven":
        nq = rng.randint(3, 12)
        c = case(kind="uneven", P=rng.choice([7, 8, 13, 16]), precision=rng.choice(["fp64", "fp32", "bf16x3"]),
                 instances=16 * nq, wavevectors=nq, N=rng.randint(40, 100))
    else:
        c = case(kind="isf", T=rng.randint(17, 130), G=_log_int(rng, 500, 4096), N=1, instances=_log_int(rng, 16, 1024),
                 precision=rng.choice(["fp64", "fp32", "bf16x3"]))
    return c


# ------------------------------------------------------------------ inputs


def _gaussian(w, mu, sd):
    return np.exp(-0.5 * ((w - mu) / sd) ** 2) / (sd * np.sqrt(2.0 * np.pi))


def _data(c, rng):
    """tau, isf, error and the moment targets: three peaks on [0, omega_max]."""
    w = np.linspace(0.0, c["omega_max"], 8193)
    x = c["omega_max"] / 512.0
    peaks = [(max(3.0 * x, 0.5), max(0.4 * x, 0.1), 0.5), (20.0 * x, 4.0 * x, 0.3), (60.0 * x, 10.0 * x, 0.2)]
    s = sum(wt * _gaussian(w, mu, sd) for mu, sd, wt in peaks)
    s /= np.trapezoid(s, w)
    single = c["spectra"] in ("spfsf", "spbsf")
    tau = np.linspace(0.0, 0.5 * BETA, c["T"])
    decay = np.exp(-np.outer(tau, w))
    if not c["zero_temperature"] and not single:
        decay = decay + np.exp(-np.outer(BETA - tau, w))
    f = np.trapezoid(s * decay, w, axis=1) * (-1.0 if single else 1.0)
    err = c["rel_error"] * np.abs(f)
    f = f + np.clip(rng.normal(0.0, 1.0, c["T"]), -3.0, 3.0) * err
    moments = (float(np.trapezoid(s * w, w)), float(np.trapezoid(s * w ** 4, w)))
    return tau, f, err, moments


def _problem(c, rng):
    tau, f, err, (first, third) = _data(c, rng)
    over = {}
    if c["first_moment"]:
        over["first_moment"] = first
    if c["third_moment"]:
        over.update(third_moment=third, third_moment_error=0.1 * third)
    return da.make_problem(tau, f, err, np.arange(c["G"]) * (c["omega_max"] / (c["G"] - 1)), TEMPERATURE,
                           model=c["model"], spectra_type=c["spectra"], zero_temperature=c["zero_temperature"],
                           renormalize=c["renormalize"], population_size=c["P"], normalize=True,
                           use_negative_first_moment=c["negative_first_moment"], **over)


def _wavevectors(c):
    """The uneven batch's problems: shapes and models that differ from one wavevector to the next."""
    rng = np.random.default_rng(7919 * c["wavevectors"] + c["P"])
    out = []
    for k in range(c["wavevectors"]):
        zero = k == 3
        out.append(dict(c, T=int(rng.choice([33, 65, 129, 257])), G=int(rng.choice([1024, 2048, 4096, 8192])),
                        omega_max=float(rng.uniform(128.0, 512.0)), zero_temperature=zero,
                        model="standard" if zero or rng.uniform() < 0.5 else "normalization"))
    return out


def _genomes(c, rng):
    """Candidate spectra: positive, smooth on the scale of the grid, with noise."""
    L = c["G"] * (1 if c["zero_temperature"] else 2)
    w = np.tile(np.arange(c["G"]) * (c["omega_max"] / (c["G"] - 1)), L // c["G"])
    out = np.empty((c["instances"], L))
    centre = rng.uniform(0.01, 0.3, c["instances"]) * c["omega_max"]
    for n in range(c["instances"]):
        out[n] = _gaussian(w, centre[n], 0.3 * centre[n] + 1.0)
    out *= 0.9 + 0.2 * rng.random(out.shape, dtype=np.float32)
    return out


def prepare(case, seed):
    """What a program holds before the call: the problem uploaded in its engine or batch, the seeds."""
    c = dict(case)
    rng = np.random.default_rng([c["T"], c["G"], c["P"], seed])
    if c["kind"] == "engine":
        return {"case": c, "engine": da.Engine(_problem(c, rng)), "seed": int(rng.integers(1, 1 << 30))}
    if c["kind"] == "isf":
        return {"case": c, "problem": _problem(c, rng), "genomes": _genomes(c, rng)}
    if c["kind"] == "batch":
        problems = [_problem(c, rng)] * c["instances"]
    else:
        each = c["instances"] // c["wavevectors"]
        problems = [p for q in _wavevectors(c) for p in [_problem(q, rng)] * each]
    first = int(rng.integers(1, 1 << 30))
    return {"case": c, "batch": da.Batch(problems), "seeds": list(range(first, first + c["instances"]))}


# -------------------------------------------------------------------- runs

ARRAYS = ("dsf", "frequency", "mean", "minimum", "squared_mean", "fitness")


def _result(o):
    out = {k: o[k] for k in ARRAYS}
    out.update(minimum_fitness=float(o["minimum_fitness"]), best_index=int(o["best_index"]),
               generation=int(o["generation"]), rng=np.array(o["rng"], dtype=np.uint64).view(np.int64))
    return out


def run(state):
    c = state["case"]
    if c["kind"] == "engine":
        return _result(state["engine"].run(state["seed"], c["N"], 0.0, precision=c["precision"]))
    if c["kind"] == "isf":
        e, chi, _ = da.model_isf(state["problem"], state["genomes"], c["precision"])
        return {"model_isf": e, "chi2": chi}
    outs = [_result(o) for o in state["batch"].run(state["seeds"], c["N"], 0.0, precision=c["precision"])]
    return {k: np.concatenate([np.atleast_1d(o[k]) for o in outs]) for k in outs[0]}


def work(case):
    """Per generation every trial's K.S (and the population, where it does not fit on the chip); once: the kernel
    matrix and the outputs."""
    c = case
    shapes = _wavevectors(c) if c["kind"] == "uneven" else [c]
    each = c["instances"] // len(shapes)
    flops = nbytes = population = 0.0
    for q in shapes:
        L = q["G"] * (1 if q["zero_temperature"] or q["spectra"] == "bdsf" else 2)
        rows = each * (1 if c["kind"] == "isf" else q["P"])
        flops += 2.0 * rows * L * q["T"] * c["N"]
        nbytes += 8.0 * q["T"] * L
        if c["kind"] == "isf":
            nbytes += 8.0 * rows * (L + q["T"] + 1)
        else:
            population += 8.0 * rows * L
            nbytes += 8.0 * each * (2 * L + 3 * c["N"] + q["P"])
    nbytes += population * (c["N"] if population > (256 << 20) else 1)
    return {"bytes": nbytes, "flops": flops}


# ------------------------------------------------------ results in 64 bits


def _kernel(c, tau, w):
    """The kernel rows over the concatenated genome (positive, then negative frequencies), trapezoid weights."""
    df = np.empty_like(w)
    df[1:-1] = 0.5 * (w[2:] - w[:-2])
    df[0], df[-1] = 0.5 * (w[1] - w[0]), 0.5 * (w[-1] - w[-2])
    sign = -1.0 if c["spectra"] in ("spfsf", "ffull") else 1.0
    kp = df * np.exp(-np.outer(tau, w))
    if c["zero_temperature"]:
        return kp, df
    return np.concatenate([kp, sign * df * np.exp(np.outer(tau - BETA, w))], axis=1), np.concatenate([df, df])


class _Stream:
    """xoshiro256+ in whole numbers, seeded as the reference seeds it."""

    M = (1 << 64) - 1

    def __init__(self, seed):
        sm = 1407513600 + seed
        words = []
        for _ in range(2):
            sm = (sm + 0x9E3779B97F4A7C15) & self.M
            z = sm
            z = ((z ^ (z >> 30)) * 0xBF58476D1CE4E5B9) & self.M
            z = ((z ^ (z >> 27)) * 0x94D049BB133111EB) & self.M
            z ^= z >> 31
            words += [z & 0xFFFFFFFF, z >> 32]
        self.s = words

    def next(self):
        a, b, c, d = self.s
        out = (a + d) & self.M
        t = (b << 17) & self.M
        c ^= a
        d ^= b
        self.s = [a ^ d, b ^ c, c ^ t, ((d << 45) | (d >> 19)) & self.M]
        return out

    def unit(self):
        return (self.next() >> 11) * 2.0 ** -53


def _exact_run(c, seed):
    """One whole run in plain 64-bit numpy; only the standard kernel without moment terms."""
    rng = np.random.default_rng([c["T"], c["G"], c["P"], seed])
    tau, f, err, _ = _data(c, rng)
    stream = _Stream(int(rng.integers(1, 1 << 30)))
    G, P, N = c["G"], c["P"], c["N"]
    w = np.arange(G) * (c["omega_max"] / (G - 1))
    K, df = _kernel(c, tau, w)
    L = K.shape[1]
    signs = L // G
    pop = np.empty((P, L))
    for i in range(P):
        u = np.array([stream.unit() for _ in range(L)])
        for s in range(signs):
            pop[i, s * G:(s + 1) * G] = u[s::signs]
        if signs == 2:
            pop[i, G] = pop[i, 0]
        pop[i] *= f[0] / np.dot(pop[i], df)

    wide = K.T.astype(np.longdouble)

    def fitness_of(x):
        # every product and sum in the order of the genome, rounded once: a trial that changes nothing that counts
        # must tie with its parent, as it does in the reference
        e = np.zeros((P, c["T"]))
        for k in range(L):
            e = (wide[k] * x[:, k:k + 1] + e).astype(np.float64)
        d = (f - e) / err
        chi = np.zeros(P)
        for t in range(c["T"]):
            chi = chi + d[:, t] * d[:, t]
        return chi / c["T"]

    fit = fitness_of(pop)
    cr, fw = np.full((P, signs), 0.9), np.full((P, signs), 0.9)
    stats = np.zeros((3, N))
    for g in range(N - 1):
        stats[:, g] = np.mean(fit), np.min(fit), np.mean(fit ** 2)
        ncr, nfw = cr.copy(), fw.copy()
        for i in range(P):
            for s in range(signs):
                if stream.unit() < 0.1:
                    ncr[i, s] = stream.unit()
                if stream.unit() < 0.1:
                    nfw[i, s] = 2.0 * stream.unit()
        trials = pop.copy()
        for i in range(P):
            donors = [i]
            while len(donors) < 4:
                d = stream.next() % P
                if d not in donors:
                    donors.append(d)
            x1, x2, x3 = (pop[d] for d in donors[1:])
            u = np.array([stream.unit() for _ in range(L)])
            scale, cross = np.repeat(nfw[i], G), np.repeat(ncr[i], G)
            mutant = np.abs((scale * (x2 - x3).astype(np.longdouble) + x1).astype(np.float64))
            trials[i] = np.where(u < cross, mutant, pop[i])
            if signs == 2:
                trials[i, G] = trials[i, 0]
        new = fitness_of(trials)
        for i in range(P):
            if new[i] <= fit[i]:
                fit[i], pop[i], cr[i], fw[i] = new[i], trials[i], ncr[i], nfw[i]
    stats[:, N - 1] = np.mean(fit), np.min(fit), np.mean(fit ** 2)
    best = int(np.argmin(fit))
    x = pop[best]
    if signs == 1:
        dsf, freq = x.copy(), w
    else:
        sp, sn = x[:G].copy(), x[G:].copy()
        if c["spectra"] == "spfsf":
            sp *= -2.0 * np.pi * (1.0 + np.exp(-BETA * w))
            sn *= -2.0 * np.pi * (1.0 + np.exp(BETA * w))
        dsf, freq = np.empty(2 * G - 1), np.empty(2 * G - 1)
        dsf[G - 1:], freq[G - 1:] = sp, w
        dsf[:G], freq[:G] = sn[::-1], -w[::-1]
    return {"dsf": dsf, "frequency": freq, "mean": stats[0], "minimum": stats[1], "squared_mean": stats[2],
            "fitness": fit, "minimum_fitness": float(fit[best]), "best_index": best, "generation": N - 1,
            "rng": np.array(stream.s, dtype=np.uint64).view(np.int64)}


def exact(case, seed):
    """The same results without this repository's code, where plain numpy is quick enough: the stack's evaluation,
    and runs of up to three million draws.  A longer run is a chain of accept-or-reject decisions in one sequential
    random stream."""
    c = dict(case)
    if c["kind"] == "isf":
        rng = np.random.default_rng([c["T"], c["G"], c["P"], seed])
        tau, f, err, _ = _data(c, rng)
        K, _ = _kernel(c, tau, np.arange(c["G"]) * (c["omega_max"] / (c["G"] - 1)))
        e = _genomes(c, rng) @ K.T
        return {"model_isf": e, "chi2": np.sum(((f - e) / err) ** 2, axis=1) / c["T"]}
    plain = (c["kind"] == "engine" and c["model"] == "standard" and c["spectra"] in ("bfull", "spfsf")
             and not c["renormalize"] and not c["first_moment"] and not c["third_moment"] and c["precision"] == "fp64")
    if plain and 2 * c["G"] * c["P"] * c["N"] <= 3_000_000:
        return _exact_run(c, seed)
    return None
