"""What the performance of this package is measured on.

A case is one call, or one short run of calls, that a user's program makes on
a problem it holds: a plain search (``Problem.run_hcs``, a ``Session``, one
``Problem.local_mc``), a guided search, a batch of uneven problems, the
differentiable relaxation forward and backward, or the fitness of a
population.  The listed sizes are this repository's own workloads
(``pyhea_amd.problem``) and the small cells of its tests; ``draw`` spreads
lattice type, cell edge, species, shells, population, proposals per round and
depth over the ranges those stand for.

Targets, populations, logits and stream keys come from the seed alone.
"""
from __future__ import annotations

import functools
import math

import numpy as np
import torch

from pyhea_amd.hcs import Batch, Problem
from pyhea_amd.lattice import neighbor_table
from pyhea_amd.problem import ProblemSpec, largest_remainder, random_target
from pyhea_amd.relax import RelaxObjective

_BASIS = {"FCC": 4, "BCC": 2}
_WEIGHT = (4.0, 1.0, 0.5)  # the shell weights of every workload


def _search(name, how, latt, edge, species, solutions, task, iters=1, depth=10, shells="true",
            weights=3, **more):
    return dict(name=name, kind="search", how=how, latt=latt, edge=edge, shells=shells,
                weights=weights, species=species, solutions=solutions, task=task, depth=depth,
                iters=iters, cand=more.get("cand", 0), accepts=more.get("accepts", 0))


def _relax(name, latt, edge, species, double):
    return dict(name=name, kind="relax", latt=latt, edge=edge, shells="true", weights=3,
                species=species, double=double)


def listed():
    eq4 = "1 1 1 1"
    bcc5 = "30 25 20 15 10"
    eq5 = "1 1 1 1 1"
    fcc6 = "25 20 20 15 10 10"
    return [
        # the shortest search: a cell of the tests, a handful of solutions, as a
        # script calls it while a configuration is tried out
        _search("tiny local search", "local", "FCC", 3, "40 35 25", 8, 64, depth=3),
        # the example configuration (4000 sites) through the drop-in call, host
        # arrays out, the reference's own third shell
        _search("drop-in fcc10", "run", "FCC", 10, eq4, 128, 256, iters=2, shells="pyhea"),
        # the plain search's own workload: two lattices a CU
        _search("plain session bcc16", "session", "BCC", 16, bcc5, 512, 256, iters=2),
        # 108000 sites, plain: one lattice a CU, neighbour table beyond an L2
        _search("plain session fcc30", "session", "FCC", 30, eq5, 256, 512),
        # a population beyond LDS, plain: the species stay in HBM (256000 sites, of
        # which a search of an unlucky target takes about a second)
        _search("plain local search fcc40", "local", "FCC", 40, fcc6, 64, 256, depth=10),
        # the time-to-fitness workload: guided and batched, one problem
        _search("guided batch fcc30", "batch", "FCC", 30, eq5, 256, 512, cand=12, accepts=8),
        # guided at the example's size, where the rounds are short
        _search("guided session fcc10", "session", "FCC", 10, eq4, 128, 256, iters=2, cand=12,
                accepts=8),
        # uneven problems in one persistent launch (odd edges, K 3-6, both types)
        dict(name="mixed batch", kind="mixed", problems=12, low=6, high=20, solutions=128,
             task=256, depth=10, iters=1),
        # gradient steps on site logits: small in float64, the two large sizes
        # in float32
        _relax("relaxation fcc10 float64", "FCC", 10, eq4, True),
        _relax("relaxation fcc30 float32", "FCC", 30, eq5, False),
        _relax("relaxation fcc50 float32", "FCC", 50, fcc6, False),
        # recount fitness of a whole population held by the host
        dict(name="fitness bcc16", kind="fitness", latt="BCC", edge=16, shells="true", weights=3,
             species=bcc5, solutions=512),
    ]


def draw(rng):
    """One more case: most are searches, as in use."""
    def logint(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    what = rng.choices(["plain", "guided", "mixed", "relax", "fitness"], [9, 4, 1, 4, 2])[0]
    if what == "mixed":
        low = rng.randint(4, 10)
        return dict(kind="mixed", problems=rng.randint(2, 12), low=low,
                    high=rng.randint(low + 2, 18), solutions=logint(8, 128),
                    task=rng.randint(64, 300), depth=rng.randint(4, 10), iters=1)
    latt = rng.choice(["FCC", "BCC"])
    edge = logint(4, 32 if latt == "FCC" else 40) if rng.random() < 0.9 else \
        (rng.randint(33, 40) if latt == "FCC" else rng.randint(41, 50))
    n = _BASIS[latt] * edge ** 3
    k = rng.randint(2, 5 if what == "guided" else 8) if rng.random() < 0.3 else rng.randint(3, 5)
    species = " ".join(str(rng.randint(1, 6) * 5) for _ in range(k))
    shells = rng.choice(["true", "true", "pyhea"])
    weights = 3 if rng.random() < 0.8 else rng.randint(1, 2)
    if what == "relax":
        return dict(kind="relax", latt=latt, edge=edge, shells=shells, weights=weights,
                    species=species, double=rng.random() < 0.3)
    cap = 60_000_000 // n if n < 120_000 else 12_000_000 // n
    solutions = max(1, min(logint(4, 512), cap // (4 if what == "guided" else 3)))
    if what == "fitness":
        return dict(kind="fitness", latt=latt, edge=edge, shells=shells, weights=weights,
                    species=species, solutions=solutions)
    c = _search("", rng.choice(["run", "session", "local"]), latt, edge, species, solutions,
                logint(32, 600), depth=rng.randint(3, 12), shells=shells, weights=weights)
    if what == "guided":
        c["how"] = rng.choice(["session", "batch"])
        c["cand"], c["accepts"] = rng.randint(4, 16), rng.randint(1, 8)
    del c["name"]
    return c


# ------------------------------------------------------------------ inputs --

@functools.lru_cache(maxsize=32)
def _table(latt, edge, shells):
    return neighbor_table(edge, latt, shells)


def _spec(latt, edge, shells, weights, fractions, seed):
    nbr, sizes = _table(latt, edge, shells)
    used = int(sum(sizes[:weights]))
    counts = largest_remainder(fractions, nbr.shape[0])
    return ProblemSpec(latt, edge, counts, list(_WEIGHT[:weights]),
                       random_target(counts, weights, seed), shells,
                       np.ascontiguousarray(nbr[:, :used]), list(sizes[:weights]))


def _case_spec(case, seed):
    return _spec(case["latt"], case["edge"], case["shells"], case["weights"],
                 [float(x) for x in case["species"].split()], seed)


def _mixed_shapes(case):
    """The problems of a mixed batch: the sizes belong to the case, so every
    seed does the same amount of work on its own targets and streams."""
    rng = np.random.default_rng([case["problems"], case["low"], case["high"]])
    shapes = []
    for i in range(case["problems"]):
        k = int(rng.integers(3, 7))
        shapes.append(("FCC" if i % 2 == 0 else "BCC",
                       int(rng.integers(case["low"], case["high"] + 1)), rng.dirichlet([2.0] * k)))
    return shapes


def _logits(spec, double, seed):
    g = torch.Generator().manual_seed(seed)
    th = torch.randn(spec.n_sites, spec.K, generator=g, dtype=torch.float64)
    return th if double else th.float()


def _population(spec, solutions, seed):
    rng = np.random.default_rng(seed)
    base = np.repeat(np.arange(spec.K, dtype=np.uint8), spec.counts)
    return rng.permuted(np.broadcast_to(base, (solutions, spec.n_sites)), axis=1)


def prepare(case, seed):
    if case["kind"] == "mixed":
        probs = [Problem.from_spec(_spec(t, e, "true", 3, f, seed + i))
                 for i, (t, e, f) in enumerate(_mixed_shapes(case))]
        return dict(case=case, batch=Batch(probs, case["solutions"], case["task"], case["depth"],
                                           seed=seed), n=len(probs))
    spec = _case_spec(case, seed)
    prob = Problem.from_spec(spec)
    state = dict(case=case, problem=prob, seed=seed)
    if case["kind"] == "relax":
        state["objective"] = RelaxObjective(prob)
        state["logits"] = _logits(spec, case["double"], seed).cuda().requires_grad_()
    elif case["kind"] == "fitness":
        state["lattices"] = _population(spec, case["solutions"], seed)
    elif case["how"] == "session":
        state["session"] = prob.session(case["solutions"], case["task"], case["depth"], seed=seed)
        if case["cand"]:
            state["session"].guide(case["cand"], 0.1, case["accepts"])
    elif case["how"] == "batch":
        state["batch"] = Batch([prob], case["solutions"], case["task"], case["depth"], seed=seed)
        state["batch"].guide(case["cand"], 0.1, case["accepts"])
        state["n"] = 1
    elif case["how"] == "local":
        state["population"] = prob.generate(case["solutions"], seed)
    return state


# --------------------------------------------------------------------- run --

def _answer(lat, fit, st):
    return dict(lattices=lat, fitness=fit,
                counters=np.array([st["evals"], st["rounds"], st["accepts"], st["draws"]]))


def run(state):
    case = state["case"]
    if case["kind"] == "relax":
        th = state["logits"]
        th.grad = None
        f2 = state["objective"](th)
        f2.backward()
        return dict(f2=f2.detach(), grad=th.grad)
    if case["kind"] == "fitness":
        return state["problem"].fitness(state["lattices"])
    if "batch" in state:
        b = state["batch"]
        b.init()
        b.step(case["iters"])
        return [_answer(*b.read(p)) for p in range(state["n"])]
    if "session" in state:
        s = state["session"]
        s.init()
        s.step(case["iters"])
        return _answer(*s.read())
    if case["how"] == "local":
        lat, fit = state["population"]
        return _answer(*state["problem"].local_mc(lat, fit, case["task"], case["depth"],
                                                  seed=state["seed"]))
    return _answer(*state["problem"].run_hcs(case["solutions"], case["iters"], case["task"],
                                             case["depth"], seed=state["seed"]))


# -------------------------------------------------------------------- work --

_Z = {("FCC", "true"): (12, 6, 24), ("FCC", "pyhea"): (12, 6, 12), ("BCC", "true"): (8, 6, 12),
      ("BCC", "pyhea"): (8, 6, 12)}


def _shape(case):
    n = _BASIS[case["latt"]] * case["edge"] ** 3
    return n, sum(_Z[case["latt"], case["shells"]][:case["weights"]]), len(case["species"].split())


def _search_work(n, sum_z, k, shells, case):
    """One swap evaluation reads both sites' neighbour indices and species and
    computes the changed entries of every shell.  A local search makes about
    N / 10 rounds plus the rejected ones that end it (guided: several accepts
    a round, about N / 80 rounds, each scoring its candidates' records)."""
    searches = case["solutions"] * (1 if case.get("how") == "local" else 2 * case["iters"])
    cand = case.get("cand", 0)
    rounds = n / (80 if cand else 10) + case["depth"]
    evals = searches * rounds * case["task"]
    return (evals * (2 * sum_z * 5 + 2 + 18 * cand) + 2 * searches * n,
            evals * (2 * sum_z + shells * 2 * k * 7 + cand * 2 * shells * k * 3))


def work(case):
    if case["kind"] == "mixed":
        by = fl = 0.0
        for t, e, f in _mixed_shapes(case):
            b, x = _search_work(_BASIS[t] * e ** 3, sum(_Z[t, "true"]), len(f), 3, case)
            by, fl = by + b, fl + x
        return dict(bytes=by, flops=fl)
    n, sum_z, k = _shape(case)
    if case["kind"] == "relax":  # the table and the logits each way, and the gradient
        el = 8 if case["double"] else 4
        return dict(bytes=2 * n * (4 * sum_z + el * k) + n * el * k,
                    flops=n * (2 * k * sum_z + 4 * case["weights"] * k * k + 40 * k))
    if case["kind"] == "fitness":
        visits = case["solutions"] * n * sum_z
        return dict(bytes=case["solutions"] * (n + 8) + 4 * n * sum_z, flops=visits)
    b, x = _search_work(n, sum_z, k, case["weights"], case)
    return dict(bytes=b, flops=x)


# ------------------------------------------------------------------- exact --

def _exact_relax(case, seed):
    spec = _case_spec(case, seed)
    n, k = spec.n_sites, spec.K
    th = _logits(spec, case["double"], seed).cuda().double()
    p = torch.softmax(th, 1)
    nbr = torch.from_numpy(spec.nbr).cuda().long()
    conc = torch.tensor(np.asarray(spec.counts, np.float64) / n).cuda()
    cc = conc[:, None] * conc[None, :]
    f2 = torch.zeros((), dtype=torch.float64, device="cuda")
    g = torch.zeros(n, k, dtype=torch.float64, device="cuda")
    off = 0
    for s, z in enumerate(spec.shell_sizes):
        q = torch.zeros_like(p)
        for c in range(off, off + z):
            q += p[nbr[:, c]]
        off += z
        t = torch.tensor(np.asarray(spec.target[s], np.float64).reshape(k, k)).cuda()
        diff = 1.0 - (p.t() @ q) / (z * n) / cc - t
        f2 += spec.weight[s] * (diff * diff).sum()
        dn = -2.0 * spec.weight[s] * diff / (z * n * cc)
        g += q @ (dn + dn.t()).t()
    grad = p * (g - (p * g).sum(1, keepdim=True))
    return dict(f2=f2, grad=grad)


def _exact_fitness(case, seed):
    spec = _case_spec(case, seed)
    n, k = spec.n_sites, spec.K
    lat = torch.from_numpy(_population(spec, case["solutions"], seed)).cuda().long()
    conc = np.asarray(spec.counts, np.float64) / n
    cc = np.outer(conc, conc)
    err = np.zeros(lat.shape[0])
    off = 0
    for s, z in enumerate(spec.shell_sizes):
        cols = torch.from_numpy(np.ascontiguousarray(spec.nbr[:, off:off + z])).cuda().long()
        off += z
        cnt = torch.stack([torch.bincount((row[:, None] * k + row[cols]).reshape(-1),
                                          minlength=k * k) for row in lat])
        gamma = cnt.cpu().numpy().astype(np.float64).reshape(-1, k, k) / (z * n)
        diff = 1.0 - gamma / cc - np.asarray(spec.target[s]).reshape(k, k)
        err += spec.weight[s] * (diff * diff).sum((1, 2))
    return np.sqrt(err)


def exact(case, seed):
    """Relaxation and fitness from their definitions in 64 bits; a search has
    no value but its own (its lattices and counters are whole numbers)."""
    if case["kind"] == "relax":
        return _exact_relax(case, seed)
    if case["kind"] == "fitness":
        return _exact_fitness(case, seed)
    return None
