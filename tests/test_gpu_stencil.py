"""The stencil-lattice search against the oracle, bit for bit, where its
layout can go wrong: rounds of one proposal, of one wave and one more, the
largest it takes and the first it does not; every species count; one to
three shells; the smallest edge; odd site counts; a composition so skewed
that a round needs several draw passes; rows in an order of their own (the
replays follow the rows); equimolar species, whose entries sit at binade
edges and are replayed."""
import numpy as np
import pytest

from oracle import Oracle
from pyhea_amd.hcs import Batch, Problem
from pyhea_amd.problem import ProblemSpec, make_problem

pytestmark = pytest.mark.gpu


def _bits(a):
    return np.asarray(a, np.float64).view(np.uint64)


def _check(spec, task, depth, lattices=3, seed=31):
    o, p = Oracle.from_spec(spec), Problem.from_spec(spec)
    lat0 = np.stack([o.permute(9, 0, 0, l) for l in range(lattices)])
    fit0 = o.fitness(lat0)
    lo, fo, so = o.local_mc(lat0, fit0, task, depth, seed=seed, iter=1, phase=2)
    lg, fg, sg = p.local_mc(lat0, fit0, task, depth, seed=seed, iter=1, phase=2)
    assert np.array_equal(lg, lo)
    assert np.array_equal(_bits(fg), _bits(fo))
    for k in ("evals", "rounds", "accepts", "draws"):
        assert sg[k] == so[k], k
    return so


@pytest.mark.parametrize("task", [1, 63, 64, 65, 129, 704, 705])
def test_round_sizes(gpu, task):
    _check(make_problem("FCC", 4, [0.3, 0.25, 0.2, 0.15, 0.1], target_seed=5), task, 2)


@pytest.mark.parametrize("latt,edge,shells,weights,k", [
    ("FCC", 3, "true", 3, 2), ("FCC", 5, "pyhea", 3, 3), ("BCC", 3, "true", 3, 4),
    ("BCC", 5, "true", 2, 5), ("FCC", 3, "true", 1, 6), ("BCC", 7, "pyhea", 3, 7),
    ("FCC", 5, "true", 3, 8), ("BCC", 9, "true", 1, 8),
])
def test_species_shells_and_edges(gpu, latt, edge, shells, weights, k):
    spec = make_problem(latt, edge, np.arange(2, k + 2), weight=[4.0, 1.0, 0.5][:weights],
                        shells=shells, target_seed=k)
    _check(spec, 96, 3)


def test_skewed_composition_takes_several_draw_passes(gpu):
    spec = make_problem("BCC", 6, None, counts=[429, 3], target_seed=4)
    st = _check(spec, 200, 3)
    assert st["draws"] > 20 * 200


def test_rows_in_any_order(gpu):
    spec = make_problem("FCC", 4, None, counts=[64] * 4, target_seed=8)
    rng = np.random.default_rng(1)
    z = np.cumsum([0] + list(spec.shell_sizes))
    nbr = np.concatenate([rng.permuted(spec.nbr[:, z[s]:z[s + 1]], axis=1) for s in range(3)],
                         axis=1)
    _check(ProblemSpec("FCC", 4, spec.counts, spec.weight, spec.target, "true", nbr,
                       spec.shell_sizes), 128, 6)


@pytest.mark.parametrize("counts", [[128] * 2, [64] * 4, [32] * 8])
def test_equimolar_replays(gpu, counts):
    spec = make_problem("FCC", 4, None, counts=counts, target_seed=2)
    spec.target[:] = 0.0
    _check(spec, 256, 8)


@pytest.mark.parametrize("latt,edge,shells,k,task", [
    ("FCC", 35, "true", 5, 64), ("FCC", 36, "pyhea", 3, 33), ("BCC", 44, "true", 8, 64),
    ("BCC", 50, "true", 2, 256),
])
def test_two_species_a_byte_equals_the_hbm_walk(gpu, monkeypatch, latt, edge, shells, k, task):
    spec = make_problem(latt, edge, np.arange(3, k + 3), shells=shells, target_seed=k)
    p = Problem.from_spec(spec)
    monkeypatch.setenv("PYHEA_AMD_SPECIES_IN_HBM", "1")  # read when a problem is created
    q = Problem.from_spec(spec)
    lat, fit = p.generate(3, seed=5)
    a = p.local_mc(lat, fit, task, 3, seed=6)
    b = q.local_mc(lat, fit, task, 3, seed=6)
    assert np.array_equal(a[0], b[0]) and np.array_equal(_bits(a[1]), _bits(b[1]))
    assert all(a[2][c] == b[2][c] for c in ("evals", "rounds", "accepts", "draws"))


@pytest.mark.parametrize("edge,shells,k", [(3, "pyhea", 4), (4, "true", 6), (4, "true", 7),
                                           (5, "pyhea", 6), (6, "true", 4), (7, "pyhea", 8)])
def test_walks_by_cell(gpu, edge, shells, k):
    """Each parity of the edge and each width of the histograms."""
    _check(make_problem("FCC", edge, np.arange(2, k + 2), shells=shells, target_seed=k), 100, 3)


def test_batch_of_every_species_count(gpu):
    """One problem per table width in one launch, against its own search."""
    specs = [make_problem("FCC" if k % 2 else "BCC", 4, np.arange(2, k + 2), target_seed=k)
             for k in range(2, 9)]
    probs = [Problem.from_spec(s) for s in specs]
    b = Batch(probs, 5, 96, 3, seed=40)
    b.init()
    b.step(2)
    for q, p in enumerate(probs):
        lat, fit, st = b.read(q)
        lo, fo, so = p.run_hcs(5, 2, 96, 3, seed=40 + q)
        assert np.array_equal(lat, lo) and np.array_equal(_bits(fit), _bits(fo))
        assert st["accepts"] == so["accepts"]
