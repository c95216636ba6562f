"""Counts, fitness and order of populations where their kernels can go wrong:
every species count and shell set, lattices that take several flushes of the
packed counters, compositions other than the problem's, populations that do
not fill a workgroup, and merges around a wave's 64 keys."""
import numpy as np
import pytest

from oracle import Oracle
from pyhea_amd.hcs import Problem
from pyhea_amd.problem import make_problem

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("latt,edge,shells,k,weights", [
    ("FCC", 3, "true", 2, 3), ("BCC", 3, "true", 3, 1), ("FCC", 5, "pyhea", 4, 2),
    ("BCC", 13, "true", 6, 3), ("FCC", 11, "true", 5, 3), ("FCC", 23, "pyhea", 5, 3),
    ("FCC", 17, "true", 6, 3), ("BCC", 6, "true", 7, 3), ("FCC", 4, "true", 8, 2),
])
@pytest.mark.parametrize("solutions", [1, 5])
def test_counts_and_fitness(gpu, latt, edge, shells, k, weights, solutions):
    spec = make_problem(latt, edge, np.arange(2, k + 2), weight=[4.0, 1.0, 0.5][:weights],
                        shells=shells, target_seed=k)
    o, p = Oracle.from_spec(spec), Problem.from_spec(spec)
    rng = np.random.default_rng(edge * k)
    lat = rng.integers(0, k, (solutions, p.n_sites)).astype(np.uint8)
    lat[0] = k - 1  # the largest counts of one entry
    want = np.stack([o.pair_counts(row) for row in lat])
    assert np.array_equal(p.pair_counts(lat), want.reshape(solutions, p.S, k, k))
    assert np.array_equal(p.fitness(lat).view(np.uint64), o.fitness(lat).view(np.uint64))


@pytest.mark.parametrize("solutions", [1, 31, 33, 64, 65])
def test_merges_around_a_wave(gpu, solutions):
    spec = make_problem("BCC", 4, [0.3, 0.3, 0.4], target_seed=3)
    o, p = Oracle.from_spec(spec), Problem.from_spec(spec)
    lo, fo, _, _ = o.run_hcs(solutions, 2, 16, 2, seed=12)
    lg, fg, _ = p.run_hcs(solutions, 2, 16, 2, seed=12)
    assert np.array_equal(lg, lo)
    assert np.array_equal(fg.view(np.uint64), fo.view(np.uint64))


@pytest.mark.parametrize("solutions,edge", [(2, 3), (63, 4), (65, 4), (130, 5)])
def test_populations_by_column_and_view(gpu, solutions, edge):
    spec = make_problem("BCC", edge, [0.3, 0.3, 0.4], target_seed=3)
    p = Problem.from_spec(spec)
    rng = np.random.default_rng(solutions)
    wide = rng.integers(0, 3, (2 * solutions, p.n_sites)).astype(np.uint8)
    rows = np.ascontiguousarray(wide[::2])
    fit, cnt = p.fitness(rows), p.pair_counts(rows)
    for form in (np.asfortranarray(rows), wide[::2], np.asfortranarray(rows.astype(np.int64)),
                 rows.tolist(), np.asfortranarray(wide)[::2]):
        assert np.array_equal(p.fitness(form).view(np.uint64), fit.view(np.uint64))
        assert np.array_equal(p.pair_counts(form), cnt)
    with pytest.raises(ValueError):
        p.fitness(np.asfortranarray(rows).T)
