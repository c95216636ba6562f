"""The guided search on stencil lattices against the general guided kernel,
bit for bit.  The general kernel runs when the species are kept in HBM
(PYHEA_AMD_SPECIES_IN_HBM=1).  Sizes where the layout can go wrong: rounds of
one proposal, of one wave and one more, the largest of the new kernel and the
first beyond it; 1, 11, 12, 13 and 30 candidates (12 are drawn ahead); one to
many accepts; every species count; blocks of 2 to 64 sites; records in LDS and
in HBM; the smallest edge; equimolar species, whose entries are replayed."""
import numpy as np
import pytest

from pyhea_amd.hcs import Problem
from pyhea_amd.problem import make_problem

pytestmark = pytest.mark.gpu


def _search(prob, L, task, depth, cand, accepts, iters=1, tau=0.1):
    s = prob.session(L, task, depth, seed=77)
    s.guide(cand, tau, accepts)
    s.init()
    s.step(iters)
    out = s.read()
    s.close()
    return out


def _same(monkeypatch, spec, L, task, depth, cand, accepts, blk=4, **kw):
    monkeypatch.setenv("PYHEA_AMD_GUIDE_BLOCK", str(blk))
    p = Problem.from_spec(spec)
    monkeypatch.setenv("PYHEA_AMD_SPECIES_IN_HBM", "1")
    q = Problem.from_spec(spec)
    a, b = (_search(x, L, task, depth, cand, accepts, **kw) for x in (p, q))
    assert np.array_equal(a[0], b[0])
    assert np.array_equal(a[1].view(np.uint64), b[1].view(np.uint64))
    assert all(a[2][c] == b[2][c] for c in ("evals", "rounds", "accepts", "draws"))


@pytest.mark.parametrize("task", [1, 64, 65, 200, 704, 705])
def test_round_sizes(gpu, monkeypatch, task):
    _same(monkeypatch, make_problem("FCC", 6, [3, 2, 2, 1, 1], target_seed=3), 4, task, 3, 12, 8)


@pytest.mark.parametrize("cand,accepts", [(1, 1), (4, 2), (11, 8), (13, 8), (30, 40)])
def test_candidates_and_accepts(gpu, monkeypatch, cand, accepts):
    _same(monkeypatch, make_problem("BCC", 9, [4, 3, 2, 1], target_seed=4), 4, 130, 3, cand, accepts)


@pytest.mark.parametrize("latt,edge,shells,k,blk", [
    ("FCC", 3, "true", 2, 1), ("FCC", 5, "pyhea", 3, 4), ("BCC", 3, "true", 4, 6),
    ("BCC", 30, "true", 5, 4), ("FCC", 20, "true", 6, 2), ("FCC", 25, "pyhea", 2, 6),
])
def test_species_shells_blocks_and_record_placement(gpu, monkeypatch, latt, edge, shells, k, blk):
    spec = make_problem(latt, edge, np.arange(2, k + 2), shells=shells, target_seed=k)
    _same(monkeypatch, spec, 3, 96, 3, 12, 8, blk=blk)


@pytest.mark.parametrize("counts", [[128] * 2, [64] * 4])
def test_equimolar_replays(gpu, monkeypatch, counts):
    spec = make_problem("FCC", 4, None, counts=counts, target_seed=2)
    spec.target[:] = 0.0
    _same(monkeypatch, spec, 4, 256, 6, 12, 8, iters=2)


@pytest.mark.parametrize("task", [192, 256, 449, 640, 641])
@pytest.mark.parametrize("accepts", [1, 2, 8])
def test_with_and_without_the_helper_wave(gpu, monkeypatch, task, accepts):
    """Workgroups of 4 to 12 waves, of which those that lose no residency have
    the wave that updates the records."""
    spec = make_problem("BCC", 12, [4, 3, 2, 1], target_seed=6)
    _same(monkeypatch, spec, 3, task, 3, 6, accepts)
