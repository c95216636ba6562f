"""The relaxed objective in one call and the gather over a stencil lattice,
where they can go wrong: each shell set and species count, site counts around
a workgroup's, lattices whose ids are not the stencil's, scaled and shared
losses, constants of the caller's own, and replays of a captured step."""
import numpy as np
import pytest
import torch

from pyhea_amd.hcs import Problem
from pyhea_amd.problem import ProblemSpec, make_problem
from pyhea_amd.relax import RelaxObjective, SoftPairCounts

pytestmark = pytest.mark.gpu


def _spec(latt, edge, shells, K, S=3, relabel=False):
    spec = make_problem(latt, edge, np.arange(2, K + 2), weight=[4.0, 1.0, 0.5][:S], shells=shells,
                        target_seed=K)
    if not relabel:
        return spec
    to = np.random.default_rng(5).permutation(spec.n_sites).astype(np.int32)
    nbr = np.empty_like(spec.nbr)
    nbr[to] = to[spec.nbr]
    return ProblemSpec(latt, edge, spec.counts, spec.weight, spec.target, shells, nbr,
                       spec.shell_sizes)


def _logits(spec, K, dtype=torch.float64, seed=3):
    g = torch.Generator().manual_seed(seed)
    return torch.randn(spec.n_sites, K, dtype=torch.float64, generator=g).to("cuda", dtype)


def _reference(th, spec):
    """Counts in FP64 torch, on the device, of the same occupancies."""
    p, out, off = torch.softmax(th.double(), 1), [], 0
    for z in spec.shell_sizes:
        idx = torch.as_tensor(np.asarray(spec.nbr[:, off:off + z]), dtype=torch.long,
                              device=th.device)
        out.append(p.T @ p[idx].sum(1))
        off += z
    return torch.stack(out)


@pytest.mark.parametrize("relabel", [False, True])
@pytest.mark.parametrize("latt,edge,shells,K,S", [
    ("FCC", 3, "true", 2, 3), ("FCC", 4, "pyhea", 4, 3), ("BCC", 3, "true", 5, 3),
    ("BCC", 8, "true", 6, 2), ("FCC", 5, "true", 7, 3), ("BCC", 5, "true", 8, 1),
    ("FCC", 7, "pyhea", 5, 2),
])
@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
def test_counts_value_and_gradient(gpu, latt, edge, shells, K, S, relabel, dtype):
    spec = _spec(latt, edge, shells, K, S, relabel)
    prob = Problem.from_spec(spec)
    obj = RelaxObjective(prob)
    th = _logits(spec, K, dtype).requires_grad_(True)
    ref_th = th.detach().double().requires_grad_(True)
    ref = _reference(ref_th, spec)
    n = SoftPairCounts.apply(th.detach(), prob)
    # float32: rows of p and q rounded to 2^-24 of themselves; the softmax's own
    # exp and division are a few of those
    tol = 1e-12 if dtype is torch.float64 else 2e-6
    assert torch.allclose(n, ref, rtol=tol, atol=0)
    f2, want = obj(th), obj.from_counts(n)
    assert f2.shape == want.shape and f2.dtype == want.dtype and f2.requires_grad
    alpha = 1.0 - (n / obj.zn[:, None, None]) / obj.cc
    room = ((alpha.abs() + obj.target.abs() + 1.0) ** 2).sum((-1, -2)).mul(obj.weight).sum()
    assert abs(f2.item() - want.item()) <= 64 * 2.0 ** -53 * room.item()
    (2.5 * f2).backward()
    (2.5 * obj.from_counts(ref)).backward()
    gmax = ref_th.grad.abs().max().item()
    assert (th.grad.double() - ref_th.grad).abs().max().item() <= (
        1e-11 if dtype is torch.float64 else 2e-5) * gmax


def test_two_terms_of_one_loss_and_no_grad(gpu):
    spec = _spec("BCC", 4, "true", 3)
    prob = Problem.from_spec(spec)
    obj = RelaxObjective(prob)
    a, b = _logits(spec, 3).requires_grad_(True), _logits(spec, 3, seed=4).requires_grad_(True)
    fa, fb = obj(a), obj(b)  # both forwards before either backward
    (fa * fb).backward()
    c, d = a.detach().clone().requires_grad_(True), b.detach().clone().requires_grad_(True)
    ga, gb = torch.autograd.grad(obj(c), c)[0], torch.autograd.grad(obj(d), d)[0]
    assert torch.allclose(a.grad, ga * fb.detach(), rtol=1e-12, atol=1e-18)
    assert torch.allclose(b.grad, gb * fa.detach(), rtol=1e-12, atol=1e-18)
    with torch.no_grad():
        assert obj(a).item() == fa.item() and not obj(a).requires_grad


def test_constants_of_the_callers_own(gpu):
    spec = _spec("BCC", 4, "true", 3)
    prob = Problem.from_spec(spec)
    th = _logits(spec, 3)
    base = RelaxObjective(prob)
    n = SoftPairCounts.apply(th, prob)
    for name, value in (("weight", base.weight.clone().requires_grad_(True)),
                        ("target", base.target.float()), ("cc", base.cc.clone().T),
                        ("weight", base.weight[:1]), ("target", base.target * 0.5)):
        obj = RelaxObjective(prob)
        setattr(obj, name, value)
        got, want = obj(th), obj.from_counts(n)
        assert torch.allclose(got, want, rtol=1e-13)
        assert got.requires_grad == want.requires_grad

    class Halved(RelaxObjective):
        def from_counts(self, n):
            return 0.5 * super().from_counts(n)

    assert torch.allclose(Halved(prob)(th), 0.5 * base(th), rtol=1e-13)
    with pytest.raises(ValueError):
        base(th.cpu())
    with pytest.raises(TypeError):
        base(th.half())


def test_replays_of_a_captured_step(gpu):
    spec = _spec("FCC", 5, "true", 4)
    prob = Problem.from_spec(spec)
    obj = RelaxObjective(prob)
    th = _logits(spec, 4).requires_grad_(True)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        for _ in range(2):
            th.grad = None
            obj(th).backward()
    torch.cuda.current_stream().wait_stream(side)
    th.grad = None
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        f2 = obj(th)
        f2.backward()
    for seed in (11, 12, 13):
        with torch.no_grad():
            th.copy_(_logits(spec, 4, seed=seed))
        graph.replay()
        torch.cuda.synchronize()
        eager = th.detach().clone().requires_grad_(True)
        want = obj(eager)
        want.backward()
        assert f2.item() == want.item() and torch.equal(th.grad, eager.grad)
