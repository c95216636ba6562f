"""Differentiable relaxation of the SRO lattice search (torch front end).

``SoftPairCounts`` maps site logits [N, K] to soft pair counts n [S, K, K]
(float64) with the HIP forward (softmax, neighbour gather, deterministic
FP64 reduction) and the hand-written HIP backward (neighbour-gather adjoint)
of ``hea_relax_forward`` / ``hea_relax_backward``; the occupancies and
neighbour sums it keeps for the backward hold ``relax_cols(K)`` elements
per site (the library's row layout; 5 for five species).  ``soft_fitness_sq`` is the relaxed
objective on top:

    gamma = n / (Z_s N),  alpha = 1 - gamma / (c_a c_b),
    F^2   = sum_s w_s sum_ab (alpha_sab - t_sab)^2

which equals the reference fitness squared (pyhea/cpp/accelerate.cpp:
165-178) when the logits are one-hot.  ``RelaxObjective`` computes it in the
same HIP call as the counts; ``from_counts`` is the same in torch ops, for
counts at hand and for constants of the caller's own.
"""
from __future__ import annotations

import ctypes as C

import numpy as np
import torch

from . import _native as Nat


def _dtype_code(t: torch.Tensor) -> int:
    if t.dtype == torch.float32:
        return 0
    if t.dtype == torch.float64:
        return 1
    raise TypeError("logits must be float32 or float64")


def relax_cols(K: int) -> int:
    """Elements per site of the occupancies p [N * KP] and neighbour sums
    q [S * N * KP] that the forward keeps for the backward, as the library
    lays them out (hea_relax_cols)."""
    kp = int(Nat.lib().hea_relax_cols(int(K)))
    if kp < 0:
        raise ValueError(f"no relaxation layout for {K} species")
    return kp


def _stream() -> C.c_void_p:
    return C.c_void_p(torch.cuda.current_stream().cuda_stream)


def _forward_args(logits: torch.Tensor, problem):
    """The checked, contiguous logits and the tensors a forward fills for the
    backward: (logits, p, q)."""
    if not logits.is_cuda:
        raise ValueError("logits must be a GPU tensor")
    lg = logits.contiguous()
    N, K, S = problem.n_sites, problem.K, problem.S
    if tuple(lg.shape) != (N, K):
        raise ValueError(f"logits must be [{N}, {K}]")
    kp = relax_cols(K)
    p = torch.empty((N, kp), dtype=lg.dtype, device=lg.device)
    q = torch.empty((S, N, kp), dtype=lg.dtype, device=lg.device)
    return lg, p, q


class SoftPairCounts(torch.autograd.Function):
    @staticmethod
    def forward(ctx, logits: torch.Tensor, problem) -> torch.Tensor:
        lg, p, q = _forward_args(logits, problem)
        n = torch.empty((problem.S, problem.K, problem.K), dtype=torch.float64, device=lg.device)
        Nat.check(Nat.lib().hea_relax_forward(problem.handle, _dtype_code(lg), lg.data_ptr(),
                                              p.data_ptr(), q.data_ptr(), n.data_ptr(),
                                              _stream()))
        ctx.save_for_backward(p, q)
        ctx.problem = problem
        return n

    @staticmethod
    def backward(ctx, dn: torch.Tensor):
        p, q = ctx.saved_tensors
        dn = dn.to(torch.float64).contiguous()
        grad = torch.empty((p.shape[0], ctx.problem.K), dtype=p.dtype, device=p.device)
        Nat.check(Nat.lib().hea_relax_backward(ctx.problem.handle, _dtype_code(p), p.data_ptr(),
                                               q.data_ptr(), dn.data_ptr(), grad.data_ptr(),
                                               _stream()))
        return grad, None


class _SoftFitnessSq(torch.autograd.Function):
    """F^2 of the logits in one call (hea_relax_objective), which also leaves
    dF^2/dn for the backward.  With the K x K algebra as tensor operations, a
    dozen launches each way, a step took 0.25 ms at any size up to 500000 sites;
    it takes 0.06 to 0.13."""

    @staticmethod
    def forward(ctx, logits: torch.Tensor, objective) -> torch.Tensor:
        problem = objective.problem
        lg, p, q = _forward_args(logits, problem)
        f2 = torch.empty((), dtype=torch.float64, device=lg.device)
        dn = torch.empty((problem.S, problem.K, problem.K), dtype=torch.float64, device=lg.device)
        Nat.check(Nat.lib().hea_relax_objective(
            problem.handle, _dtype_code(lg), lg.data_ptr(), p.data_ptr(), q.data_ptr(),
            objective.zn.data_ptr(), objective.cc.data_ptr(), objective.target.data_ptr(),
            objective.weight.data_ptr(), f2.data_ptr(), dn.data_ptr(), _stream()))
        ctx.save_for_backward(p, q, dn)
        ctx.problem = problem
        return f2

    @staticmethod
    def backward(ctx, df2: torch.Tensor):
        p, q, dn = ctx.saved_tensors
        df2 = df2.to(torch.float64).contiguous()
        grad = torch.empty((p.shape[0], ctx.problem.K), dtype=p.dtype, device=p.device)
        Nat.check(Nat.lib().hea_relax_backward_scaled(
            ctx.problem.handle, _dtype_code(p), p.data_ptr(), q.data_ptr(), dn.data_ptr(),
            df2.data_ptr(), grad.data_ptr(), _stream()))
        return grad, None


class RelaxObjective:
    """Constants of the relaxed objective for one problem (device tensors)."""

    def __init__(self, problem, device="cuda"):
        self.problem = problem
        S, K, N = problem.S, problem.K, problem.n_sites
        conc = torch.tensor(np.asarray(problem.counts, np.float64) / N, device=device)
        self.cc = conc[:, None] * conc[None, :]
        self.zn = torch.tensor([float(z) * N for z in problem.shell_sizes[:S]], device=device,
                               dtype=torch.float64)
        self.target = torch.tensor(np.asarray(problem.target, np.float64).reshape(S, K, K),
                                   device=device)
        self.weight = torch.tensor(np.asarray(problem.weight, np.float64), device=device)

    def from_counts(self, n: torch.Tensor) -> torch.Tensor:
        """F^2 from (soft or integer) pair counts n [..., S, K, K]."""
        alpha = 1.0 - (n / self.zn[:, None, None]) / self.cc
        return ((alpha - self.target) ** 2).sum((-1, -2)).mul(self.weight).sum(-1)

    def _plain(self, device) -> bool:
        """Whether from_counts is the one above on plain constants, as
        hea_relax_objective computes it; constants that were exchanged for other
        types, shapes or differentiable tensors go through from_counts."""
        if "from_counts" in self.__dict__ or type(self).from_counts is not _FROM_COUNTS:
            return False
        S, K = self.problem.S, self.problem.K
        for t, shape in ((self.zn, (S,)), (self.cc, (K, K)), (self.target, (S, K, K)),
                         (self.weight, (S,))):
            if (type(t) is not torch.Tensor or t.dtype is not torch.float64 or t.shape != shape
                    or t.device != device or t.requires_grad or not t.is_contiguous()):
                return False
        return True

    def __call__(self, logits: torch.Tensor) -> torch.Tensor:
        if logits.is_cuda and self._plain(logits.device):
            return _SoftFitnessSq.apply(logits, self)
        return self.from_counts(SoftPairCounts.apply(logits, self.problem))

    def count_gradient(self, n: torch.Tensor) -> torch.Tensor:
        """d F^2 / d n at pair counts n [..., S, K, K] (closed form)."""
        alpha = 1.0 - (n / self.zn[:, None, None]) / self.cc
        return -2.0 * self.weight[:, None, None] * (alpha - self.target) / (
            self.zn[:, None, None] * self.cc)


_FROM_COUNTS = RelaxObjective.from_counts


def soft_fitness_sq(logits: torch.Tensor, problem) -> torch.Tensor:
    return RelaxObjective(problem, logits.device)(logits)


def site_gain(problem, lattices: torch.Tensor, dn: torch.Tensor) -> torch.Tensor:
    """u [L, N, K] float32: first-order F^2 change of turning each site into
    each species, at the lattices (uint8 [L, N]) with dn = dF^2/dn [L,S,K,K]."""
    L = lattices.shape[0]
    u = torch.empty((L, problem.n_sites, problem.K), dtype=torch.float32, device=lattices.device)
    dn = dn.to(torch.float64).contiguous()
    Nat.check(Nat.lib().hea_site_gain(problem.handle, L, lattices.contiguous().data_ptr(),
                                      dn.data_ptr(), u.data_ptr(), _stream()))
    return u
