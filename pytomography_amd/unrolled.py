"""Unrolled, differentiable BSREM + relative-difference prior.

The forward pass is the reference's BSREM sub-iteration loop
(PreconditionedGradientAscentAlgorithm.__call__, preconditioned_gradient_ascent.py:80-129,
with BSREM's preconditioner :436-474 and RelativeDifferencePrior :156-183):

    y      = x + x * D_m * (B_m(g_m / (H_m x + s_m + delta)) - n_m - r_m(x))
    x_next = y, with y <= floor set to floor            (addition_after_iteration)
    D_m    = relax / (w_m * sum_m n_m + delta),  n_m = B_m 1,  r_m = beta w_m grad V

where H_m is ``SPECTSystemMatrix.forward`` and B_m the reference back
projection ``backward`` (a gather at 270-beta, not the transpose of H_m).

The reverse pass stores only the iterates (one object per sub-iteration) and
recomputes every projection from them: no rotated volume is ever kept.  For
an upstream gradient xbar of x_next, with p = H_m x + s_m + delta,
mu = xbar * [y > floor] and v = x * D_m * mu,

    t       = B_m^T v                                   (spect_backward_transpose)
    gbar_m += t / p
    xbar'   = mu * (1 + D_m * G) + H_m^T(-g_m t / p^2) - J_r^T v
    betabar -= <v, r_m> / beta

with G = B_m(g_m/p) - n_m - r_m, H_m^T the exact adjoint (spect_backward
ADJOINT) and J_r^T the transposed Jacobian of the prior gradient
(spect_rdp_hessian_vjp).  D_m does not depend on g, x_0 or beta.
"""
from __future__ import annotations

from typing import Callable

import torch

import pytomography_amd
from pytomography_amd import _lib


class UnrolledBSREM:
    """BSREM + RDP unrolled over ``n_iters`` x ``n_subsets`` sub-iterations,
    differentiable with respect to the projections g, the initial object x_0
    and the prior weight beta (``__call__`` returns a tensor wired into
    torch.autograd)."""

    def __init__(self, system_matrix, prior, additive_term: torch.Tensor | None = None,
                 n_iters: int = 10, n_subsets: int = 4,
                 relaxation_sequence: Callable = lambda _: 1,
                 addition_after_iteration: float = 1e-4) -> None:
        self.sm = system_matrix
        self.prior = prior
        self.prior.set_object_meta(system_matrix.object_meta)
        self.additive_term = additive_term
        self.n_iters = n_iters
        self.n_subsets = n_subsets
        self.relaxation_sequence = relaxation_sequence
        self.floor = float(addition_after_iteration)
        self._norm_cache: dict = {}
        if n_subsets > 1:
            self.sm.set_n_subsets(n_subsets)

    # ------------------------------------------------------------------ setup
    def _subsets(self):
        return list(range(self.n_subsets)) if self.n_subsets > 1 else [None]

    def _weight(self, k) -> float:
        return 1.0 if k is None else self.sm.get_weighting_subset(k)

    def _norms(self, dt, device):
        """n_m = B_m 1 computed in float64 and rounded to ``dt``, as
        compute_normalization_factor (spect_system_matrix.py:106-118)."""
        key = (dt, str(device))
        if key not in self._norm_cache:
            norms = []
            for k in self._subsets():
                n = self.sm._angle_index(k, device).numel()
                ones = torch.ones((n, *self.sm.proj_meta.shape[1:]), dtype=torch.float64, device=device)
                norms.append(self.sm._backward(ones, k, _lib.BP_REFERENCE).to(dt).contiguous())
            total = torch.stack(norms).sum(axis=0).contiguous()
            self._norm_cache[key] = (norms, total)
        return self._norm_cache[key]

    def _precond(self, n_iter, k, total):
        """D_m in the update kernel's order of operations."""
        return self.relaxation_sequence(n_iter) / (self._weight(k) * total + pytomography_amd.delta)

    def _additive(self, g):
        if self.additive_term is None:
            return torch.zeros_like(g)
        return self.additive_term.to(g.device, g.dtype).contiguous()

    def _ratio(self, g_m, hf, s_m):
        dt = hf.dtype
        pred = torch.empty_like(hf)
        ratio = torch.empty_like(hf)
        _lib.check(_lib.lib().spect_poisson_ratio(
            _lib.dtype_code(dt), g_m.data_ptr(), hf.data_ptr(), s_m.data_ptr(), pred.data_ptr(),
            ratio.data_ptr(), hf.numel(), float(pytomography_amd.delta), _lib.stream_ptr(hf.device)))
        return pred, ratio

    # The iterations and their derivative blur every plane with its own PSF, as
    # backward_transpose does: the operators that are differentiated are the
    # ones that are applied.  (A system matrix with projections of its own -- a
    # subclass's, or a wrapper put on the object or the class -- or on the
    # per-angle path is called as it is.)
    def _own(self, name) -> bool:
        from pytomography_amd.projectors.SPECT.spect_system_matrix import FUSED_PROJECTIONS
        called = getattr(getattr(self.sm, name), "__func__", None)
        return called is not FUSED_PROJECTIONS[name] or not self.sm.fused

    def _forward(self, x, k):
        if self._own("forward"):
            return self.sm.forward(x, k)
        return self.sm._project(x, k, "spect_forward", planes=True)

    def _backward(self, p, k, mode=_lib.BP_REFERENCE):
        name = "backward" if mode == _lib.BP_REFERENCE else "backward_adjoint"
        if self._own(name):
            return getattr(self.sm, name)(p, k)
        return self.sm._backward(p, k, mode, planes=True)

    def _subset_proj(self, t, k):
        return t if k is None else self.sm.get_projection_subset(t, k).contiguous()

    # ---------------------------------------------------------------- forward
    def run(self, g: torch.Tensor, x0: torch.Tensor, beta: float):
        """Returns (x_K, checkpoints): the iterate before every sub-iteration."""
        dt = x0.dtype
        device = x0.device
        g = _lib.require_device_tensor(g, "projections", dt)
        s = self._additive(g)
        norms, total = self._norms(dt, device)
        x = _lib.require_device_tensor(x0.detach(), "object", dt).clone()
        ckpts = []
        for j in range(self.n_iters):
            for k in self._subsets():
                ckpts.append(x.clone())
                w = self._weight(k)
                r = self.prior.gradient(x, beta_scale=w, beta=beta)
                hf = self._forward(x, k)
                _, ratio = self._ratio(self._subset_proj(g, k), hf, self._subset_proj(s, k))
                b = self._backward(ratio, k)
                nk = norms[0 if k is None else k]
                _lib.check(_lib.lib().spect_bsrem_update(
                    _lib.dtype_code(dt), x.data_ptr(), b.data_ptr(), nk.data_ptr(),
                    total.data_ptr(), r.data_ptr(), x.numel(), float(self.relaxation_sequence(j)),
                    float(w), float(pytomography_amd.delta), self.floor, _lib.stream_ptr(device)))
        return x, ckpts

    # ---------------------------------------------------------------- reverse
    def vjp(self, ckpts, g: torch.Tensor, beta: float, xbar: torch.Tensor):
        """Returns (gbar, x0bar, betabar) for upstream gradient ``xbar`` of x_K."""
        dt = ckpts[0].dtype
        device = ckpts[0].device
        g = _lib.require_device_tensor(g, "projections", dt)
        s = self._additive(g)
        norms, total = self._norms(dt, device)
        delta = pytomography_amd.delta
        lam = xbar.detach().to(device, dt).contiguous()
        gbar = torch.zeros_like(g)
        betabar = torch.zeros((), dtype=torch.float64, device=device)
        steps = [(j, k) for j in range(self.n_iters) for k in self._subsets()]
        for (j, k), x in zip(reversed(steps), reversed(ckpts)):
            w = self._weight(k)
            g_m, s_m = self._subset_proj(g, k), self._subset_proj(s, k)
            r = self.prior.gradient(x, beta_scale=w, beta=beta)
            hf = self._forward(x, k)
            pred, ratio = self._ratio(g_m, hf, s_m)
            b = self._backward(ratio, k)
            nk = norms[0 if k is None else k]
            d = self._precond(j, k, total)
            pre = x * d
            G = (b - nk) - r
            y = x + pre * G
            mu = lam * (y > self.floor).to(dt)
            v = (pre * mu).contiguous()
            t = self.sm.backward_transpose(v, k)
            p = pred + delta
            gt = t / p
            if k is None:
                gbar += gt
            else:
                idx = self.sm._angle_index(k, device).long()
                gbar.index_add_(0, idx, gt)
            q = (-(g_m * gt) / p).contiguous()
            lam = mu * (1 + d * G) + self._backward(q, k, _lib.BP_ADJOINT) \
                - self.prior.hessian_vjp(x, v, beta_scale=w, beta=beta)
            if beta != 0:
                betabar -= (v.double() * r.double()).sum() / beta
            else:
                r1 = self.prior.gradient(x, beta_scale=w, beta=1.0)
                betabar -= (v.double() * r1.double()).sum()
        return gbar, lam, float(betabar)

    # --------------------------------------------------------------- autograd
    def __call__(self, projections: torch.Tensor, object_initial: torch.Tensor | None = None,
                 beta: torch.Tensor | float | None = None) -> torch.Tensor:
        dt = projections.dtype
        if object_initial is None:
            object_initial = torch.ones(self.sm._shape, dtype=dt, device=projections.device)
        if beta is None:
            beta = torch.tensor(float(self.prior.beta), dtype=torch.float64)
        if not torch.is_tensor(beta):
            beta = torch.tensor(float(beta), dtype=torch.float64)
        return _UnrolledFunction.apply(object_initial, projections, beta, self)


class _UnrolledFunction(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x0, g, beta, runner):
        b = float(beta)
        xk, ckpts = runner.run(g.detach(), x0.detach(), b)
        ctx.runner = runner
        ctx.ckpts = ckpts
        ctx.beta = b
        ctx.save_for_backward(g)
        ctx.beta_meta = (beta.dtype, beta.device)
        return xk

    @staticmethod
    def backward(ctx, xbar):
        (g,) = ctx.saved_tensors
        gbar, x0bar, bbar = ctx.runner.vjp(ctx.ckpts, g.detach(), ctx.beta, xbar)
        ctx.ckpts = None
        bdt, bdev = ctx.beta_meta
        return x0bar, gbar.to(g.dtype), torch.tensor(bbar, dtype=bdt, device=bdev), None
