"""mHC residual hyper-connections (hc_mult = 4) on the fused gfx950 mixing kernels.

The reference configures manifold-constrained hyper-connections for its DeepSeek block (hc_mult = 4,
hc_sinkhorn_iters = 20, hc_eps = 1e-6; baseline/indexer.py:48-50) and ships their 4x4 Sinkhorn projection as
an operator of its own (baseline/sinkhorn.py).  HyperConnection keeps the four residual streams of a token,
x [N, 4, C], and computes per token, from the RMS-normalised flattened streams,
    logits = alpha * (x_norm @ phi) + base   ->  pre [4], post [4], res [4, 4];
the layer input h = sigmoid(pre) . x runs in ks_mhc_pre, and the residual update
    x' = Sinkhorn(res) x + 2 sigmoid(post) f(h)
in ks_mhc_post, whose kernel normalises each token's 4x4 logits in registers (the Sinkhorn of
torch.ops.ks_mi355x.sinkhorn, repeat = hc_sinkhorn_iters) and mixes the streams in the same pass.  Where nothing
has to be differentiated or traced, the logits are formed on the way too (ks_mhc_input); otherwise they stay torch
operations (`logits`), through which gradients reach phi, alpha and base.
"""
from __future__ import annotations

import torch
import torch.nn as nn
from torch.autograd import forward_ad

from . import _lib


class HyperConnection(nn.Module):
    def __init__(self, dim: int, hc_mult: int = 4, hc_sinkhorn_iters: int = 20, hc_eps: float = 1e-6,
                 norm_eps: float = 1e-6):
        super().__init__()
        if hc_mult != 4:
            raise ValueError("the fused mixing kernels are built for hc_mult = 4")
        n = hc_mult
        self.dim, self.hc_mult = dim, n
        self.hc_sinkhorn_iters, self.hc_eps, self.norm_eps = hc_sinkhorn_iters, hc_eps, norm_eps
        self.phi = nn.Parameter(torch.randn(n * dim, 2 * n + n * n) * (n * dim) ** -0.5)
        self.alpha = nn.Parameter(torch.full((3,), 0.1))
        self.base = nn.Parameter(torch.zeros(2 * n + n * n))

    def logits(self, x: torch.Tensor):
        """(pre [N, 4], post [N, 4], res [N, 4, 4]) float32 from the streams x bf16 [N, 4, C]."""
        n = self.hc_mult
        xf = x.flatten(1).float()
        xn = xf * torch.rsqrt(xf.pow(2).mean(-1, keepdim=True) + self.norm_eps)
        z = xn @ self.phi
        pre = self.alpha[0] * z[:, :n] + self.base[:n]
        post = self.alpha[1] * z[:, n:2 * n] + self.base[n:2 * n]
        res = (self.alpha[2] * z[:, 2 * n:] + self.base[2 * n:]).view(-1, n, n)
        return pre.contiguous(), post.contiguous(), res.contiguous()

    def _fused(self, x: torch.Tensor) -> bool:
        """Whether `pre` may form the logits inside the kernel: plain contiguous tensors of the kernel's types on one
        GPU, with no gradient (reverse or forward mode), autocast, vmap, trace or dispatch mode that has to see the torch
        operations, and no `logits` of a subclass's or the instance's own."""
        if type(self).logits is not HyperConnection.logits or "logits" in self.__dict__:
            return False
        if not isinstance(self.norm_eps, (int, float)):
            return False
        ts = (x, self.phi, self.alpha, self.base)
        if any(type(t) not in (torch.Tensor, nn.Parameter) for t in ts):  # a tracer's proxies too, before any is asked
            return False
        if torch.compiler.is_compiling() or torch.jit.is_tracing() or torch._C._functorch.maybe_current_level() is not None:
            return False
        if torch.is_autocast_enabled() or forward_ad._current_level >= 0 or torch._C._len_torch_dispatch_stack() > 0:
            return False
        if torch.is_grad_enabled() and any(t.requires_grad for t in ts):
            return False
        return (all(t.is_cuda and t.device == x.device and t.is_contiguous() for t in ts)
                and x.dtype == torch.bfloat16 and x.dim() == 3 and x.shape[0] > 0 and x.shape[1:] == (4, self.dim)
                and self.dim % 8 == 0 and all(t.dtype == torch.float32 for t in ts[1:])
                and self.phi.shape == (4 * self.dim, 24) and self.alpha.shape == (3,) and self.base.shape == (24,))

    def pre(self, x: torch.Tensor):
        """The layer input h bf16 [N, C] and the logits the residual update needs."""
        if self._fused(x):
            return _lib.torch_ops().mhc_input(x, self.phi, self.alpha, self.base, self.norm_eps)
        pre, post, res = self.logits(x)
        return _lib.torch_ops().mhc_pre(x, pre), post, res

    def post(self, x: torch.Tensor, f: torch.Tensor, post: torch.Tensor, res: torch.Tensor) -> torch.Tensor:
        """The next streams x' bf16 [N, 4, C] from the layer output f bf16 [N, C]."""
        return _lib.torch_ops().mhc_post(x, f, res, post, self.hc_sinkhorn_iters, self.hc_eps)

    def forward(self, x: torch.Tensor, layer) -> torch.Tensor:
        h, post, res = self.pre(x)
        return self.post(x, layer(h), post, res)
