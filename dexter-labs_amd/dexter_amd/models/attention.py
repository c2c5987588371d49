"""A self-attention layer that calls the path the way DreamZero's DiT does.

Follows ``SelfAttention.forward`` (``models/dreamzero/model.py:158-183``):
project q/k/v, QK-RMSNorm + rotary through ``ops.qk_norm_rope``, read
``cache_len`` **before** appending, append k/v only when ``write``, attend
with ``ops.blockwise_causal_attention`` over the cache plus the new block,
project out. It exists to show the drop-in: nothing here names a kernel, the
registry picks the gfx950 implementations.

With ``write=True`` the prologue and the append run as one kernel
(``KVCache.append_fused``). For decode chunks (at most 128 tokens, ``dim`` a
multiple of 512) the q/k/v projections join them: ``ops.qkv_norm_rope`` runs
the projections, the prologue and the cache write in two kernels, and up to
4096 features the output projection is ``ops.linear_chunk``. Longer
chunks use ``torch.nn.functional.linear`` (hipBLASLt) for the projections and,
with a host cache length, ``ops.qk_norm_rope_attention`` for the prologue,
append and attention in one call.
"""

from __future__ import annotations

import torch
import torch.nn.functional as F
from torch import nn
from torch.autograd import forward_ad
from torch.overrides import _get_current_function_mode_stack
from torch.utils._device import DeviceContext

from .. import ops
from ..registry import NoKernelError, select
from .kv_cache import KVCache


def _computes_only(*params) -> bool:
    """Whether a torch op on ``params`` would do no more than compute (``forward`` runs
    without gradients): no autocast, no forward-mode level, no functorch transform, no
    dispatch or function mode (a default device aside, which leaves a linear alone), no
    trace and no tensor subclass, all of which a kernel called by address passes by."""
    return (not torch.is_autocast_enabled("cuda") and forward_ad._current_level < 0
            and torch._C._functorch.peek_interpreter_stack() is None
            and torch._C._len_torch_dispatch_stack() == 0
            and (torch._C._len_torch_function_stack() == 0
                 or all(type(m) is DeviceContext for m in _get_current_function_mode_stack()))
            and torch._C._get_tracing_state() is None
            and all(p is None or type(p) in (nn.Parameter, torch.Tensor) for p in params))


class SelfAttention(nn.Module):
    def __init__(self, dim: int, heads: int, eps: float = 1e-6,
                 dtype: torch.dtype = torch.bfloat16, device=None) -> None:
        super().__init__()
        if dim % heads:
            raise ValueError("dim must be a multiple of heads")
        self.heads, self.head_dim, self.eps = heads, dim // heads, eps
        kw = dict(dtype=dtype, device=device)
        self.q = nn.Linear(dim, dim, **kw)
        self.k = nn.Linear(dim, dim, **kw)
        self.v = nn.Linear(dim, dim, **kw)
        self.o = nn.Linear(dim, dim, **kw)
        # Wan's QK norm spans the full dim (applied before the head split).
        self.q_norm = nn.Parameter(torch.ones(dim, **kw))
        self.k_norm = nn.Parameter(torch.ones(dim, **kw))

    @torch.no_grad()
    def forward(self, x: torch.Tensor, cos: torch.Tensor, sin: torch.Tensor,
                kv_cache: KVCache | None, layer: int,
                block_boundaries: torch.Tensor | None = None, write: bool = False,
                fused_append: bool = True, fused_qkv: bool = True) -> torch.Tensor:
        b, seq, dim = x.shape
        shape = (b, seq, self.heads, self.head_dim)
        # Read before appending; with a device cursor this is the cursor itself,
        # which the commit after all layers advances.
        cache_len = kv_cache.cache_len if kv_cache is not None else 0
        append = kv_cache is not None and write

        if fused_qkv and b * seq <= 128 and dim % 512 == 0 and self.head_dim % 16 == 0:
            if append:
                kv_cache._check_room(seq)
            q, k, v = ops.qkv_norm_rope(
                x, self.q.weight, self.q.bias, self.k.weight, self.k.bias, self.v.weight,
                self.v.bias, self.q_norm, self.k_norm, cos, sin, self.heads, self.eps,
                cache=kv_cache.cache[layer] if append else None,
                start=kv_cache._start() if append else 0,
                status=kv_cache.status if append else None)
            return self._attend(q, k, v, kv_cache, layer, cache_len, block_boundaries)

        q = F.linear(x, self.q.weight, self.q.bias).view(shape)
        k = F.linear(x, self.k.weight, self.k.bias).view(shape)
        v = F.linear(x, self.v.weight, self.v.bias).view(shape)
        if fused_append and not isinstance(cache_len, torch.Tensor):
            if append:
                kv_cache._check_room(seq)
            out = ops.qk_norm_rope_attention(
                q, k, v, self.q_norm, self.k_norm, cos, sin,
                kv_cache=kv_cache.cache[layer] if kv_cache is not None else None,
                cache_len=cache_len, append=append, block_boundaries=block_boundaries,
                eps=self.eps)
            return self._project_out(out)
        if append and fused_append:
            q, k = kv_cache.append_fused(layer, q, k, v, self.q_norm, self.k_norm, cos, sin,
                                         self.eps)
        else:
            q, k = ops.qk_norm_rope(q, k, self.q_norm, self.k_norm, cos, sin, self.eps)
            if append:
                kv_cache.append(layer, k, v)
        return self._attend(q, k, v, kv_cache, layer, cache_len, block_boundaries)

    def _attend(self, q, k, v, kv_cache, layer, cache_len, block_boundaries):
        out = ops.blockwise_causal_attention(
            q, k, v,
            kv_cache=kv_cache.cache[layer] if kv_cache is not None else None,
            cache_len=cache_len,
            block_boundaries=block_boundaries,
        )
        return self._project_out(out)

    def _project_out(self, out):
        # Decode chunks up to 4096 features go to the chunk GEMM (83 x 3072: 11.8 against
        # 16.7 us); at 5120 it and hipBLASLt are mixed.
        x = out.flatten(2)
        b, seq, dim = x.shape
        weight, bias = self.o.weight, self.o.bias  # read once: a parametrization computes them
        linear = F.linear
        if 0 < b * seq <= 128 and dim % 512 == 0 and dim <= 4096 and _computes_only(weight, bias):
            try:
                linear = select("gemm", "linear_chunk", x, weight, bias)
            except NoKernelError:  # a weight layout the kernel does not take
                pass
        return linear(x, weight, bias)
