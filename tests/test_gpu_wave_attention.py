"""The wave-split attention kernel (small calls: one launch, key tiles dealt to a
workgroup's waves) against the fp32 oracle and the general kernels (MI355X).

Sizes sit at the edges of its tiles: 32 queries per work item, 32 keys per tile,
8 waves (4 when there are more work items than CUs), one or two tiles held per
wave, a cache end inside a tile. The parity bar is the other kernels' own
(max-abs 2e-2, mean-abs 2e-3 against fp32).
"""

from __future__ import annotations

import pytest
import torch

import dexter_amd.ops as ops
from dexter_amd.ops.gfx950 import _lib
from oracle import attention as oatt

from _util import assert_parity

pytestmark = pytest.mark.gpu
WAVE = 5  # DX_TUNE_ATTN_KERNEL


def _rand(shape, dtype, scale=1.0, seed=0):
    g = torch.Generator().manual_seed(seed)
    return (torch.randn(shape, generator=g) * scale).to(dtype)


def _wave(*args, **kw):
    with _lib.tuning(_lib.TUNE_ATTN_KERNEL, WAVE):
        return ops.blockwise_causal_attention(*args, **kw)


# (Lq, Lk, cache, heads, kv_heads, batch, block starts or "causal")
SHAPES = [
    (1, 1, 0, 2, 2, 1, None), (31, 32, 0, 2, 1, 1, None), (33, 33, 31, 2, 2, 2, None),
    (32, 257, 0, 4, 2, 1, None), (83, 512, 0, 4, 4, 1, None), (83, 83, 1245, 2, 2, 1, None),
    (16, 1100, 0, 2, 2, 1, None), (99, 99, 70, 2, 2, 1, [0, 83]), (64, 64, 33, 4, 4, 1, "causal"),
    (300, 300, 0, 4, 2, 1, "causal"), (130, 130, 40, 2, 2, 2, [0, 50, 100]),
    (96, 96, 20, 2, 2, 1, [40, 0, 70]), (80, 80, 10, 2, 2, 1, [-30, 20]),
    (300, 300, 0, 40, 40, 1, "causal"),  # 400 work items: four waves each
    (257, 65, 0, 40, 8, 1, None),        # 360, cross-attention
]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("dim", [64, 128])
@pytest.mark.parametrize("lq,lk,cache_len,h,hkv,b,mask", SHAPES)
def test_edges(device, built_lib, dtype, dim, lq, lk, cache_len, h, hkv, b, mask):
    q = _rand((b, lq, h, dim), dtype, 0.5, 1)
    # k and v as slices of one projection: row strides other than H*D.
    kv = _rand((b, lk, 2, hkv, dim), dtype, 1.0, 2)
    cache = _rand((2, b, cache_len + 5, hkv, dim), dtype, 0.7, 3) if cache_len else None
    bb = torch.tensor(mask) if isinstance(mask, list) else None
    causal = mask == "causal"
    ref = oatt.blockwise_causal_attention(q, kv[:, :, 0], kv[:, :, 1], cache, cache_len, bb, None,
                                          causal, keep_fp32=True)
    dev = lambda t: None if t is None else t.to(device)  # noqa: E731
    kvd = dev(kv)
    kw = dict(kv_cache=dev(cache), cache_len=cache_len, block_boundaries=dev(bb), causal=causal)
    # q head-major in memory: another order of strides.
    qd = dev(q).transpose(1, 2).contiguous().transpose(1, 2)
    got = _wave(qd, kvd[:, :, 0], kvd[:, :, 1], **kw)
    again = _wave(qd, kvd[:, :, 0], kvd[:, :, 1], **kw)
    seen = ~torch.isnan(ref)
    assert torch.equal(torch.isnan(got.cpu()), ~seen)
    assert_parity(got.cpu()[seen], ref[seen], what=f"{dtype} D={dim} {lq}x{lk}+{cache_len} {mask}")
    assert torch.equal(got.cpu()[seen], again.cpu()[seen])
    with _lib.tuning(_lib.TUNE_ATTN_KERNEL, 3):
        other = ops.blockwise_causal_attention(qd, kvd[:, :, 0], kvd[:, :, 1], **kw)
    assert_parity(got.cpu()[seen], other.cpu()[seen].float(), what="against the paired kernel")


@pytest.mark.parametrize("scale", [-0.09, 0.0])
def test_scales_and_cursor(device, built_lib, scale):
    q, k, v = (_rand((1, 83, 4, 128), torch.bfloat16, 1.0, s).to(device) for s in (1, 2, 3))
    cache = _rand((2, 1, 400, 4, 128), torch.bfloat16, 1.0, 4).to(device)
    ref = oatt.blockwise_causal_attention(q.cpu(), k.cpu(), v.cpu(), cache.cpu(), 290, None, scale,
                                          False, keep_fp32=True)
    cursor = torch.tensor([290], dtype=torch.int32, device=device)
    got = _wave(q, k, v, kv_cache=cache, cache_len=cursor, softmax_scale=scale)
    assert_parity(got, ref)
    assert torch.equal(got, _wave(q, k, v, kv_cache=cache, cache_len=290, softmax_scale=scale))


@pytest.mark.parametrize("dim", [64, 128])
def test_ragged(device, built_lib, dim):
    lens = [0, 100, 333]
    q, k, v = (_rand((3, 99, 4, dim), torch.bfloat16, 0.5, s).to(device) for s in (1, 2, 3))
    cache = _rand((2, 3, 340, 4, dim), torch.bfloat16, 1.0, 4).to(device)
    bb = torch.tensor([0, 83], device=device)
    with _lib.tuning(_lib.TUNE_ATTN_KERNEL, WAVE):
        got = ops.blockwise_causal_attention_varlen(q, k, v, kv_cache=cache, cache_lens=lens,
                                                    block_boundaries=bb)
    for i, c in enumerate(lens):
        ref = oatt.blockwise_causal_attention(q[i:i + 1].cpu(), k[i:i + 1].cpu(), v[i:i + 1].cpu(),
                                              cache[:, i:i + 1].cpu(), c, bb.cpu(), None, False,
                                              keep_fp32=True)
        assert_parity(got[i:i + 1], ref, what=f"seq {i}")


def test_future_keys_never_reach_the_result(device, built_lib):
    """Inf and NaN in keys that a work item cannot see leave its rows bit for bit."""
    q, k, v = (_rand((1, 96, 2, 128), torch.bfloat16, 1.0, s).to(device) for s in (1, 2, 3))
    bb = torch.tensor([0, 32, 64], device=device)
    base = _wave(q, k, v, block_boundaries=bb)
    k2, v2 = k.clone(), v.clone()
    k2[:, 64:], v2[:, 64:] = float("inf"), float("nan")
    got = _wave(q, k2, v2, block_boundaries=bb)
    assert torch.equal(got[:, :64], base[:, :64])


def test_small_calls_take_it_by_default(device, built_lib):
    """The planner's choice equals the forced kernel bit for bit where it fits."""
    q = _rand((1, 300, 16, 128), torch.bfloat16, 1.0, 1).to(device)
    k, v = (_rand((1, 300, 8, 128), torch.bfloat16, 1.0, s).to(device) for s in (2, 3))
    assert torch.equal(ops.blockwise_causal_attention(q, k, v, causal=True),
                       _wave(q, k, v, causal=True))
