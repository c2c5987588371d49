"""Queries that span more than 32-bit byte offsets (MI355X): attention kernels that fetch
their query rows through a buffer descriptor, against fp32 on sampled rows."""

from __future__ import annotations

import pytest
import torch

import dexter_amd.ops as ops
from oracle import attention as oatt

from _util import DUAL, GENERAL, PAIRED, SINGLE, WAVE, WIDE, assert_parity, attention_kernel

pytestmark = pytest.mark.gpu


def _check(q, k, v, rows):
    got = ops.blockwise_causal_attention(q, k, v)[:, rows].cpu()
    ref = oatt.blockwise_causal_attention(q[:, rows].cpu(), k.cpu(), v.cpu(), None, 0, None, None,
                                          False, keep_fp32=True)
    assert_parity(got, ref)


def _strided(device, lq, h, d, step):
    """[1, lq, h, d] rows ``step`` elements apart, the rest of the buffer unwritten."""
    base = torch.empty((lq - 1) * step + h * d, device=device, dtype=torch.bfloat16)
    q = torch.as_strided(base, (1, lq, h, d), (0, step, d, 1))
    return q.copy_(torch.randn(1, lq, h, d, device=device))


def _step(rows, span):
    """The least row stride (elements, 16-byte rows) at which `rows` rows reach `span` bytes."""
    return -(-span // (rows - 1) // 16) * 8


def test_wide_heads(device, built_lib):
    """64 heads x 256, 131,136 queries: 4 GiB and 2 MB from the first row to the last."""
    h, d, lq, lk = 64, 256, 131136, 128
    assert attention_kernel(torch.bfloat16, 1, lq, lk, h, d) == WIDE
    q = torch.randn(1, lq, h, d, device=device, dtype=torch.bfloat16)
    k, v = (torch.randn(1, lk, 16, d, device=device, dtype=torch.bfloat16) for _ in range(2))
    _check(q, k, v, [*range(48, 128, 2), *range(lq - 24, lq)])


def test_wide_heads_item_past_a_descriptor(device, built_lib):
    """A q view with 128 rows over 2 GiB: the general kernel, which reads q by pointer."""
    h, d, lq, lk = 32, 256, 130, 300
    assert attention_kernel(torch.bfloat16, 1, lq, lk, h, d) == WIDE
    step = _step(128, 2**31)
    assert attention_kernel(torch.bfloat16, 1, lq, lk, h, d, q_sl=step) == GENERAL
    k, v = (torch.randn(1, lk, h, d, device=device, dtype=torch.bfloat16) for _ in range(2))
    _check(_strided(device, lq, h, d, step), k, v, list(range(lq)))


def test_wave_split(device, built_lib):
    """A q view whose 200 rows span 4 GiB."""
    h, d, lq, lk = 16, 128, 200, 64
    step = _step(lq, 2**32)
    assert attention_kernel(torch.bfloat16, 1, lq, lk, h, d, q_sl=step) == WAVE
    k, v = (torch.randn(1, lk, h, d, device=device, dtype=torch.bfloat16) for _ in range(2))
    _check(_strided(device, lq, h, d, step), k, v, list(range(lq)))


def test_wave_split_item_past_a_descriptor(device, built_lib):
    """32 rows over 2 GiB: the kernel that the call had without the wave split."""
    h, d, lq, lk = 16, 128, 40, 256
    step = _step(32, 2**31)
    assert attention_kernel(torch.bfloat16, 1, lq, lk, h, d, q_sl=step) == DUAL
    k, v = (torch.randn(1, lk, h, d, device=device, dtype=torch.bfloat16) for _ in range(2))
    _check(_strided(device, lq, h, d, step), k, v, list(range(lq)))


def test_paired(device, built_lib):
    """64 heads x 128, 262,272 queries: 4 GiB and 2 MB."""
    h, d, lq, lk = 64, 128, 262272, 64
    assert attention_kernel(torch.bfloat16, 1, lq, lk, h, d) == PAIRED
    q = torch.randn(1, lq, h, d, device=device, dtype=torch.bfloat16)
    k, v = (torch.randn(1, lk, 8, d, device=device, dtype=torch.bfloat16) for _ in range(2))
    _check(q, k, v, [*range(100, 256, 4), *range(lq - 25, lq)])


@pytest.mark.parametrize("d", [64, 128])
def test_paired_item_past_a_descriptor(device, built_lib, d):
    """256 rows over 2 GiB, a call that splits its keys otherwise."""
    h, lq, lk = 48, 300, 1000
    step = _step(256, 2**31)
    assert attention_kernel(torch.bfloat16, 1, lq, lk, h, d) == PAIRED
    assert attention_kernel(torch.bfloat16, 1, lq, lk, h, d, q_sl=step) == SINGLE
    k, v = (torch.randn(1, lk, h, d, device=device, dtype=torch.bfloat16) for _ in range(2))
    _check(_strided(device, lq, h, d, step), k, v, list(range(lq)))


def test_ragged_item_past_a_descriptor(device, built_lib):
    h, d, lq, lens = 48, 128, 257, [900, 0, 100]
    step = _step(256, 2**31)
    assert attention_kernel(torch.bfloat16, 3, lq, lq, h, d, lens=lens, q_sl=step) == SINGLE
    base = torch.empty((lq - 1) * step + 3 * h * d, device=device, dtype=torch.bfloat16)
    q = torch.as_strided(base, (3, lq, h, d), (h * d, step, d, 1))
    q.copy_(torch.randn(3, lq, h, d, device=device))
    k, v = (torch.randn(3, lq, h, d, device=device, dtype=torch.bfloat16) for _ in range(2))
    cache = torch.randn(2, 3, 900, h, d, device=device, dtype=torch.bfloat16)
    got = ops.blockwise_causal_attention_varlen(q, k, v, kv_cache=cache, cache_lens=lens,
                                                block_boundaries=None).cpu()
    for i, c in enumerate(lens):
        ref = oatt.blockwise_causal_attention(q[i:i + 1].cpu(), k[i:i + 1].cpu(), v[i:i + 1].cpu(),
                                              cache[:, i:i + 1].cpu(), c, None, None, False,
                                              keep_fp32=True)
        assert_parity(got[i:i + 1], ref, what=f"seq {i}")
