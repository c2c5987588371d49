"""Host-side shape rules of the norm ops, compared with torch's own (no GPU)."""

import itertools

import pytest
import torch

from dexter_amd.ops.gfx950 import norm
from dexter_amd.ops.gfx950._common import flat_as, rows_ok

SHAPES = [(2, 3, 8), (1, 3, 8), (2, 1, 8), (1, 1, 8), (2, 3, 1), (3, 8), (1, 8), (8,), (1,), (),
          (2, 1, 3, 8), (4, 2, 3, 8), (0, 3, 8), (2, 5, 8)]


@pytest.mark.parametrize("shapes", itertools.product(SHAPES, SHAPES, [(2, 3, 8), (8,)]))
def test_broadcast_is_torchs(shapes):
    sizes = [torch.Size(s) for s in shapes]
    try:
        want = torch.broadcast_shapes(*sizes)
    except RuntimeError:
        with pytest.raises(RuntimeError):
            norm._broadcast(*sizes)
        return
    got = norm._broadcast(*sizes)
    assert got == want and isinstance(got, torch.Size)


def _forms():
    base = torch.arange(4 * 6 * 5 * 16, dtype=torch.float32).reshape(4, 6, 5, 16)
    for shape in [(4, 5, 16), (1, 5, 16), (4, 1, 16), (1, 1, 16), (4, 5, 1)]:
        b, seq, cols = shape
        for t in (base[:b, 0, :seq, :cols], base[:b, 2, :seq, :cols], base[:b, :seq, 0, :cols],
                  base[:1, 1, :1, :cols], base[0, 0, :seq, :cols], base[0, 1, :1, :cols],
                  base[1, 1, 1, :cols], base[:b, 0, :seq, :1], base[0, 0, 0, 0],
                  base[:b, 0, :seq, :cols].transpose(0, 1).contiguous().transpose(0, 1),
                  base.transpose(2, 3)[:b, 0, :cols, :seq].transpose(1, 2),
                  base[:b, 0, :seq, :cols * 2:2] if cols > 1 else base[:b, 0, :seq, :1],
                  base[:b, 0, :1, :cols].expand(b, seq, cols)):
            yield t, torch.Size(shape)


@pytest.mark.parametrize("t,shape", list(_forms()))
def test_rows_read_the_expanded_operand(t, shape):
    try:
        want = t.expand(shape)
    except RuntimeError:
        pytest.skip("operand does not broadcast to this shape")
    b, seq = norm._row_grid(shape)
    rows, sb, sl = norm._rows3(t, shape, b, seq)
    got = rows.as_strided((b, seq, shape[-1]), (sb, sl, 1))
    assert torch.equal(got, want.reshape(b, seq, shape[-1]))
    assert (sb == 0 or b > 1) and (sl == 0 or seq > 1)


def test_rows_of_a_batch_past_the_grid_limit():
    shape = torch.Size((norm._MAX_BATCH_GRID + 1, 2, 8))
    t = torch.arange(2 * 8, dtype=torch.float32).reshape(1, 2, 8)
    b, seq = norm._row_grid(shape)
    rows, sb, sl = norm._rows3(t, shape, b, seq)
    assert (b, seq) == (1, shape[0] * 2) and sb == 0
    assert torch.equal(rows.as_strided((seq, 8), (sl, 1))[-2:], t[0])


@pytest.mark.parametrize("t,ok", [
    (torch.zeros(2, 3, 8, dtype=torch.bfloat16), True),
    (torch.zeros(2, 3, 9, dtype=torch.bfloat16)[..., :8], False),
    (torch.zeros(1, 1, 9, dtype=torch.bfloat16)[..., :8], True),
    (torch.zeros(2, 8, 3, dtype=torch.bfloat16).transpose(1, 2), False),
    (torch.zeros(2, 8, 1, dtype=torch.bfloat16), False),
    (torch.zeros(24, dtype=torch.bfloat16)[1:17].view(2, 8), False),
    (torch.zeros(2, 3, 4), True),
])
def test_rows_ok(t, ok):
    assert rows_ok(t) is ok


@pytest.mark.parametrize("t", [torch.arange(12.0), torch.arange(12.0).view(3, 4),
                               torch.arange(24.0)[::2], torch.arange(12), torch.tensor(3.0)])
def test_flat_as(t):
    got = flat_as(t, torch.device("cpu"), torch.float32)
    assert got.is_contiguous() and got.dim() == 1 and got.dtype == torch.float32
    assert torch.equal(got, t.reshape(-1).float())
