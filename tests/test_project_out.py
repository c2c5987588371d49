"""Which output projections go to the chunk kernel (the choice alone, on CPU tensors)."""

import contextlib

import pytest
import torch
import torch.nn.functional as F
import torch.nn.utils.parametrize
from torch.autograd import forward_ad
from torch.overrides import TorchFunctionMode
from torch.utils._python_dispatch import TorchDispatchMode

from dexter_amd.models import attention
from dexter_amd.ops.gfx950 import proj


def _project(monkeypatch, tokens, dim, edit=lambda m: None):
    module = attention.SelfAttention(dim, dim // 64, dtype=torch.float32)
    edit(module)
    calls = []

    def select(family, mode, *args):
        calls.append((family, mode))
        return F.linear

    monkeypatch.setattr(attention, "select", select)
    with torch.no_grad():
        out = module._project_out(torch.randn(1, tokens, dim // 64, 64))
    assert out.shape == (1, tokens, dim)
    return calls


@pytest.mark.parametrize("tokens,dim,chunk", [
    (1, 512, True), (128, 512, True), (129, 512, False), (0, 512, False), (8, 576, False)])
def test_sizes(monkeypatch, tokens, dim, chunk):
    assert _project(monkeypatch, tokens, dim) == ([("gemm", "linear_chunk")] if chunk else [])


# torch turns CUDA autocast off without a device.
@pytest.mark.parametrize("inside", [pytest.param("autocast", marks=pytest.mark.gpu),
                                    "forward_ad", "vmap"])
def test_torch_transforms_keep_torchs_linear(monkeypatch, inside):
    if inside == "vmap":
        calls = []

        def one(x):
            calls.append(_project(monkeypatch, 8, 512))
            return x

        torch.vmap(one, randomness="same")(torch.zeros(2))
        assert calls == [[]]
        return
    with contextlib.ExitStack() as stack:
        stack.enter_context(torch.autocast("cuda", dtype=torch.bfloat16)
                            if inside == "autocast" else forward_ad.dual_level())
        assert inside != "autocast" or torch.is_autocast_enabled("cuda")
        assert _project(monkeypatch, 8, 512) == []


@pytest.mark.parametrize("mode", ["dispatch", "function"])
def test_a_torch_mode_sees_the_projection(monkeypatch, mode):
    seen = []

    class Dispatch(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            seen.append(func)
            return func(*args, **(kwargs or {}))

    class Function(TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            seen.append(func)
            return func(*args, **(kwargs or {}))

    module = attention.SelfAttention(512, 8, dtype=torch.float32)
    calls = []
    monkeypatch.setattr(attention, "select", lambda *args: calls.append(args) or F.linear)
    with torch.no_grad(), Dispatch() if mode == "dispatch" else Function():
        module._project_out(torch.randn(1, 8, 8, 64))
    assert not calls
    assert any(f is F.linear or "mm" in str(f) or "linear" in str(f) for f in seen)


def test_a_default_device_keeps_the_kernel(monkeypatch):
    with torch.device("cpu"):
        assert _project(monkeypatch, 8, 512) == [("gemm", "linear_chunk")]


def test_a_trace_records_torchs_linear(monkeypatch):
    module = attention.SelfAttention(512, 8, dtype=torch.float32).requires_grad_(False)
    monkeypatch.setattr(attention, "select", lambda *args: pytest.fail("kernel under a trace"))
    with torch.no_grad():
        traced = torch.jit.trace(lambda x: module._project_out(x), torch.randn(1, 8, 8, 64),
                                 check_trace=False)
    assert "aten::linear" in str(traced.graph)


def test_a_weight_subclass_keeps_torchs_linear(monkeypatch):
    class Tagged(torch.Tensor):
        pass

    def edit(m):
        w = m.o.weight.data.as_subclass(Tagged)
        del m.o.weight
        m.o.weight = w

    assert _project(monkeypatch, 8, 512, edit) == []


def test_a_parametrized_weight_is_computed_once(monkeypatch):
    """A stateful parametrization (spectral norm in training mode) advances one step a call."""
    class Count(torch.nn.Module):
        steps = 0

        def forward(self, w):
            Count.steps += 1
            return w

    def edit(m):
        torch.nn.utils.parametrize.register_parametrization(m.o, "weight", Count())
        Count.steps = 0

    assert _project(monkeypatch, 8, 512, edit) == [("gemm", "linear_chunk")]
    assert Count.steps == 1


class _OnGpu(torch.Tensor):
    """Passes for a CUDA tensor in the predicate."""
    is_cuda = True


def test_the_kernel_declines_what_its_entry_point_refuses():
    """Each limit of dx_linear_chunk is the predicate's, so such calls keep torch's linear."""
    def takes(rows, cols, step=None, tokens=8):
        step = cols if step is None else step
        store = torch.empty(max((rows - 1) * step + cols, 1), dtype=torch.bfloat16)
        w = torch.as_strided(store, (rows, cols), (step, 1)).as_subclass(_OnGpu)
        x = torch.empty(1, tokens, cols, dtype=torch.bfloat16).as_subclass(_OnGpu)
        return proj._accepts_linear(x, w, None)

    assert takes(512, 512) and takes(512, 512, 520) and takes(16, 512, 2**22 - 8)
    assert not takes(512, 512, 0) and not takes(512, 512, 504)  # expanded, overlapping rows
    assert not takes(16, 512, 2**22)
    assert not takes(0, 512) and not takes(16, 0)
    assert not takes(16, 2**20 + 512) and takes(16, 2**20)


def test_a_pin_that_cannot_be_met_is_raised(monkeypatch):
    """As for every other op; without a pin, no kernel for the call means torch's linear."""
    module = attention.SelfAttention(512, 8, dtype=torch.float32)
    x = torch.randn(1, 8, 8, 64)
    with torch.no_grad():
        plain = module._project_out(x)
        assert torch.equal(plain, F.linear(x.flatten(2), module.o.weight, module.o.bias))
        monkeypatch.setenv("DEXTER_KERNEL", "gemm/linear_chunk:mistyped")
        with pytest.raises(LookupError, match="pinned gemm/linear_chunk:mistyped"):
            module._project_out(x)
