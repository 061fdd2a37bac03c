"""Casts into a new tensor allocated natively, and through Python where the allocation belongs to others."""

from __future__ import annotations

import pytest
import torch
from torch.overrides import TorchFunctionMode
from torch.utils._python_dispatch import TorchDispatchMode

from oracle import c_oracle

pytestmark = pytest.mark.gpu


def _bits(t):
    return t.detach().cpu().view(torch.uint8)


@pytest.mark.parametrize("dtype", (torch.bfloat16, torch.float16, torch.float8_e4m3fn, torch.float8_e5m2))
@pytest.mark.parametrize("kind", ("tensor", "parameter", "subclass", "mode", "inference", "empty"))
def test_a_cast_output_is_a_plain_tensor_of_the_input_shape(cuda, dtype, kind):
    import sr_states

    class Sub(torch.Tensor):
        pass

    class Mode(TorchFunctionMode):
        calls = 0

        def __torch_function__(self, func, types, args=(), kwargs=None):
            Mode.calls += func is torch.empty_like
            return func(*args, **(kwargs or {}))

    host = torch.randn(0 if kind == "empty" else 33, 7, generator=torch.Generator().manual_seed(1))
    x = host.to(cuda)
    if kind == "parameter":
        x = torch.nn.Parameter(x)
    elif kind == "subclass":
        x = x.as_subclass(Sub)
    if kind == "mode":
        with Mode():
            y = sr_states.cast(x, dtype=dtype, seed=5, offset=2**32 - 3)
        assert Mode.calls == 1
    elif kind == "inference":
        with torch.inference_mode():
            y = sr_states.cast(x, dtype=dtype, seed=5, offset=2**32 - 3)
        assert y.is_inference()
    else:
        y = sr_states.cast(x, dtype=dtype, seed=5, offset=2**32 - 3)
    assert type(y) is (Sub if kind == "subclass" else torch.Tensor) and not y.requires_grad
    assert y.shape == x.shape and y.dtype == dtype and y.device == x.device and y.is_contiguous()
    assert torch.equal(_bits(y), _bits(c_oracle.cast(host, dtype=dtype, seed=5, offset=2**32 - 3)))


def test_a_cast_without_room_raises_the_allocator_error(cuda):
    import sr_states

    x = torch.zeros(64 << 20, device=cuda)
    torch.cuda.empty_cache()
    torch.cuda.set_per_process_memory_fraction(1e-9)
    try:
        with pytest.raises(torch.OutOfMemoryError):
            sr_states.cast(x, dtype=torch.bfloat16)
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)
    assert sr_states.cast(x, dtype=torch.bfloat16).count_nonzero() == 0


def test_a_dispatch_mode_sees_the_allocation_of_empty_like(cuda):
    import sr_states

    class Mode(TorchDispatchMode):
        def __init__(self):
            super().__init__()
            self.calls = []

        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            self.calls.append((func, dict(kwargs or {})))
            return func(*args, **(kwargs or {}))

    x = torch.randn(33, 7, device=cuda)
    with Mode() as expected:
        torch.empty_like(x, dtype=torch.float16, memory_format=torch.contiguous_format)
    with Mode() as seen:
        sr_states.cast(x, dtype=torch.float16, seed=5)
    assert seen.calls == expected.calls
