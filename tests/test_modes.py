"""What keeps an operation apart from the kernels (CPU only): modes and
transforms that follow torch operations are noticed, a default device is not
one of them, and a torch without the names that are asked composes the
operations instead of raising."""
from __future__ import annotations

import pytest
import torch
from torch.overrides import TorchFunctionMode
from torch.utils._python_dispatch import TorchDispatchMode

from nibblegemm_amd import ops, quant


class Functions(TorchFunctionMode):
    def __torch_function__(self, func, types, args=(), kwargs=None):
        return func(*args, **(kwargs or {}))


class Dispatch(TorchDispatchMode):
    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        return func(*args, **(kwargs or {}))


def test_modes_and_transforms_are_noticed():
    t = torch.ones(4)
    assert not quant.modes_follow() and not ops._tracked(t)
    with torch.device("cpu"):
        assert not quant.modes_follow()
        with Functions():
            assert quant.modes_follow()
    for mode in (Functions(), Dispatch()):
        with mode:
            assert quant.modes_follow() and ops._tracked(t)
    seen = []
    torch.vmap(lambda b: seen.append(quant.modes_follow()) or b + 1)(torch.ones(2, 3))
    torch.jit.trace(lambda b: seen.append(quant.modes_follow()) or b + 1, t, check_trace=False)
    assert seen == [True, True]
    with torch.autograd.forward_ad.dual_level():
        assert ops._tracked(t)
    assert ops._tracked(t.requires_grad_())
    with torch.no_grad():
        assert not ops._tracked(t)


@pytest.mark.parametrize("missing", ["_functorch", "_len_torch_dispatch_stack", "_len_torch_function_stack",
                                     "_is_tracing", "_get_function_stack_at"])
def test_a_torch_without_a_name_composes(monkeypatch, missing):
    class Other:
        def __getattr__(self, name):
            if name == missing:
                raise AttributeError(name)
            return getattr(torch._C, name)

    assert quant._mode_probes(torch._C) is not None
    assert quant._mode_probes(Other()) is None
    monkeypatch.setattr(quant, "_PROBES", None)
    assert ops._tracked(torch.ones(4))


def test_a_torch_without_forward_levels_composes(monkeypatch):
    monkeypatch.delattr(torch.autograd.forward_ad, "_current_level")
    assert ops._tracked(torch.ones(4))
