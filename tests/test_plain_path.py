"""Which calls skip the torch.library dispatcher (``hip._plain``), on the CPU."""

from __future__ import annotations

import torch
from torch.autograd import forward_ad
from torch.utils._python_dispatch import TorchDispatchMode

from omniwave_amd.hip import _plain


class _Mode(TorchDispatchMode):
    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        return func(*args, **(kwargs or {}))


class _Sub(torch.Tensor):
    pass


def test_plain_tensors_only() -> None:
    t, p = torch.ones(2), torch.nn.Parameter(torch.ones(2))
    assert _plain(t, p, None)
    assert not _plain(t, t.as_subclass(_Sub))


def test_nothing_that_must_see_the_operator_is_passed_by() -> None:
    t = torch.ones(3)
    with _Mode():
        assert not _plain(t)
    with torch.device("cpu"):  # a torch function mode
        assert not _plain(t)
    with forward_ad.dual_level():
        assert not _plain(t)
    seen = []
    torch.func.vmap(lambda v: (seen.append(_plain(t)), v)[1])(t)
    torch.func.grad(lambda v: (seen.append(_plain(t)), v.sum())[1])(t)
    torch.jit.trace(lambda v: (seen.append(_plain(t)), v + 1)[1], t, check_trace=False)
    assert seen and not any(seen)
    assert _plain(t)
