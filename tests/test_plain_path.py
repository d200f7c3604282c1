"""Which calls skip the torch.library dispatcher (``hip._plain``), on the CPU, and what of autograd
has to hold where they do."""

from __future__ import annotations

import pytest
import torch
from torch.autograd import forward_ad
from torch.utils._python_dispatch import TorchDispatchMode

import omniwave_amd
from omniwave_amd import hip
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


def test_a_profiler_sees_the_operator() -> None:
    t = torch.ones(3)
    with torch.autograd.profiler.profile():
        assert not _plain(t)
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CPU]):
        assert not _plain(t)
    steps = torch.profiler.schedule(wait=1, warmup=0, active=1, repeat=1)
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CPU], schedule=steps) as prof:
        plain = []
        for _ in range(3):  # waiting, recording, done
            plain.append(_plain(t))
            prof.step()
    assert plain == [True, False, True]
    assert _plain(t)


PARAMS = ("norm_weight", "a_u", "a_v", "a_o", "b_u", "b_v", "b_o", "gamma")


def _block_inputs():
    t = {"x": torch.zeros(1, 4, 4, 64), "norm_weight": torch.ones(64), "gamma": torch.ones(64)}
    t.update({k: torch.zeros(16, 16) for k in ("a_u", "a_v", "a_o")})
    t.update({"b_u": torch.zeros(1, 64, 128), "b_v": torch.zeros(1, 64, 128), "b_o": torch.zeros(1, 128, 64)})
    return {k: v.bfloat16() for k, v in t.items()}, omniwave_amd.build_route_plan(4, 4, 64, 16, 64, "local")


@pytest.mark.parametrize("name", ["x", *PARAMS, "stats_in"])
def test_a_chained_block_loses_no_gradient(monkeypatch, name) -> None:
    """Chained blocks have no backward: a call with an input that requires grad raises, at once or
    when its result is differentiated."""
    monkeypatch.setattr(hip, "_require", lambda *a: None)
    monkeypatch.setattr(hip, "_run_chain", lambda x, *a: (torch.zeros_like(x), torch.zeros(16, 1), True))
    t, plan = _block_inputs()
    t["stats_in"] = torch.zeros(16, 1)
    t[name].requires_grad_(True)

    def step():
        out, _ = hip.bigemm_block_chain_hip(t["x"], t["stats_in"], t["norm_weight"], plan, t["a_u"], t["a_v"], t["a_o"],
                                            t["b_u"], t["b_v"], t["b_o"], t["gamma"])
        assert out.requires_grad
        out.sum().backward()

    with pytest.raises(RuntimeError, match="inference-only|no autograd formula"):
        step()
    with torch.no_grad():
        assert not hip.bigemm_block_chain_hip(t["x"], t["stats_in"], t["norm_weight"], plan, t["a_u"], t["a_v"], t["a_o"],
                                              t["b_u"], t["b_v"], t["b_o"], t["gamma"])[0].requires_grad


@pytest.mark.parametrize("name", ["x", *PARAMS, "drop_scale"])
def test_every_input_that_requires_grad_is_tracked(monkeypatch, name) -> None:
    monkeypatch.setattr(hip, "_require", lambda *a: None)
    monkeypatch.setattr(hip, "_run_forward", lambda x, *a: (torch.zeros_like(x), None))
    t, plan = _block_inputs()
    t["drop_scale"] = torch.ones(1)
    t[name].requires_grad_(True)
    out = hip.bigemm_block_hip(t["x"], t["norm_weight"], plan, *[t[k] for k in PARAMS[1:]], drop_scale=t["drop_scale"])
    assert out.requires_grad
