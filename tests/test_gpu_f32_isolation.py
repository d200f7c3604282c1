"""fp32 token groups stay apart (``-m gpu``): a value that is no number, or the largest one, in one
token group changes no other group's result.

The three-part kernels form two token groups in one matrix product, and with an odd number of groups
per image (14x14: 13) the two belong to different images.  The operator's other reach across groups
is the sum of the parameter gradients, so those aren't compared here.
"""

from __future__ import annotations

import math
import sys

import pytest
import torch

import omniwave_amd
from omniwave_amd import _native
from omniwave_amd.backward import bigemm_backward
from omniwave_amd.hip import bigemm_block_hip, bigemm_delta_hip

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda", 0)
G = 16
EPS = 1e-6
FLAGS = _native.OW_FUSE_NORM | _native.OW_FUSE_RESIDUAL
LARGEST = torch.finfo(torch.float32).max
ODD = [math.nan, math.inf, LARGEST]
IDS = ["nan", "inf", "largest"]
CASES = [  # batch, H, W, C, d, rd, route, level
    (2, 14, 14, 512, 128, 256, "local", 0),      # split in four: a wave's pair holds both images' tiles
    (16, 14, 14, 512, 128, 256, "shifted", 0),   # split in two
    (20, 14, 14, 512, 128, 256, "radix", 1),     # whole pairs per wave
    (3, 4, 4, 128, 64, 128, "radix", 1),         # one tile per image
    (60, 14, 14, 256, 64, 128, "local", 0),      # d = 64, whole pairs per wave
]
CASE_IDS = [f"{b}x{h}x{w}x{c}-d{d}-{r}{l}" for b, h, w, c, d, rd, r, l in CASES]


def _inputs(b, h, w, c, d, rd, route, level):
    gen = torch.Generator().manual_seed(5)
    plan = omniwave_amd.build_route_plan(h, w, c, G, d, route, level)
    q_c = -(-c // d)
    normal = lambda *s, fan: (torch.randn(*s, generator=gen) / fan ** 0.5).to(DEV)
    p = {"a_u": normal(G, G, fan=G), "a_v": normal(G, G, fan=G), "a_o": normal(G, G, fan=G),
         "b_u": normal(q_c, d, rd, fan=d), "b_v": normal(q_c, d, rd, fan=d), "b_o": normal(q_c, rd, d, fan=rd),
         "gamma": torch.rand(c, generator=gen).to(DEV) + 0.5}
    x, dy = (torch.randn(b, h, w, c, generator=gen).to(DEV) for _ in range(2))
    return plan, p, torch.rand(c, generator=gen).to(DEV) + 0.5, x, dy


def _outside(plan, b, image, token):
    """[b, H * W]: the rows that share no token group with ``token`` of ``image``."""
    tok = torch.as_tensor(plan.token_indices).long().reshape(-1, G)
    group = tok[(tok == token).any(dim=1)].reshape(-1)
    n_tok = plan.height * plan.width
    keep = torch.ones(b, n_tok, dtype=torch.bool)
    keep[image, group[(group >= 0) & (group < n_tok)]] = False
    return keep.to(DEV)


def _touched(plan):
    """A token of the last group of image 0: with an odd number of groups it shares a pair with
    image 1's first."""
    last = torch.as_tensor(plan.token_indices).long().reshape(-1, G)[-1]
    return 0, int(last[(last >= 0) & (last < plan.height * plan.width)][0])


@pytest.mark.parametrize("value", ODD, ids=IDS)
@pytest.mark.parametrize("b,h,w,c,d,rd,route,level", CASES, ids=CASE_IDS)
def test_forward_keeps_groups_apart(b, h, w, c, d, rd, route, level, value) -> None:
    print(f"\n[gpu-case] isolation forward {b}x{h}x{w}x{c} d={d} {route}{level} {value}", file=sys.stderr, flush=True)
    plan, p, nw, x, _ = _inputs(b, h, w, c, d, rd, route, level)
    image, token = _touched(plan)
    bad = x.clone()
    bad.view(b, h * w, c)[image, token, 1] = value
    keep = _outside(plan, b, image, token)
    for run in (lambda t: bigemm_delta_hip(x=t, plan=plan, **p),
                lambda t: bigemm_block_hip(t, nw, plan, **p, eps=EPS)):
        want, got = run(x).view(b, h * w, c), run(bad).view(b, h * w, c)
        assert torch.equal(got[keep], want[keep])
        if value != LARGEST:
            assert not got[image, token].isfinite().all()
    # a dropped image passes through untouched beside one that is no number
    scale = torch.ones(b, device=DEV)
    scale[1:] = 0.0
    out = bigemm_block_hip(bad, nw, plan, **p, eps=EPS, drop_scale=scale)
    assert torch.equal(out[1:], x[1:])


@pytest.mark.parametrize("where", ["x", "dy"])
@pytest.mark.parametrize("value", ODD, ids=IDS)
@pytest.mark.parametrize("b,h,w,c,d,rd,route,level", CASES, ids=CASE_IDS)
def test_backward_keeps_groups_apart(b, h, w, c, d, rd, route, level, value, where) -> None:
    print(f"\n[gpu-case] isolation backward {b}x{h}x{w}x{c} d={d} {route}{level} {value} in {where}", file=sys.stderr,
          flush=True)
    plan, p, nw, x, dy = _inputs(b, h, w, c, d, rd, route, level)
    image, token = _touched(plan)
    bad = {"x": x, "dy": dy}
    bad[where] = bad[where].clone()
    bad[where].view(b, h * w, c)[image, token, 1] = value
    keep = _outside(plan, b, image, token)
    args = (p["gamma"], p["a_u"], p["a_v"], p["a_o"], p["b_u"], p["b_v"], p["b_o"], plan)
    for weight, flags in ((nw, FLAGS), (None, 0)):
        dx = lambda g, t: bigemm_backward(g, t, weight, *args, flags, EPS)[0].view(b, h * w, c)
        want, got = dx(dy, x), dx(bad["dy"], bad["x"])
        assert torch.equal(got[keep], want[keep])


# Tensor of the largest values, and the scales of others that keep every product and sum a number.
LARGE = [("x", {"a_u": -30, "a_v": -30, "b_u": -98, "b_v": -98}), ("b_o", {"b_u": -35, "b_v": -35}),
         ("a_o", {"b_o": -60})]


def _large(t):
    """Values of either sign that round up to infinity in bf16."""
    gen = torch.Generator().manual_seed(6)
    sign = torch.where(torch.rand(t.shape, generator=gen) < 0.5, -1.0, 1.0)
    big = sign * LARGEST * (1.0 - 2.0 ** -10 * torch.rand(t.shape, generator=gen))
    assert big.bfloat16().isinf().all()
    return big.to(DEV)


@pytest.mark.parametrize("name,scales", LARGE, ids=[name for name, _ in LARGE])
@pytest.mark.parametrize("d,c", [(128, 512), (64, 256)])
def test_largest_values_are_numbers(d, c, name, scales) -> None:
    """delta with one tensor of the largest fp32 values against float64."""
    plan, p, _, x, _ = _inputs(2, 14, 14, c, d, 2 * d, "local", 0)
    w = {k: v * 2.0 ** scales.get(k, 0) for k, v in {**p, "x": x, "gamma": torch.ones(c, device=DEV)}.items()}
    w[name] = _large(w[name])
    x = w.pop("x")
    got = bigemm_delta_hip(x=x, plan=plan, **w).cpu().double()
    tok = torch.as_tensor(plan.token_indices).long().reshape(-1)
    n = 14 * 14
    live = (tok >= 0) & (tok < n)
    t = x.double().cpu().view(2, n, c)[:, tok.clamp(0, n - 1)] * live[:, None]
    t = t.reshape(2, -1, G, c // d, d).permute(0, 1, 3, 2, 4)
    w64 = {k: v.double().cpu() for k, v in w.items()}
    u, v = w64["a_u"] @ t @ w64["b_u"], w64["a_v"] @ t @ w64["b_v"]
    o = w64["a_o"] @ (torch.nn.functional.silu(u) * v @ w64["b_o"])
    o = o.permute(0, 1, 3, 2, 4).reshape(2, -1, c)
    want = torch.zeros(2, n, c, dtype=torch.float64).index_copy(1, tok[live], o[:, live])
    assert got.isfinite().all()
    # the bound of the three-part forward (sqrt(4 * 96) roundings of 2^-24)
    assert (got.view(2, n, c) - want).norm() <= 1.2e-6 * want.norm()


@pytest.mark.parametrize("name,scales", [LARGE[0], ("dy", {"a_o": -100, "b_o": -60})], ids=["x", "dy"])
@pytest.mark.parametrize("d,c", [(128, 512), (64, 256)])
def test_largest_values_have_gradients(d, c, name, scales) -> None:
    """Gradients of the operator that are numbers."""
    plan, p, _, x, dy = _inputs(2, 14, 14, c, d, 2 * d, "local", 0)
    w = {k: v * 2.0 ** scales.get(k, 0) for k, v in {**p, "x": x, "dy": dy}.items()}
    w[name] = _large(w[name])
    grads = bigemm_backward(w["dy"], w["x"], None, w["gamma"], w["a_u"], w["a_v"], w["a_o"], w["b_u"], w["b_v"], w["b_o"],
                            plan, 0, EPS)
    assert grads[1] is None and all(g.isfinite().all() for g in grads[:1] + grads[2:])


def test_gate_of_large_products() -> None:
    """U far below zero beside a V so large that U V overflows: silu(U) is zero and so is delta.
    A = I, every weight of B_u -1e20 / d and of B_v 1e20 / d: U = -1e20, V = 1e20 for x = 1."""
    d, c, rd = 128, 128, 256
    plan = omniwave_amd.build_route_plan(8, 8, c, G, d, "local", 0)
    eye = torch.eye(G, device=DEV)
    b_u = torch.full((1, d, rd), -1e20 / d, device=DEV)
    delta = bigemm_delta_hip(x=torch.ones(2, 8, 8, c, device=DEV), plan=plan, a_u=eye, a_v=eye, a_o=eye, b_u=b_u, b_v=-b_u,
                             b_o=torch.ones(1, rd, d, device=DEV), gamma=torch.ones(c, device=DEV))
    assert not delta.any()
