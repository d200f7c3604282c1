"""fp32 kernels of images past the matrix-core kernels' 32-bit offsets (``-m gpu``), at small shapes: the
dispatch is told that the images don't fit, and the results are compared with float64."""

from __future__ import annotations

import sys

import pytest
import torch

import omniwave_amd
from omniwave_amd import _native, hip
from omniwave_amd.backward import bigemm_backward
from omniwave_amd.hip import bigemm_block_hip, bigemm_delta_hip
from omniwave_amd.routing import plan_key
from oracle.bigemm import bigemm_delta_reference, block_reference, rel_l2
from oracle.routing import build_route_plan as oracle_plan
from test_gpu_bwd_x3 import EPS, FLAGS, reference, rel

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda", 0)
G = 16
CASES = [  # batch, H, W, C, d, rd, route, level, drop-path
    (1, 4, 4, 64, 64, 128, "local", 0, False),      # one tile
    (3, 7, 9, 96, 64, 256, "radix", 2, True),       # cut-off strided group, pad tokens
    (2, 5, 7, 70, 64, 128, "local", 0, False),      # rows that are not 16-byte aligned
    (3, 7, 7, 256, 128, 256, "radix", 1, True),     # strided groups, an odd number of tiles
    (2, 14, 14, 384, 128, 128, "shifted", 0, False),
]
IDS = [f"{b}x{h}x{w}x{c}-d{d}-rd{rd}-{r}{l}" for b, h, w, c, d, rd, r, l, _ in CASES]


def _inputs(b, h, w, c, d, rd, drop):
    gen = torch.Generator().manual_seed(13)
    q_c = -(-c // d)
    normal = lambda *s, fan: torch.randn(*s, generator=gen) / fan ** 0.5
    p = {"norm_weight": torch.rand(c, generator=gen) + 0.5, "gamma": torch.rand(c, generator=gen) + 0.5,
         "a_u": normal(G, G, fan=G), "a_v": normal(G, G, fan=G), "a_o": normal(G, G, fan=G),
         "b_u": normal(q_c, d, rd, fan=d), "b_v": normal(q_c, d, rd, fan=d), "b_o": normal(q_c, rd, d, fan=rd)}
    x, dy = (torch.randn(b, h, w, c, generator=gen) for _ in range(2))
    scale = torch.tensor([1.25, 0.0, 1.25][:b]) if drop else None
    return p, x, dy, scale


@pytest.mark.parametrize("b,h,w,c,d,rd,route,level,drop", CASES, ids=IDS)
def test_forward(monkeypatch, b, h, w, c, d, rd, route, level, drop) -> None:
    print(f"\n[gpu-case] large-image fp32 forward {b}x{h}x{w}x{c} d={d} rd={rd} {route}{level}", file=sys.stderr,
          flush=True)
    plan = omniwave_amd.build_route_plan(h, w, c, G, d, route, level)
    p, x, _, scale = _inputs(b, h, w, c, d, rd, drop)
    monkeypatch.setattr(hip._geometry(plan_key(plan)), "x3", False)
    layouts, pack = [], hip._pack
    monkeypatch.setattr(hip, "_pack", lambda *a: (layouts.append(a[-1]), pack(*a))[1])
    dev = {k: v.to(DEV) for k, v in p.items()}
    nw = dev.pop("norm_weight")
    delta = bigemm_delta_hip(x=x.to(DEV), plan=plan, **dev).cpu()
    out = bigemm_block_hip(x.to(DEV), nw, plan, **dev, eps=EPS, drop_scale=scale.to(DEV) if drop else None).cpu()
    assert layouts == ["", ""]  # the plain fp32 weights, for both calls
    oplan = oracle_plan(h, w, c, G, d, route, level)
    p64 = {k: v.double() for k, v in p.items()}
    branch = block_reference(x.double(), oplan, p64, residual=False)
    del p64["norm_weight"]
    # a chain of 16 + d + rd + 16 fp32 additions at random signs, 2^-24 each, and as much again for the
    # gate's and the folds' roundings, which the later sums average
    tol = 2.0 ** -24 * (2 * (32 + d + rd)) ** 0.5
    assert rel_l2(delta, bigemm_delta_reference(x=x.double(), plan=oplan, **p64)) <= tol
    if drop:
        branch = branch * scale.double().view(b, 1, 1, 1)
        assert torch.equal(out[scale == 0], x[scale == 0])
    slack = (out.double().norm() * 2.0 ** -24 / branch.norm()).item()  # the sum with x
    assert rel_l2(out.double() - x.double(), branch) <= tol + slack


@pytest.mark.parametrize("b,h,w,c,d,rd,route,level,drop", CASES, ids=IDS)
def test_backward(monkeypatch, b, h, w, c, d, rd, route, level, drop) -> None:
    print(f"\n[gpu-case] large-image fp32 backward {b}x{h}x{w}x{c} d={d} rd={rd} {route}{level}", file=sys.stderr,
          flush=True)
    plan = omniwave_amd.build_route_plan(h, w, c, G, d, route, level)
    p, x, dy, scale = _inputs(b, h, w, c, d, rd, drop)
    lib, calls = _native.lib(), []
    gather = lib.ow_bwd_gather
    monkeypatch.setattr(lib, "ow_bwd_x3_fits", lambda *a: 0)
    monkeypatch.setattr(lib, "ow_bwd_gather", lambda *a: (calls.append("gather"), gather(*a))[1])
    dev = {k: v.to(DEV) for k, v in p.items()}
    got = bigemm_backward(dy.to(DEV), x.to(DEV), dev["norm_weight"], dev["gamma"], dev["a_u"], dev["a_v"], dev["a_o"],
                          dev["b_u"], dev["b_v"], dev["b_o"], plan, FLAGS, EPS, scale.to(DEV) if drop else None)
    assert calls == ["gather"]
    slots = b * plan.token_indices.shape[0] * G
    # as in the forward, six products deep, and the sums over the slots
    tol = 2.0 ** -24 * (512 + slots) ** 0.5
    for name, a, e in zip(("x", *p), got, reference(dy, x, p, plan, d, scale)):
        assert rel(a, e) <= tol, name
