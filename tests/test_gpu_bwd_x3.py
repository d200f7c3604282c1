"""fp32 backward on the three-part kernels (``-m gpu``) against float64 autograd: one tile, an odd
number of tiles (half a pair), pairs that fill no workgroup, several ranges of slots, both tile
widths and expansions, strided and cut-off channel groups, pad slots, drop-path."""

from __future__ import annotations

import sys

import pytest
import torch

import omniwave_amd
import omniwave_amd.block
from omniwave_amd import _native
from omniwave_amd.backward import bigemm_backward

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda", 0)
G = 16
FLAGS = _native.OW_FUSE_NORM | _native.OW_FUSE_RESIDUAL
EPS = 1e-6


def rel(a, b):
    return ((a.double().cpu() - b).norm() / b.norm()).item()


def reference(grad, x, p, plan, d, scale):
    """The block of ``plan`` in float64 and its gradients."""
    leaves = {k: v.double().requires_grad_(True) for k, v in p.items()}
    x64 = x.double().requires_grad_(True)
    b, h, w, c = x.shape
    flat = x64.reshape(b, h * w, c)
    normed = flat * torch.rsqrt(flat.square().mean(dim=-1, keepdim=True) + EPS) * leaves["norm_weight"]
    tok, chan = torch.as_tensor(plan.token_indices).long(), torch.as_tensor(plan.channel_indices).long()
    tok, chan = tok.reshape(-1), chan.reshape(-1)
    tv, cv = (tok >= 0) & (tok < h * w), (chan >= 0) & (chan < c)
    t = normed[:, tok.clamp(0, h * w - 1)][:, :, chan.clamp(0, c - 1)] * tv[:, None] * cv[None, :]
    t = t.reshape(b, -1, G, chan.numel() // d, d).permute(0, 1, 3, 2, 4)
    u, v = leaves["a_u"] @ t @ leaves["b_u"], leaves["a_v"] @ t @ leaves["b_v"]
    o = leaves["a_o"] @ (torch.nn.functional.silu(u) * v @ leaves["b_o"])
    o = o.permute(0, 1, 3, 2, 4).reshape(b, -1, chan.numel())
    rows = torch.zeros(b, h * w, chan.numel(), dtype=torch.float64).index_copy(1, tok[tv], o[:, tv])
    delta = torch.zeros(b, h * w, c, dtype=torch.float64).index_copy(2, chan[cv], rows[:, :, cv]) * leaves["gamma"]
    if scale is not None:
        delta = delta * scale.double().view(b, 1, 1)
    out = (flat + delta).reshape(x.shape)
    names = ("norm_weight", "gamma", "a_u", "a_v", "a_o", "b_u", "b_v", "b_o")
    return torch.autograd.grad(out, (x64, *(leaves[k] for k in names)), grad.double())


@pytest.mark.parametrize("b,h,w,c,d,rd,route,level,drop", [
    (1, 4, 4, 64, 64, 128, "local", 0, False),     # one tile
    (3, 4, 4, 128, 64, 256, "radix", 1, True),     # an odd number of tiles, strided groups
    (2, 7, 7, 200, 128, 256, "shifted", 0, False), # pad slots, a cut-off group
    (1, 9, 13, 96, 64, 128, "radix", 2, False),
    (5, 14, 14, 256, 128, 128, "local", 0, False),
    (9, 14, 14, 512, 128, 256, "radix", 1, True),  # several ranges of slots
    (7, 28, 28, 256, 64, 128, "shifted", 0, False),
])
def test_fp32_backward_against_float64(b, h, w, c, d, rd, route, level, drop) -> None:
    print(f"\n[gpu-case] fp32 backward b={b} {h}x{w}x{c} d={d} rd={rd} {route}{level}", file=sys.stderr, flush=True)
    gen = torch.Generator().manual_seed(11)
    plan = omniwave_amd.build_route_plan(h, w, c, G, d, route, level)
    q_c = -(-c // d)
    normal = lambda *s, fan: torch.randn(*s, generator=gen) / fan ** 0.5
    p = {"norm_weight": torch.rand(c, generator=gen) + 0.5, "gamma": torch.rand(c, generator=gen) + 0.5,
         "a_u": normal(G, G, fan=G), "a_v": normal(G, G, fan=G), "a_o": normal(G, G, fan=G),
         "b_u": normal(q_c, d, rd, fan=d), "b_v": normal(q_c, d, rd, fan=d), "b_o": normal(q_c, rd, d, fan=rd)}
    x, grad = torch.randn(b, h, w, c, generator=gen), torch.randn(b, h, w, c, generator=gen)
    scale = (torch.rand(b, generator=gen) >= 0.3).float() / 0.7 if drop else None
    if drop:
        scale[0] = 1.0 / 0.7
    dev = {k: v.to(DEV) for k, v in p.items()}
    got = bigemm_backward(grad.to(DEV), x.to(DEV), dev["norm_weight"], dev["gamma"], dev["a_u"], dev["a_v"], dev["a_o"],
                          dev["b_u"], dev["b_v"], dev["b_o"], plan, FLAGS, EPS, scale.to(DEV) if drop else None)
    again = bigemm_backward(grad.to(DEV), x.to(DEV), dev["norm_weight"], dev["gamma"], dev["a_u"], dev["a_v"],
                            dev["a_o"], dev["b_u"], dev["b_v"], dev["b_o"], plan, FLAGS, EPS,
                            scale.to(DEV) if drop else None)
    want = reference(grad, x, p, plan, d, scale)
    for name, a, s, e in zip(("x", "norm_weight", "gamma", "a_u", "a_v", "a_o", "b_u", "b_v", "b_o"), got, again, want):
        assert torch.equal(a, s), name  # fixed summation order
        # a chain of at most 256 + 256 fp32 additions per product and six products deep, at random
        # signs: sqrt(512) half-ulps is 1.3e-6; cancellation in the gate's derivative within that
        assert rel(a, e) <= 2.0 ** -24 * 512 ** 0.5, name


def _block(h, c, d, route, level):
    torch.manual_seed(3)
    block = omniwave_amd.block.OmniWeaveBlock(h, h, c, d, route, level).to(DEV)
    with torch.no_grad():
        block.gamma.fill_(1.0)
    return block


def test_empty_batch_has_zero_gradients() -> None:
    block = _block(4, 64, 64, "local", 0)
    x = torch.empty(0, 4, 4, 64, device=DEV, requires_grad=True)
    grads = torch.autograd.grad(block(x), (x, *block.parameters()), torch.empty_like(x))
    assert grads[0].shape == x.shape and all(not g.any() for g in grads[1:])


def test_captured_step_replays_like_the_eager_one() -> None:
    block = _block(7, 256, 128, "radix", 1)
    x = torch.randn(9, 7, 7, 256, device=DEV).requires_grad_(True)
    dy = torch.randn_like(x)
    step = lambda: torch.autograd.grad(block(x), (x, *block.parameters()), dy)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        step()
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        held = step()
    for seed in range(3):
        with torch.no_grad():
            x.copy_(torch.randn(x.shape, generator=torch.Generator().manual_seed(seed)))
        want = [g.clone() for g in step()]
        graph.replay()
        torch.cuda.synchronize()
        assert all(torch.equal(a, b) for a, b in zip(held, want))
