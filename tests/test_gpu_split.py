"""Small d = 128, rd = 256 launches (``-m gpu``): the kernel that splits a pair's expanded dimension
over a workgroup's waves against the persistent kernel, bit for bit.

Both round at the same places and add in the same order, so an image's result can't depend on the
batch it came in.  The large batch repeats the images until the persistent kernel takes it.
"""

from __future__ import annotations

import sys

import pytest
import torch

import omniwave_amd
from omniwave_amd import _native
from omniwave_amd.backbone import space_to_depth_nhwc
from omniwave_amd.hip import (_plan_desc, bigemm_block_chain_hip, bigemm_block_hip, bigemm_block_s2d_hip,
                              bigemm_delta_hip)

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda", 0)
CASES = [  # batch, H, W, C, route, level, copies
    (1, 1, 1, 128, "local", 0, 1300),      # one real row of a pair
    (1, 14, 14, 512, "local", 0, 25),      # 13 token groups: the last pair is half pad
    (3, 5, 7, 384, "shifted", 0, 60),      # three groups: scales from the statistics pass
    (2, 7, 7, 1024, "local", 0, 24),
    (3, 3, 5, 256, "radix", 1, 220),       # strided by 2, 4 and 8
    (5, 14, 14, 512, "radix", 2, 6),
    (7, 7, 7, 1024, "radix", 1, 8),
    (2, 8, 6, 1152, "radix", 0, 30),       # nine groups
    (40, 7, 7, 1024, "local", 0, 2),       # 640 workgroups, the most the kernel takes
]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
@pytest.mark.parametrize("b,h,w,c,route,level,copies", CASES,
                         ids=[f"{b}x{h}x{w}x{c}-{r}{l}" for b, h, w, c, r, l, _ in CASES])
def test_small_batches_equal_large_ones(b, h, w, c, route, level, copies, dtype) -> None:
    print(f"\n[gpu-case] split {b}x{h}x{w}x{c} {route}{level} {dtype}", file=sys.stderr, flush=True)
    q_c = c // 128
    pairs = -(-b * -(-h * w // 16) // 2)
    assert pairs * q_c <= 640 < -(-copies * b * -(-h * w // 16) // 2) * q_c
    gen = torch.Generator().manual_seed(5)
    plan = omniwave_amd.build_route_plan(h, w, c, 16, 128, route, level)
    x = torch.randn(b, h, w, c, generator=gen).to(dtype).to(DEV)
    p = {k: torch.randn(*s, generator=gen).to(DEV) * f for k, s, f in (
        ("a_u", (16, 16), 0.25), ("a_v", (16, 16), 0.25), ("a_o", (16, 16), 0.25), ("b_u", (q_c, 128, 256), 0.09),
        ("b_v", (q_c, 128, 256), 0.09), ("b_o", (q_c, 256, 128), 0.06), ("gamma", (c,), 1.0))}
    nw = torch.rand(c, generator=gen).to(DEV) + 0.5
    drop = torch.rand(b, generator=gen).to(dtype).to(DEV)
    big = x.repeat(copies, 1, 1, 1)

    def same(small, large):
        assert torch.isfinite(small).all()
        assert torch.equal(small, large[:small.shape[0]]) and torch.equal(small, large[-small.shape[0]:])

    with torch.no_grad():
        same(bigemm_delta_hip(x=x, plan=plan, **p), bigemm_delta_hip(x=big, plan=plan, **p))
        out = bigemm_block_hip(x, nw, plan, **p)
        same(out, bigemm_block_hip(big, nw, plan, **p))
        same(bigemm_block_hip(x, nw, plan, **p, drop_scale=drop),
             bigemm_block_hip(big, nw, plan, **p, drop_scale=drop.repeat(copies)))
        if h % 2 == 0 and w % 2 == 0:
            assert torch.equal(bigemm_block_s2d_hip(x, nw, plan, **p, factor=2), space_to_depth_nhwc(out, 2))
        y, s = bigemm_block_chain_hip(x, None, nw, plan, **p)
        big_y, big_s = bigemm_block_chain_hip(big, None, nw, plan, **p)
        same(y, big_y)
        same(s, big_s)
        for got, want in zip(bigemm_block_chain_hip(y, s, nw, plan, **p),
                             bigemm_block_chain_hip(big_y, big_s, nw, plan, **p)):
            same(got, want)

    def with_scales(t):
        order = ("gamma", "a_u", "a_v", "a_o", "b_u", "b_v", "b_o")
        with torch.no_grad():
            return torch.ops.omniwave_amd.bigemm_fwd(t, nw, *(p[k] for k in order), _plan_desc(plan),
                                                     _native.OW_FUSE_NORM, 1e-6, None, True)

    for got, want in zip(with_scales(x), with_scales(big)):
        same(got, want)
