"""fp32 forward on the bf16 matrix cores (``-m gpu``): the three-part kernel against float64.

Each of the chain's four products adds at most 96 matrix-core results per value in fp32 (six for
each of 16 K steps), every addition rounding by 2^-24 at random, so the error stays near
sqrt(4 * 96) * 2^-24 = 1.2e-6 of the result's norm.
"""

from __future__ import annotations

import sys

import pytest
import torch

import omniwave_amd
from omniwave_amd.hip import bigemm_block_hip, bigemm_delta_hip
from oracle.bigemm import bigemm_delta_reference, block_reference, rel_l2
from oracle.routing import build_route_plan as oracle_plan

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda", 0)
TOL = 1.2e-6
CASES = [  # batch, H, W, C, d, rd, route, level: how the waves of a workgroup split the work
    (1, 3, 5, 128, 128, 256, "local", 0),       # one token group: half a pair, split in four
    (3, 7, 9, 300, 128, 256, "radix", 1),       # ragged channels in a strided order, pad tokens
    (5, 2, 2, 200, 128, 128, "radix", 2),       # five images in one workgroup, a chunk per wave
    (1, 9, 9, 96, 64, 128, "shifted", 0),       # d = 64 split in four: two waves store
    (2, 5, 7, 70, 64, 256, "local", 0),         # unaligned rows
    (20, 14, 14, 512, 128, 256, "radix", 1),    # 520 units: whole pairs per wave
    (16, 14, 14, 512, 128, 256, "shifted", 0),  # 416 units: pairs split in two
    (40, 12, 12, 256, 64, 128, "radix", 1),     # 720 units, d = 64
    (41, 7, 7, 1024, 128, 128, "local", 0),     # odd number of token groups
]


@pytest.mark.parametrize("b,h,w,c,d,rd,route,level", CASES, ids=[f"{b}x{h}x{w}x{c}-d{d}-rd{rd}-{r}{l}"
                                                               for b, h, w, c, d, rd, r, l in CASES])
def test_x3_forward_matches_float64(b, h, w, c, d, rd, route, level) -> None:
    print(f"\n[gpu-case] x3 {b}x{h}x{w}x{c} d={d} rd={rd} {route}{level}", file=sys.stderr, flush=True)
    gen = torch.Generator().manual_seed(7)
    plan = omniwave_amd.build_route_plan(h, w, c, 16, d, route, level)
    q_c = plan.channel_indices.shape[0]
    x = torch.randn(b, h, w, c, generator=gen)
    params = dict(
        a_u=torch.randn(16, 16, generator=gen) / 4, a_v=torch.randn(16, 16, generator=gen) / 4,
        a_o=torch.randn(16, 16, generator=gen) / 4,
        b_u=torch.randn(q_c, d, rd, generator=gen) / d ** 0.5, b_v=torch.randn(q_c, d, rd, generator=gen) / d ** 0.5,
        b_o=torch.randn(q_c, rd, d, generator=gen) / rd ** 0.5, gamma=torch.rand(c, generator=gen) + 0.5,
    )
    nw = torch.rand(c, generator=gen) + 0.5
    scale = (torch.rand(b, generator=gen) < 0.6).float() / 0.6
    dp = {k: v.to(DEV) for k, v in params.items()}
    delta = bigemm_delta_hip(x=x.to(DEV), plan=plan, **dp).cpu()
    out = bigemm_block_hip(x.to(DEV), nw.to(DEV), plan, **dp, drop_scale=scale.to(DEV)).cpu()
    oplan = oracle_plan(h, w, c, 16, d, route, level)
    p64 = {k: v.double() for k, v in params.items()}
    assert rel_l2(delta, bigemm_delta_reference(x=x.double(), plan=oplan, **p64)) <= TOL
    branch = block_reference(x.double(), oplan, {**p64, "norm_weight": nw.double()}, residual=False)
    want = branch * scale.double().reshape(b, 1, 1, 1)
    got = out.double() - x.double()
    # the sum rounds to fp32: at most 2^-24 of |out| per value
    slack = (out.double().norm() * 2.0 ** -24 / want.norm()).item() if want.norm() > 0 else 0.0
    assert rel_l2(got, want) <= TOL + slack
    assert torch.equal(out[scale == 0], x[scale == 0])  # a dropped image passes through untouched
