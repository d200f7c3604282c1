"""Ragged channel counts and unaligned rows in the 16-bit forward (``-m gpu``).

Contiguous groups whose last one is cut off by the row's end: every remainder of a 16-byte vector,
rows at every alignment, the sizes at which the resident kernel takes over, against float64.
"""

from __future__ import annotations

import sys

import pytest
import torch

import omniwave_amd
from omniwave_amd import _native
from omniwave_amd.backbone import space_to_depth_nhwc
from omniwave_amd.hip import bigemm_block_hip, bigemm_block_s2d_hip, bigemm_delta_hip
from oracle.bigemm import bigemm_delta_reference, block_reference, rel_l2
from oracle.routing import build_route_plan as oracle_plan

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda", 0)
# Five roundings to 16 bits in a row (the normed input's scale, P, U and V's gate, W, delta), each
# of a random error below eps / sqrt(3), and the weights': together below 3 eps of the norm.
TOL = {torch.bfloat16: 3 * 2.0 ** -8, torch.float16: 3 * 2.0 ** -11}
CASES = [  # batch, H, W, C, d, rd, route
    (2, 5, 7, 1, 64, 128, "local"),
    (3, 3, 5, 7, 64, 256, "radix"),
    (2, 9, 9, 65, 64, 128, "shifted"),
    (2, 9, 9, 72, 64, 128, "local"),       # C % 8 == 0: 65 .. 127 with two groups
    (70, 7, 9, 96, 64, 128, "shifted"),
    (1, 4, 4, 120, 64, 128, "radix"),
    (3, 5, 5, 127, 64, 128, "local"),
    (2, 8, 6, 130, 64, 128, "local"),
    (2, 8, 6, 160, 64, 128, "local"),      # three groups
    (3, 6, 7, 200, 64, 128, "shifted"),    # four groups, aligned
    (33, 8, 8, 248, 64, 128, "radix"),
    (2, 6, 6, 250, 64, 128, "local"),
    (2, 6, 6, 72, 64, 256, "local"),
    (2, 5, 6, 131, 128, 128, "shifted"),
    (2, 7, 7, 136, 128, 256, "local"),
    (9, 7, 7, 300, 128, 256, "radix"),
    (1, 3, 3, 511, 128, 256, "local"),
]


def _inputs(b, h, w, c, d, rd, dtype):
    gen = torch.Generator().manual_seed(11)
    q_c = -(-c // d)
    x = torch.randn(b, h, w, c, generator=gen).to(dtype)
    params = dict(
        a_u=torch.randn(16, 16, generator=gen) / 4, a_v=torch.randn(16, 16, generator=gen) / 4,
        a_o=torch.randn(16, 16, generator=gen) / 4,
        b_u=torch.randn(q_c, d, rd, generator=gen) / d ** 0.5, b_v=torch.randn(q_c, d, rd, generator=gen) / d ** 0.5,
        b_o=torch.randn(q_c, rd, d, generator=gen) / rd ** 0.5, gamma=torch.rand(c, generator=gen) + 0.5,
    )
    nw = torch.rand(c, generator=gen) + 0.5
    scale = (torch.arange(b) % 3 != 1).to(dtype) * 1.25
    return x, params, nw, scale


def _at(x: torch.Tensor, offset: int) -> torch.Tensor:
    """x on the device, ``offset`` elements past an allocation's start, the rest of it NaN."""
    buf = torch.full((x.numel() + 64,), float("nan"), dtype=x.dtype, device=DEV)
    buf[offset:offset + x.numel()] = x.to(DEV).flatten()
    return buf[offset:offset + x.numel()].view(x.shape)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
@pytest.mark.parametrize("b,h,w,c,d,rd,route", CASES,
                         ids=[f"{b}x{h}x{w}x{c}-d{d}-rd{rd}-{r}" for b, h, w, c, d, rd, r in CASES])
def test_ragged_forward_matches_float64(b, h, w, c, d, rd, route, dtype) -> None:
    print(f"\n[gpu-case] ragged {b}x{h}x{w}x{c} d={d} rd={rd} {route} {dtype}", file=sys.stderr, flush=True)
    x, params, nw, scale = _inputs(b, h, w, c, d, rd, dtype)
    plan = omniwave_amd.build_route_plan(h, w, c, 16, d, route, 0)
    dp, dnw = {k: v.to(DEV) for k, v in params.items()}, nw.to(DEV)
    oplan = oracle_plan(h, w, c, 16, d, route, 0)
    p64 = {k: v.double() for k, v in params.items()}
    x64 = x.double()
    delta_want = bigemm_delta_reference(x=x64, plan=oplan, **p64)
    branch = block_reference(x64, oplan, {**p64, "norm_weight": nw.double()}, residual=False)
    for offset in (0, 8, 1, 2):
        xd = _at(x, offset)
        delta = bigemm_delta_hip(x=xd, plan=plan, **dp).cpu()
        assert rel_l2(delta, delta_want) <= TOL[dtype], offset
        out = bigemm_block_hip(xd, dnw, plan, **dp).cpu().double()
        dropped = bigemm_block_hip(xd, dnw, plan, **dp, drop_scale=scale.to(DEV)).cpu()
        for got, factor in ((out, None), (dropped.double(), scale.double())):
            want = branch if factor is None else branch * factor.reshape(b, 1, 1, 1)
            # the sum's own rounding: half an ulp of |out| per value
            slack = (got.norm() * TOL[dtype] / 6 / want.norm()).item()
            assert rel_l2(got - x64, want) <= TOL[dtype] + slack, offset
        assert torch.equal(dropped[scale == 0], x[scale == 0])
        if h % 2 == 0 and w % 2 == 0:
            moved = bigemm_block_s2d_hip(xd, dnw, plan, **dp, factor=2).cpu().double()
            assert torch.equal(moved, space_to_depth_nhwc(out, 2)), offset


@pytest.mark.parametrize("offset", [0, 1])
@pytest.mark.parametrize("c", [1, 8, 63, 96, 200, 511, 1000])
def test_row_scales_of_any_width(c, offset) -> None:
    """``ow_rms_scale`` at widths and alignments with no kernel of their own.  The mean square and
    its sum with eps round to bf16 (2^-9 each, halved by the root), then the root does (2^-9)."""
    for rows in (1, 31, 200):
        x = torch.randn(rows, c, generator=torch.Generator().manual_seed(c)).to(torch.bfloat16)
        xd, got = _at(x, offset), torch.full((rows + 1,), -1.0, device=DEV)
        _native.check(_native.lib().ow_rms_scale(xd.data_ptr(), got.data_ptr(), rows, c, 1e-6, _native.OW_DTYPE_BF16,
                                                 torch.cuda.current_stream().cuda_stream), "ow_rms_scale")
        got = got.cpu().double()
        assert got[rows] == -1.0
        want = torch.rsqrt(x.double().square().mean(dim=-1) + 1e-6)
        assert ((got[:rows] - want).abs() <= want * 2.0 ** -7).all()
