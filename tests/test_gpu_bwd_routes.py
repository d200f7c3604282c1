"""Gather and scatter of the backward on the GPU (``-m gpu``): every channel order and both access
paths against indexing with the plan's tables, bit for bit."""

from __future__ import annotations

import ctypes
import sys

import pytest
import torch

import omniwave_amd
from omniwave_amd import _native
from omniwave_amd.routing import device_tables, native_plan

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda", 0)
CODE = {torch.bfloat16: _native.OW_DTYPE_BF16, torch.float16: _native.OW_DTYPE_F16}
CASES = [  # batch, H, W, C, d, level, element offset of x / dy / g
    (2, 5, 7, 128, 64, 1, 0),    # two groups, pad tokens
    (1, 3, 3, 256, 64, 2, 0),    # four groups, rotated by two, one group of tokens
    (3, 4, 4, 512, 128, 3, 0),
    (2, 7, 7, 1024, 128, 1, 0),  # eight groups: lane pairs
    (1, 2, 2, 512, 64, 5, 0),    # eight groups of 64
    (2, 3, 5, 512, 128, 1, 1),   # rows that are not 16-byte aligned: element access
    (2, 3, 5, 96, 64, 1, 0),     # ragged groups: element access
    (2, 5, 5, 192, 64, 2, 0),    # three groups: element access
    (2, 4, 6, 256, 128, 0, 0),   # contiguous groups
]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "f16"])
@pytest.mark.parametrize("b,h,w,c,d,level,off", CASES)
def test_gather_scatter_match_indexing(b, h, w, c, d, level, off, dtype) -> None:
    print(f"\n[gpu-case] gather/scatter {b}x{h}x{w}x{c} d={d} level={level} off={off} {dtype}", file=sys.stderr,
          flush=True)
    gen = torch.Generator().manual_seed(4)
    plan = omniwave_amd.build_route_plan(h, w, c, 16, d, "radix", level)
    n, q_s, q_c = h * w, plan.token_indices.shape[0], plan.channel_indices.shape[0]
    slots = b * q_s * 16
    x, dy = (torch.randn(b * n * c + off, generator=gen).to(dtype) for _ in range(2))
    r = torch.rand(b * n, generator=gen) + 0.5
    tok, ch = device_tables(plan, DEV)
    xt, dyt = (torch.full((q_c, slots, d), 7.0, dtype=dtype, device=DEV) for _ in range(2))
    lib, oplan = _native.lib(), native_plan(plan)
    stream = torch.cuda.current_stream(DEV).cuda_stream
    xd, dyd = x.to(DEV)[off:], dy.to(DEV)[off:]
    _native.check(lib.ow_bwd_gather(xd.data_ptr(), dyd.data_ptr(), r.to(DEV).data_ptr(), tok.data_ptr(), ch.data_ptr(),
                                    ctypes.byref(oplan), b, CODE[dtype], xt.data_ptr(), dyt.data_ptr(), stream),
                  "ow_bwd_gather")

    def tiles(t):  # [b, n, c] -> [q_c, slots, d], pads 0
        t = torch.nn.functional.pad(t, (0, 1, 0, 1))
        t = t[:, plan.token_indices.reshape(-1)][:, :, plan.channel_indices.reshape(-1)]
        return t.reshape(b * q_s * 16, q_c, d).transpose(0, 1)

    scaled = (x[off:].float().view(b, n, c) * r.view(b, n, 1)).to(dtype)
    assert torch.equal(xt.cpu(), tiles(scaled))
    assert torch.equal(dyt.cpu(), tiles(dy[off:].view(b, n, c)))

    g = torch.full((b * n * c + off,), 7.0, dtype=dtype, device=DEV)
    _native.check(lib.ow_bwd_scatter(dyt.data_ptr(), tok.data_ptr(), ch.data_ptr(), ctypes.byref(oplan), b, CODE[dtype],
                                     g[off:].data_ptr(), stream), "ow_bwd_scatter")
    assert torch.equal(g.cpu()[off:], dy[off:])  # the routes are permutations
    assert bool((g.cpu()[:off] == 7.0).all())
