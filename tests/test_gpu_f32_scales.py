"""fp32 RMSNorm row scales (``-m gpu``) against float64: ``ow_rms_scale`` at the edges of its 16-lane
and single-float forms, and the block whose kernel forms them itself (few token pairs) against the
same images in a batch that takes the separate pass."""

from __future__ import annotations

import sys

import pytest
import torch

import omniwave_amd
from omniwave_amd import _native
from omniwave_amd.block import OmniWeaveBlock

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda", 0)


@pytest.mark.parametrize("rows,c,off", [(1, 4, 0), (17, 64, 0), (33, 68, 0), (16, 1024, 0), (5, 96, 1), (9, 70, 0)])
def test_rms_scale_f32(rows, c, off) -> None:
    print(f"\n[gpu-case] f32 row scales rows={rows} c={c} off={off}", file=sys.stderr, flush=True)
    gen = torch.Generator().manual_seed(8)
    x = torch.randn(rows * c + off, generator=gen)
    xd, got = x.to(DEV)[off:], torch.empty(rows, device=DEV)
    _native.check(_native.lib().ow_rms_scale(xd.data_ptr(), got.data_ptr(), rows, c, 1e-6, _native.OW_DTYPE_F32,
                                             torch.cuda.current_stream(DEV).cuda_stream), "ow_rms_scale")
    want = torch.rsqrt(x[off:].double().view(rows, c).square().mean(dim=1) + 1e-6)
    # a sum of positive terms: at most c / 16 + 8 roundings deep, halved by the root, then its own
    assert ((got.double().cpu() - want).abs() / want).max() <= 2.0 ** -24 * (c / 32 + 8)


@pytest.mark.parametrize("h,c,d,off", [(14, 512, 128, 0), (9, 300, 128, 0), (5, 70, 64, 1), (7, 96, 64, 0)])
def test_few_pairs_form_their_own_scales(h, c, d, off) -> None:
    print(f"\n[gpu-case] f32 inline scales {h}x{h}x{c} off={off}", file=sys.stderr, flush=True)
    torch.manual_seed(9)
    block = OmniWeaveBlock(h, h, c, d, "shifted", 0).to(DEV).eval()
    with torch.no_grad():
        block.gamma.fill_(1.0)
    many = 1 + 2 * torch.cuda.get_device_properties(DEV).multi_processor_count
    x = (torch.randn(many * h * h * c + off, device=DEV) * 3)[off:].view(many, h, h, c)
    with torch.inference_mode():
        whole = block(x)
        few = torch.cat([block(x[:1]), block(x[1:2])])
    # the delta's products in another order and a scale one rounding apart (see the bounds of the
    # three-part kernel: sqrt(4 * 96) half-ulps of its norm)
    delta = (whole[:2] - x[:2]).double()
    slack = (x[:2].double().norm() * 2.0 ** -24 / delta.norm()).item()
    assert ((few - whole[:2]).double().norm() / delta.norm()).item() <= 1.2e-6 + 2 * slack
