"""fp32 backward building blocks on the GPU (``-m gpu``) against float64: the per-tile outer
product, the token mixing and the RMSNorm backward at the edges of their paths."""

from __future__ import annotations

import sys

import pytest
import torch

from omniwave_amd import _native

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda", 0)
F32 = _native.OW_DTYPE_F32


def rel(a, b):
    return ((a.double().cpu() - b).norm() / b.norm()).item()


def stream():
    return torch.cuda.current_stream(DEV).cuda_stream


# (tiles, d, waves, element offset): one tile, an odd number over the waves, more waves than tiles,
# a width with no compile-time form, rows that are not 16-byte aligned.
@pytest.mark.parametrize("tiles,d,waves,off", [(1, 64, 4, 0), (37, 64, 8, 0), (5, 128, 16, 0), (33, 32, 4, 0),
                                               (9, 128, 4, 1)])
def test_tile_outer_and_mix_f32(tiles, d, waves, off) -> None:
    print(f"\n[gpu-case] f32 tile parts tiles={tiles} d={d} waves={waves} off={off}", file=sys.stderr, flush=True)
    gen = torch.Generator().manual_seed(5)
    n = tiles * 16 * d
    buf = [torch.randn(n + off, generator=gen) for _ in range(2)]
    m = [torch.randn(16, 16, generator=gen) for _ in range(2)]
    dev = [b.to(DEV)[off:] for b in buf]
    md = [t.to(DEV) for t in m]
    t64 = [b[off:].double().view(tiles, 16, d) for b in buf]
    lib = _native.lib()
    part = torch.empty(16, 16, waves, device=DEV)
    _native.check(lib.ow_tile_outer(dev[0].data_ptr(), dev[1].data_ptr(), part.data_ptr(), waves, tiles, d, F32,
                                    stream()), "ow_tile_outer")
    want = torch.einsum("tic,tjc->ij", t64[0], t64[1])
    # a serial fp32 chain of tiles * d / waves terms: 2^-24 each, at random
    assert rel(part.sum(dim=2), want) <= 2.0 ** -24 * (tiles * d) ** 0.5 * 4
    if d not in (64, 128):
        return
    out = torch.empty(n, device=DEV)
    for two in (False, True):
        _native.check(lib.ow_tile_mix(dev[0].data_ptr(), md[0].data_ptr(), dev[1].data_ptr() if two else None,
                                      md[1].data_ptr() if two else None, out.data_ptr(), tiles, d, F32, stream()),
                      "ow_tile_mix")
        want = m[0].double() @ t64[0] + (m[1].double() @ t64[1] if two else 0)
        assert rel(out.view(tiles, 16, d), want) <= 2.0 ** -24 * 32 ** 0.5


@pytest.mark.parametrize("rows,c,off", [(1, 4, 0), (7, 96, 0), (9, 128, 0), (5, 132, 0), (3, 1024, 0), (6, 70, 0),
                                        (5, 256, 1)])
@pytest.mark.parametrize("norm,residual", [(True, True), (True, False), (False, True)])
def test_rmsnorm_bwd_f32(rows, c, off, norm, residual) -> None:
    print(f"\n[gpu-case] f32 rmsnorm backward rows={rows} c={c} off={off}", file=sys.stderr, flush=True)
    gen = torch.Generator().manual_seed(6)
    x, g, dy = (torch.randn(rows * c + off, generator=gen) for _ in range(3))
    r = torch.rand(rows, generator=gen) + 0.5
    xd, gd, dyd = (t.to(DEV)[off:] for t in (x, g, dy))
    dx = torch.empty(rows * c + off, device=DEV)[off:]
    _native.check(_native.lib().ow_bwd_rmsnorm(xd.data_ptr(), gd.data_ptr(), r.to(DEV).data_ptr() if norm else None,
                                               dyd.data_ptr(), dx.data_ptr(), rows, c, int(residual), F32, stream()),
                  "ow_bwd_rmsnorm")
    x64, g64, dy64 = (t[off:].double().view(rows, c) for t in (x, g, dy))
    r64 = r.double().view(rows, 1) if norm else torch.ones(rows, 1, dtype=torch.float64)
    want = r64 * g64
    if norm:
        want = want - x64 * r64 ** 3 / c * (g64 * x64).sum(dim=1, keepdim=True)
    if residual:
        want = want + dy64
    assert rel(dx.view(rows, c), want) <= 2.0 ** -24 * c ** 0.5 + 4 * 2.0 ** -24
