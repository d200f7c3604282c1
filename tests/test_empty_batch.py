"""The backward of an empty batch: dx of its shape and zero parameter gradients, for every dtype and
tile; on the CPU (no kernel is needed) and through autograd on the GPU (``-m gpu``)."""

from __future__ import annotations

import ctypes
import sys

import pytest
import torch

import omniwave_amd
from omniwave_amd import _native
from omniwave_amd.backward import bigemm_backward

DTYPES = [torch.bfloat16, torch.float16, torch.float32]
SHAPES = [(4, 64, 64), (7, 128, 64), (14, 256, 128)]  # H = W, C, d: 1, 4 and 13 token groups


@pytest.mark.parametrize("norm", [True, False])
@pytest.mark.parametrize("dtype", DTYPES, ids=str)
@pytest.mark.parametrize("h,c,d", SHAPES)
def test_backward_of_nothing(h, c, d, dtype, norm) -> None:
    plan = omniwave_amd.build_route_plan(h, h, c, 16, d, "local", 0)
    q_c, rd = c // d, 2 * d
    ones = lambda *s: torch.ones(*s, dtype=dtype)
    x = ones(0, h, h, c)
    params = (ones(c) if norm else None, ones(c), ones(16, 16), ones(16, 16), ones(16, 16), ones(q_c, d, rd),
              ones(q_c, d, rd), ones(q_c, rd, d))
    flags = _native.OW_FUSE_NORM | _native.OW_FUSE_RESIDUAL if norm else 0
    dx, *grads = bigemm_backward(x, x, *params, plan, flags, 1e-6)
    assert dx.shape == x.shape and dx.dtype == dtype
    for g, p in zip(grads, params):
        assert (g is None) == (p is None)
        assert p is None or (g.shape == p.shape and g.dtype == p.dtype and not g.any())


def test_the_single_call_backward_takes_no_empty_batch() -> None:
    lib = _native.lib()
    one, bf16 = ctypes.c_void_p(256), _native.OW_DTYPE_BF16
    small, dts = (ctypes.c_void_p * 5)(*[256] * 5), (ctypes.c_int32 * 5)(*[bf16] * 5)
    for c, d in ((128, 64), (512, 128)):
        plan = _native.make_plan(14, 14, c, 16, d, "local", 0)
        assert lib.ow_bwd_block_workspace(ctypes.byref(plan), 0, 2 * d, bf16, _native.OW_FUSE_NORM, 0, 1) == 0
        rc = lib.ow_bwd_block(one, one, small, dts, one, one, one, bf16, one, None, one, one, ctypes.byref(plan), 0, 2 * d,
                              bf16, _native.OW_FUSE_NORM, 1e-6, one, one, None, 0, one, 1 << 30, None)
        assert rc == 2 and b"single-call" in lib.ow_last_error()


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", DTYPES, ids=str)
@pytest.mark.parametrize("h,c,d", SHAPES)
def test_empty_batch_through_a_block(h, c, d, dtype) -> None:
    print(f"\n[gpu-case] empty batch {h}x{h}x{c} d={d} {dtype}", file=sys.stderr, flush=True)
    dev = torch.device("cuda", 0)
    block = omniwave_amd.block.OmniWeaveBlock(h, h, c, d, "local", 0).to(dev, dtype)
    x = torch.empty(0, h, h, c, device=dev, dtype=dtype, requires_grad=True)
    grads = torch.autograd.grad(block(x), (x, *block.parameters()), torch.empty_like(x))
    assert grads[0].shape == x.shape and all(not g.any() for g in grads[1:])
