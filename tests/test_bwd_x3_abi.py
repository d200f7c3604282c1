"""C entry points of the three-part fp32 backward without a GPU: sizes, and what they refuse."""

from __future__ import annotations

import ctypes

import pytest

from omniwave_amd import _native

lib = _native.lib()
F32 = _native.OW_DTYPE_F32


@pytest.mark.parametrize("d,rd", [(64, 128), (64, 256), (128, 128), (128, 256)])
def test_sizes(d, rd) -> None:
    # both chunk orders of three matrices, six bytes a value
    assert lib.ow_bwd_x3_packed_bytes(3, d, rd) == 3 * 2 * 3 * d * rd * 6
    assert lib.ow_bwd_x3_packed_bytes(0, d, rd) == 0


def test_unsupported_tiles_have_no_packed_size() -> None:
    assert lib.ow_bwd_x3_packed_bytes(1, 32, 128) == 0
    assert lib.ow_bwd_x3_packed_bytes(1, 64, 64) == 0


@pytest.mark.parametrize("n_tok,channels,q_s", [(56 * 56, 128, 196), (4, 1024, 1), (96 * 96, 1024, 576)])
def test_images_of_the_network_fit(n_tok, channels, q_s) -> None:
    assert lib.ow_bwd_x3_fits(n_tok, channels, q_s)


def test_images_past_the_offsets_do_not_fit() -> None:
    # a workgroup's eight token groups lie in at most 8 / q_s + 2 images, below 1 GiB together
    edge = (1 << 30) // (2 * 4 * 64)
    assert lib.ow_bwd_x3_fits(edge - 1, 64, edge // 16)
    assert not lib.ow_bwd_x3_fits(edge, 64, edge // 16)
    assert not lib.ow_bwd_x3_fits(4, 64, 0)


def _channel(**over):
    one = ctypes.c_void_p(4096)
    a = {"ptrs": [one] * 3, "packed_bytes": lib.ow_bwd_x3_packed_bytes(1, 64, 128), "batch": 1, "n_tok": 16,
         "channels": 64, "q_s": 1, "q_c": 1, "d": 64, "rd": 128, "n_partial": 1}
    a.update(over)
    x, dy, packed = a["ptrs"]
    return lib.ow_bwd_channel_x3(x, dy, None, one, one, one, packed, a["packed_bytes"], one, one, one, one, one, one, one,
                                 one, a["batch"], a["n_tok"], a["channels"], a["q_s"], a["q_c"], a["d"], a["rd"], one,
                                 one, a["n_partial"], one, None)


@pytest.mark.parametrize("over", [
    {"d": 32}, {"rd": 64}, {"batch": -1}, {"q_c": 0}, {"q_s": 0}, {"n_tok": 0}, {"packed_bytes": 16},
    {"n_partial": 2}, {"n_tok": 1 << 24}, {"ptrs": [None, ctypes.c_void_p(4096), ctypes.c_void_p(4096)]},
    {"ptrs": [ctypes.c_void_p(4096), ctypes.c_void_p(4096), ctypes.c_void_p(4100)]},
])
def test_refused_before_any_launch(over) -> None:
    assert _channel(**over) != 0


def test_an_empty_batch_launches_nothing() -> None:
    assert _channel(batch=0, n_partial=0) == 0
    assert lib.ow_bwd_channel_x3_partials(0, 1) == 0
    assert lib.ow_bwd_param_reduce_x3_ranges(0, 1) == 0


def test_reduction_refuses_bad_ranges() -> None:
    one = ctypes.c_void_p(4096)
    for ranges, slots in ((0, 32), (3, 32), (1, 24), (1, 0)):
        assert lib.ow_bwd_param_reduce_x3(*[one] * 7, ranges, slots, 1, 64, 128, None) != 0
