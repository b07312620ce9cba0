"""Which of the block's kernels a call takes, at the limits of what they are built for."""
from __future__ import annotations

import ctypes

import pytest


@pytest.mark.parametrize("rows,grads,exp", [(10, True, True), (65535 * 63, True, True), (65535 * 63 + 1, True, False),
                                            (65535 * 63 + 1, False, True), (65535 * 64, True, False)])
def test_gated_convolution_leaves_out_what_the_weight_sums_refuse(rows, grads, exp):
    """Past eg_ple_conv_backward_sums' rows a call whose norm or convolution weights need
    gradients keeps its normed rows and takes eg_ple_weight_grads, which has no such limit."""
    from engraft_ngram_amd import _lib, ple
    assert ple._gated_ok(rows, rows - 9, 256, 4, 3, grads) is exp
    # the C entry agrees on where its range ends: a workspace of 0 bytes is refused by its size
    # within the range (EG_ERR_WORKSPACE), by the shape past it (EG_ERR_UNSUPPORTED)
    rc = _lib.load().eg_ple_weight_sums(*[None] * 6, 9, rows - 9, 1, 256, *[None] * 5, ctypes.c_size_t(0), None)
    assert rc == (_lib.EG_ERR_WORKSPACE if rows <= 65535 * 63 else _lib.EG_ERR_UNSUPPORTED)


@pytest.mark.parametrize("t_len,n,taps,dil", [(0, 256, 4, 3), (5, 320, 4, 3), (5, 256, 3, 3), (5, 256, 4, 2)])
def test_gated_convolution_is_built_for_one_shape(t_len, n, taps, dil):
    from engraft_ngram_amd import ple
    assert not ple._gated_ok(9 + t_len, t_len, n, taps, dil, False)
