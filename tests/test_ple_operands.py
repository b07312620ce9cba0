"""gemm_h3 and HalfPlanes refuse operands whose shapes the kernels would read
out of range, before any launch."""
from __future__ import annotations

import pytest
import torch

A, B = torch.zeros((4, 32)), torch.zeros((6, 32))


@pytest.mark.parametrize("of", [(A, B), (A[:3], A), (A.bfloat16(),), (A[0],), (), (A, A, A)])
def test_half_planes_refuses(of):
    from engraft_ngram_amd.ple import HalfPlanes
    with pytest.raises(ValueError, match="HalfPlanes"):
        HalfPlanes(of)


class _Planes:
    """Planes of an operand [rows, cols], as HalfPlanes records them."""

    def __init__(self, *shapes):
        self.shapes, self.rows, self.planes = shapes, shapes[0][0], A


@pytest.mark.parametrize("a,b,b2,planes,planes2", [
    ((A,), (B[:, :31],), None, None, None),                # another k
    ((A, A), (B,), None, None, None),                      # another number of sources
    ((A,), (B,), (A[:, 1:],), None, None),                 # the second group's k
    ((A[0],), (B,), None, None, None),
    ((A,), (B,), None, _Planes((8, 32)), None),            # planes of a larger matrix
    ((A,), (B,), None, _Planes((6, 64)), None),
    ((A,), (B,), (B,), None, _Planes((4, 32))),
    ((A,), (B,), None, None, _Planes((6, 32))),            # planes of a group that is not there
    ((A, A[:3]), (B, B), None, None, None),                # sources of different rows
    ((A,), (B.to("meta"),), None, None, None),             # another device
])
def test_gemm_h3_refuses(a, b, b2, planes, planes2):
    from engraft_ngram_amd.ple import gemm_h3
    with pytest.raises(ValueError):
        gemm_h3(a, b, b2, planes_b=planes, planes_b2=planes2)
