"""eg_ple_conv_gated (the convolution over normed rows it computes from the
gate's factors) against eg_ple_gate + eg_ple_conv with those rows in memory:
output, pre-activation and new history bit for bit, at the edges of its
32-position runs, its 256-channel blocks and the history's 9 rows."""
from __future__ import annotations

import sys

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("t,h0,hc,n", [(1, 0, 4, 2560), (1, 9, 4, 2560), (8, 1, 1, 256), (9, 0, 3, 512),
                                       (31, 4, 4, 256), (32, 9, 2, 768), (33, 12, 4, 512), (100, 9, 4, 2560)])
def test_conv_gated_is_the_convolution_of_the_normed_rows(cuda, t, h0, hc, n):
    from engraft_ngram_amd import _lib
    print(f"[gpu-test] conv_gated t={t} h0={h0} hc={hc} n={n}", file=sys.stderr, flush=True)
    g = torch.Generator(device=cuda).manual_seed(t + h0 + n)
    key, hidden = (torch.randn((t, hc * n), generator=g, device=cuda) for _ in range(2))
    value = torch.randn((t, n), generator=g, device=cuda)
    hist = torch.randn((h0, hc * n), generator=g, device=cuda)
    nk, nq, nc = (1 + 0.1 * torch.randn(hc * n, generator=g, device=cuda) for _ in range(3))
    conv = torch.randn((hc * n, 4), generator=g, device=cuda)
    st, p = _lib.stream_ptr(cuda), _lib.ptr
    res = []
    for gated in (False, True):
        full = torch.cat([hist, torch.full((t, hc * n), 7.0, device=cuda)])
        s, gate = (torch.empty((t, hc), device=cuda) for _ in range(2))
        rstd = torch.empty((t, hc, 3), device=cuda)
        out, pre = (torch.empty((t, hc * n), device=cuda) for _ in range(2))
        _lib.call("eg_ple_gate", p(key), p(value), p(hidden), p(nk), p(nq), p(nc), t, hc, n, 1e-6,
                  None if gated else p(full[h0:]), p(s), p(gate), p(rstd), st)
        if gated:
            new = torch.empty((min(9, h0 + t), hc * n), device=cuda)
            _lib.call("eg_ple_conv_gated", p(hist), h0, t, hc, n, p(value), p(gate), p(rstd), p(nc), p(conv), 4, 3,
                      p(hidden), p(out), p(pre), p(new), st)
        else:
            _lib.call("eg_ple_conv", p(full), h0, t, hc, n, p(conv), 4, 3, 0, p(hidden), p(value), p(gate), p(out),
                      p(pre), st)
            new = full[-9:]
        torch.cuda.synchronize()
        res.append((out, pre, new, s, gate, rstd))
    for a, b in zip(*res):
        assert torch.equal(a, b)
