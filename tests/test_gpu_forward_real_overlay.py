"""The real row format's forward (IQ4_NL, 16 heads of 160) under an overlay,
its own kernel, against the gather of the same rows (eg_gather's general
kernel) added to the residual in fp32 and rounded by torch: bit for bit, for
every replacement format, through the search and the bitmap, and with
overlay indices outside their store (NaN, no read)."""
from __future__ import annotations

import sys

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_pos", [1, 5, 333])
@pytest.mark.parametrize("fmt", ["f32", "q8_0", "bf16", "mxfp8", "iq4_nl"])
def test_real_forward_under_an_overlay(cuda, n_pos, fmt):
    from engraft_ngram_amd import synthetic as S
    from engraft_ngram_amd import table as T
    from engraft_ngram_amd.overlay import DeviceOverlay
    print(f"[gpu-test] iq4_nl forward under a {fmt} overlay, {n_pos} positions", file=sys.stderr, flush=True)
    heads, per, dim = 16, 300, 160
    hp = S.hash_params(heads * per, seed=7)

    g = torch.Generator(device=cuda).manual_seed(n_pos)

    def store(f, n):
        s = T.RowStore.empty(f, n, dim, cuda, row_stride=T.RowStore.padded_stride(f, dim))
        if f in ("f32", "bf16"):
            s.payload.copy_(torch.randn((n, dim), generator=g, device=cuda) * 0.02)
            return s
        s.payload.random_(0, 120, generator=g)  # any byte is a value, but e4m3's NaN
        scale = (torch.rand((n, dim // 32), generator=g, device=cuda) * 1e-3).to(torch.float16)
        if f == "q8_0":
            s.scales.copy_(scale)
        elif f == "mxfp8":
            s.scales.random_(110, 120, generator=g)
        else:
            s.payload[:, :90].view(n, 5, 18)[:, :, :2] = scale.view(torch.uint8).view(n, 5, 2)
        return s
    tab = T.DeviceTable(store("iq4_nl", heads * per), **hp)
    tok = torch.randint(0, 40, (n_pos,), generator=g, device=cuda)
    res = torch.randn((n_pos, heads * dim), generator=g, device=cuda).to(torch.bfloat16)
    rows = tab.rows(tok)
    read = torch.unique(rows)
    for ids in (read[::2], read[:1], torch.arange(0, heads * per, 3, device=cuda)):
        ids = ids.to(torch.int32).contiguous()
        n = ids.numel()
        index = torch.randperm(n, generator=g, device=cuda).to(torch.int32)
        index[0] = n + 5  # outside the store
        for idx, bits in ((None, False), (index, False), (None, True)):
            ov = DeviceOverlay(ids, store(fmt, n), idx)
            if bits:
                ov.with_bitmap(tab.n_rows)
            out, got_rows = tab.forward(tok, res, overlay=ov, return_rows=True)
            want = (res.float() + tab.gather(rows, overlay=ov)).to(torch.bfloat16)
            assert torch.equal(got_rows[0], rows)
            a, b = (x.view(torch.int16).cpu().numpy() for x in (out, want))
            nan = torch.isnan(want.float()).cpu().numpy()
            assert np.array_equal(a[~nan], b[~nan]) and bool(torch.isnan(out.float()).cpu()[torch.from_numpy(nan)].all())
