"""eg_ple_conv_gated (the convolution over normed rows it computes from the
gate's factors) against eg_ple_gate + eg_ple_conv with those rows in memory:
output, pre-activation and new history bit for bit, at the edges of its
16-position runs, its 256-channel blocks and the history's 9 rows."""
from __future__ import annotations

import sys

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("t,h0,hc,n", [(1, 0, 4, 2560), (1, 9, 4, 2560), (8, 1, 1, 256), (9, 0, 3, 512),
                                       (15, 9, 2, 256), (16, 9, 4, 256), (17, 3, 2, 512), (31, 4, 4, 256), (32, 9, 2, 768), (33, 12, 4, 512), (100, 9, 4, 2560)])
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


@pytest.mark.parametrize("t,h0,hc,n", [(1, 0, 1, 256), (9, 2, 2, 256), (54, 9, 4, 512), (63, 0, 3, 256),
                                       (64, 12, 2, 512), (135, 9, 4, 256)])
@pytest.mark.parametrize("tail", [False, True])
def test_conv_backward_sums_against_the_separate_kernels(cuda, t, h0, hc, n, tail):
    """eg_ple_conv_backward_sums + eg_ple_weight_sums against eg_ple_conv_backward
    without the forward's pre-activation (its general kernel) and
    eg_ple_weight_grads, at the edges of the 63-row chunks and nine-row turns:
    d_full bit for bit, the sums over t positions within t 2^-23 of the sum of
    the terms' magnitudes (two fp32 sums of the same terms)."""
    from engraft_ngram_amd import _lib
    print(f"[gpu-test] conv_backward_sums t={t} h0={h0} hc={hc} n={n} tail={tail}", file=sys.stderr, flush=True)
    g = torch.Generator(device=cuda).manual_seed(t + h0 + n)
    rnd = lambda *s: torch.randn(s, generator=g, device=cuda)
    C = hc * n
    key, hidden, d_out, value, hist, conv = rnd(t, C), rnd(t, C), rnd(t, C), rnd(t, n), rnd(h0, C), rnd(C, 4)
    nk, nq, nc = (1 + 0.1 * rnd(C) for _ in range(3))
    tail_rows = min(9, h0 + t) if tail else 0
    d_tail = rnd(tail_rows, C) if tail else None
    d_s = rnd(t, hc)
    full, out, pre = torch.cat([hist, torch.empty((t, C), device=cuda)]), rnd(t, C), rnd(t, C)
    s, gate, rstd = rnd(t, hc), rnd(t, hc), rnd(t, hc, 3)
    st, p = _lib.stream_ptr(cuda), _lib.ptr
    _lib.call("eg_ple_gate", p(key), p(value), p(hidden), p(nk), p(nq), p(nc), t, hc, n, 1e-6, p(full[h0:]), p(s),
              p(gate), p(rstd), st)
    _lib.call("eg_ple_conv", p(full), h0, t, hc, n, p(conv), 4, 3, 0, p(hidden), p(value), p(gate), p(out), p(pre), st)
    want, got = (torch.full((h0 + t, C), 7.0, device=cuda) for _ in range(2))
    _lib.call("eg_ple_conv_backward", p(full), h0, t, hc, n, p(conv), 4, 3, None, p(d_out), p(d_tail), tail_rows,
              p(want), st)
    size = int(_lib.load().eg_ple_weight_sums_workspace_size(h0, t, hc, n))
    ws = torch.full((size // 4,), float("nan"), device=cuda)
    _lib.call("eg_ple_conv_backward_sums", p(hist), h0, t, hc, n, p(value), p(gate), p(rstd), p(nc), p(conv), p(pre),
              p(d_out), p(d_tail), tail_rows, p(got), p(ws), size, st)
    torch.cuda.synchronize()
    assert torch.equal(got, want)
    # the run kernel without the sums, from the pre-activation
    again = torch.full((h0 + t, C), 7.0, device=cuda)
    _lib.call("eg_ple_conv_backward", None, h0, t, hc, n, p(conv), 4, 3, p(pre), p(d_out), p(d_tail), tail_rows,
              p(again), st)
    assert torch.equal(again, want)

    def outs():
        return [torch.empty(C, device=cuda) for _ in range(3)] + [torch.empty((C, 4), device=cuda)]
    a, b = outs(), outs()
    _lib.call("eg_ple_weight_sums", p(key), p(hidden), p(rstd), p(d_s), p(nk), p(nq), h0, t, hc, n, *map(p, a), p(ws),
              size, st)
    size = int(_lib.load().eg_ple_weight_grads_workspace_size(t, hc, n, 4))
    ws = torch.empty(size // 4, device=cuda)

    def grads(key, hidden, d_s, d_out, d_normed, full, into):
        _lib.call("eg_ple_weight_grads", p(key), p(value), p(hidden), p(gate), p(rstd), p(d_s), p(nk), p(nq), p(d_out),
                  p(d_normed), p(full), h0, p(pre), t, hc, n, 4, 3, *map(p, into), p(ws), size, st)
    grads(key, hidden, d_s, d_out, want[h0:].contiguous(), full, b)
    torch.cuda.synchronize()
    x = pre.double()
    da = (d_out.double() * torch.sigmoid(x) * (1 + x * (1 - torch.sigmoid(x)))).abs()
    kr, hr = (y.double().view(t, hc, n) * rstd[..., i:i + 1].double() for i, y in ((0, key), (1, hidden)))
    ds = d_s.double().unsqueeze(-1) / n ** 0.5
    z = (value.double().unsqueeze(1) * gate.double().unsqueeze(-1) * rstd[..., 2:].double()).reshape(t, C)
    mags = [(ds * hr * nq.double().view(hc, n) * kr).abs().sum(0).reshape(-1),
            (ds * kr * nk.double().view(hc, n) * hr).abs().sum(0).reshape(-1),
            (want[h0:].double() * z).abs().sum(0)]
    pad = torch.cat([torch.zeros((9, C), device=cuda), full]).double().abs()[h0:]
    mags.append(torch.stack([(da * pad[3 * k:3 * k + t]).sum(0) for k in range(4)], dim=1))
    for u, v, m in zip(a, b, mags):
        assert bool(((u.double() - v.double()).abs() <= (t + 8) * 2.0 ** -23 * m + 1e-30).all())


@pytest.mark.parametrize("weights", [False, True])
def test_history_written_over_before_the_backward(cuda, weights):
    """A loop that keeps its history in one buffer overwrites it after the
    forward; the backward's gradients are those of the history the forward read."""
    from engraft_ngram_amd import ple

    class HP:
        hc_mult, n_embd, f_norm_rms_eps, ple_ngram_size = 2, 256, 1e-6, 3
    g = torch.Generator(device=cuda).manual_seed(4)
    rnd = lambda *s: torch.randn(s, generator=g, device=cuda)
    hc, n, t = 2, 256, 70
    w = ple.PleWeights(rnd(hc * n, n) / 16, rnd(n, n) / 16, *(1 + 0.1 * rnd(hc * n) for _ in range(3)), rnd(hc * n, 4))
    emb, hidden, hist, r = rnd(t, n), rnd(t, hc, n) + 0.5, rnd(9, hc, n), rnd(t, hc, n)
    res = []
    for overwrite in (False, True):
        leaves = [emb.clone().requires_grad_(True)]
        ws = {k: v.clone().requires_grad_(weights) for k, v in vars(w).items()}
        leaves += [v for v in ws.values() if weights]
        buf = hist.clone()
        out, new = ple.ple_forward(leaves[0], hidden, ple.PleWeights(**ws), buf, HP)
        if overwrite:
            buf.copy_(new.detach())
        res.append(torch.autograd.grad(out, leaves, r))
    for a, b in zip(*res):
        assert torch.equal(a, b)


def test_gradients_past_the_weight_sums_rows(cuda, monkeypatch):
    """A call of more rows than eg_ple_conv_backward_sums takes keeps its normed rows (the limit set
    to the call's own here): outputs and history as within the limit bit for bit, every
    gradient within T 2^-20 of its largest entry (other orders of the sums over T positions)."""
    from engraft_ngram_amd import _lib, ple
    print("[gpu-test] gradients past the weight sums' rows", file=sys.stderr, flush=True)

    class HP:
        hc_mult, n_embd, f_norm_rms_eps, ple_ngram_size = 2, 256, 1e-6, 3
    g = torch.Generator(device=cuda).manual_seed(9)
    rnd = lambda *s: torch.randn(s, generator=g, device=cuda)
    hc, n, t = 2, 256, 70
    w = ple.PleWeights(rnd(hc * n, n) / 16, rnd(n, n) / 16, *(1 + 0.1 * rnd(hc * n) for _ in range(3)), rnd(hc * n, 4))
    emb, hidden, hist, r = rnd(t, n), rnd(t, hc, n) + 0.5, rnd(9, hc, n), rnd(t, hc, n)
    real, res = _lib.call, []
    for limit in (ple.SUMS_MAX_ROWS, t + 8):
        monkeypatch.setattr(ple, "SUMS_MAX_ROWS", limit)
        called = []
        monkeypatch.setattr(_lib, "call", lambda name, *a: (called.append(name), real(name, *a))[1])
        leaves = [x.clone().requires_grad_(True) for x in (emb, hidden, hist, *vars(w).values())]
        out, new = ple.ple_forward(leaves[0], leaves[1], ple.PleWeights(*leaves[3:]), leaves[2], HP)
        res.append((out, new, *torch.autograd.grad(out, leaves, r)))
        past = limit < t + 9
        assert ("eg_ple_weight_grads" in called) is past and ("eg_ple_conv_backward_sums" in called) is not past
    assert torch.equal(res[0][0], res[1][0]) and torch.equal(res[0][1], res[1][1])
    for a, b in zip(res[0][2:], res[1][2:]):
        assert float((a - b).abs().max()) <= t * 2.0 ** -20 * float(a.abs().max())
