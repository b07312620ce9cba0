"""ple_forward on both sides of the lengths where its products change kernels
(FEW_ROWS, H3_MIN_ROWS): the forward without gradients against the oracle with
the history carried across, a weight modified between two calls, and the block
under checkpointing.

Bars: test_gpu_ple.py's (output 1e-4, history 1e-5 or 1e-4, score 1e-4), the
output's beside what the score's own error moves it by, |value| |gate - oracle's|
(the gate's slope is 1/sqrt|s| near a score of zero); the gate within 2^-22 of
the gate of the block's own score."""
from __future__ import annotations

import sys

import pytest
import torch

from oracle import ple as P
from tests.test_gpu_ple import _BARS, _HP, _dev_weights
from tests.test_oracle_ple import ple_weights

pytestmark = pytest.mark.gpu

HC, N = 4, 2560
CHUNKS = (32, 33, 64, 65, 150)


def _say(msg: str) -> None:
    print(f"[gpu-test] {msg}", file=sys.stderr, flush=True)


def _entry(gemm: str, t: int) -> str:
    if t <= 32:
        return "eg_gemm_f32_rows"
    return {"fp32": "eg_gemm_f32", "bf16x3": "eg_gemm_bf16x3",
            "bf16x6": "eg_gemm_f16x3" if t > 64 else "eg_gemm_bf16x6"}[gemm]


def _gate(s):
    s = s.double()
    return torch.sigmoid(torch.sign(s) * torch.sqrt(torch.clamp(s.abs(), min=1e-6)))


@pytest.fixture(scope="module")
def chunks():
    """(weights, per chunk: emb, hidden and the oracle's output, history, score, gate and value)."""
    w = ple_weights(HC, N, seed=13)
    g = torch.Generator().manual_seed(14)
    hist, res = torch.zeros(0, HC, N), []
    for t in CHUNKS:
        emb, hidden = torch.randn((t, N), generator=g) * 0.1, torch.randn((t, HC, N), generator=g) * 0.1
        out, hist, s, gate = P.ple_forward(emb, hidden, w, hist, HC, N, 1e-6, 3)
        res.append((emb, hidden, out, hist, s, gate, emb @ w["w_value"].T))
    return w, res


def _check_chunk(got, hist, diag, chunk, gemm):
    _, _, out, exp_hist, s, gate, value = chunk
    bar_h, _, bar_s = _BARS[gemm]
    assert (diag["s"].cpu() - s).abs().max().item() <= bar_s
    assert (diag["gate"].cpu().double() - _gate(diag["s"].cpu())).abs().max().item() <= 2.0 ** -22
    moved = value.abs().unsqueeze(1) * (diag["gate"].cpu() - gate).abs().unsqueeze(-1)
    assert bool(((got.cpu() - out).abs() <= 1e-4 + moved).all())
    assert (hist.cpu() - exp_hist).abs().max().item() <= bar_h


@pytest.mark.parametrize("gemm", ["fp32", "bf16x3", "bf16x6"])
def test_forward_without_gradients_across_the_lengths(cuda, monkeypatch, chunks, gemm):
    from engraft_ngram_amd import _lib, ple
    w, res = chunks
    wd = _dev_weights(w, cuda)
    real, called = _lib.call, []
    monkeypatch.setattr(_lib, "call", lambda name, *a: (called.append(name), real(name, *a))[1])
    for _ in range(2):  # the second time with the weights' planes of the first
        hist = torch.zeros(0, HC, N, device=cuda)
        for t, chunk in zip(CHUNKS, res):
            _say(f"ple_forward lengths {gemm} t={t}")
            called.clear()
            diag = {}
            got, hist = ple.ple_forward(chunk[0].to(cuda), chunk[1].to(cuda), wd, hist, _HP, diag=diag, gemm=gemm)
            assert [c for c in called if c.startswith("eg_gemm")] == [_entry(gemm, t)]
            _check_chunk(got, hist, diag, chunk, gemm)


def test_weight_modified_between_two_calls_against_the_oracle(cuda, chunks):
    """Past H3_MIN_ROWS, the planes kept of both projections' weights."""
    from engraft_ngram_amd import ple
    _say("ple_forward weights modified between calls")
    w, res = chunks
    w = {k: v.clone() for k, v in w.items()}
    wd = _dev_weights(w, cuda)
    emb, hidden = res[-1][:2]
    empty = torch.zeros(0, HC, N)
    for _ in range(2):
        diag = {}
        out, hist, s, gate = P.ple_forward(emb, hidden, w, empty, HC, N, 1e-6, 3)
        got, new = ple.ple_forward(emb.to(cuda), hidden.to(cuda), wd, empty.to(cuda), _HP, diag=diag)
        _check_chunk(got, new, diag, (emb, hidden, out, hist, s, gate, emb @ w["w_value"].T), "bf16x6")
        for x in (w, vars(wd)):
            x["w_key"].mul_(-1.5)
            x["w_value"][::7] *= 0.5


@pytest.mark.parametrize("t", [33, 96])
@pytest.mark.parametrize("gemm", ["fp32", "bf16x3", "bf16x6"])
@pytest.mark.parametrize("reentrant", [False, True])
def test_checkpointed_bit_identical(cuda, t, gemm, reentrant):
    """Output and gradients as without checkpointing, bit for bit; the first pass of a
    re-entrant checkpoint runs under no_grad and takes the products of a differentiated call all the same
    (its inputs require gradients)."""
    from torch.utils.checkpoint import checkpoint

    from engraft_ngram_amd import ple
    _say(f"ple_forward under checkpoint t={t} {gemm} reentrant={reentrant}")

    class HP:
        hc_mult, n_embd, f_norm_rms_eps, ple_ngram_size = 2, 512, 1e-6, 3
    hc, n = 2, 512
    wd = _dev_weights(ple_weights(hc, n, seed=15), cuda)
    g = torch.Generator(device=cuda).manual_seed(16)
    emb, hidden, r = (torch.randn(s, generator=g, device=cuda) for s in ((t, n), (t, hc, n), (t, hc, n)))
    h0 = torch.zeros(0, hc, n, device=cuda)

    def block(e, h):
        return ple.ple_forward(e, h, wd, h0, HP, gemm=gemm)[0]

    res = []
    for ckpt in (False, True):
        e, h = emb.clone().requires_grad_(True), hidden.clone().requires_grad_(True)
        out = checkpoint(block, e, h, use_reentrant=reentrant) if ckpt else block(e, h)
        out.backward(r)
        res.append((out.detach(), e.grad, h.grad))
    for a, b in zip(*res):
        assert torch.equal(a, b)
