"""What ple_forward keeps of its weights between calls (their bf16 and fp16
planes and transposes): a weight modified in place, another stream, and calls
captured into a graph, each against a call with fresh weights, bit for bit."""
from __future__ import annotations

import sys

import pytest
import torch

pytestmark = pytest.mark.gpu

HC, N = 2, 256


class _HP:
    hc_mult, n_embd, f_norm_rms_eps, ple_ngram_size = HC, N, 1e-6, 3


def _say(msg: str) -> None:
    print(f"[gpu-test] {msg}", file=sys.stderr, flush=True)


def _inputs(dev, t, seed):
    g = torch.Generator(device=dev).manual_seed(seed)
    rnd = lambda *s: torch.randn(s, generator=g, device=dev)
    w = dict(w_key=rnd(HC * N, N) / 16, w_value=rnd(N, N) / 16, conv1d=rnd(HC * N, 4),
             **{k: 1 + 0.1 * rnd(HC * N) for k in ("norm_key", "norm_query", "norm_conv")})
    return w, rnd(t, N), rnd(t, HC, N), rnd(9, HC, N), rnd(t, HC, N)


def _call(w, emb, hidden, hist, d_out, gemm, grads):
    from engraft_ngram_amd import ple
    if not grads:
        with torch.no_grad():
            return list(ple.ple_forward(emb, hidden, ple.PleWeights(**w), hist, _HP, gemm=gemm))
    e = emb.detach().requires_grad_(True)
    out, new = ple.ple_forward(e, hidden, ple.PleWeights(**w), hist, _HP, gemm=gemm)
    return [out.detach(), new.detach(), *torch.autograd.grad(out, e, d_out)]


def _fresh(w, *rest):
    return _call({k: v.clone() for k, v in w.items()}, *rest)


def _equal(got, exp):
    torch.cuda.synchronize()
    for a, b in zip(got, exp):
        assert torch.equal(a, b)


# 48 positions: bf16 planes and transposes; 96: fp16 planes where the default takes them
CASES = [(t, gemm, grads) for t in (48, 96) for gemm in ("bf16x6", "bf16x3") for grads in (False, True)]


@pytest.mark.parametrize("t,gemm,grads", CASES)
def test_weight_modified_in_place_and_another_stream(cuda, t, gemm, grads):
    _say(f"weight cache t={t} {gemm} grads={grads}")
    w, *rest = _inputs(cuda, t, t)
    rest += [gemm, grads]
    first = _call(w, *rest)
    _equal(_call(w, *rest), first)
    w["w_key"].mul_(1.5)
    w["w_value"][3] = 0.25
    second = _fresh(w, *rest)
    _equal(_call(w, *rest), second)
    assert not torch.equal(first[0], second[0])
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream):
        w["w_value"].neg_()
        got = _call(w, *rest)
    torch.cuda.current_stream().wait_stream(stream)
    _equal(got, _fresh(w, *rest))
    _equal(_call(w, *rest), got)


@pytest.mark.parametrize("t", [48, 96])
def test_planes_of_superseded_weights_are_let_go(cuda, t):
    """Training both projections: what is held does not grow with the steps."""
    _say(f"planes of superseded weights t={t}")
    w, *rest = _inputs(cuda, t, 5)
    held = []
    for _ in range(12):
        for grads in (False, True):
            _call(w, *rest, "bf16x6", grads)
        w["w_key"].mul_(1.01)
        w["w_value"].mul_(1.01)
        held.append(torch.cuda.memory_allocated())
    assert held[-1] <= held[0], [h - held[0] for h in held]


@pytest.mark.parametrize("t,gemm,grads", CASES)
def test_captured_call_takes_the_weights_of_the_replay(cuda, t, gemm, grads):
    """Warmed up and captured on one stream, the weights modified in place
    between replays, with eager calls and synchronizations between them; and an
    eager call after a capture that was never replayed."""
    _say(f"weight cache under capture t={t} {gemm} grads={grads}")
    w, *rest = _inputs(cuda, t, t + 1)
    rest += [gemm, grads]
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream):
        for _ in range(2):
            _call(w, *rest)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream):
            out = _call(w, *rest)
        for i in range(3):
            w["w_key"].mul_(1.25)
            w["w_value"][i] += 0.5
            graph.replay()
            _equal(out, _fresh(w, *rest))
            _equal(_call(w, *rest), out)
        v, *rest = _inputs(cuda, t, t + 2)
        rest += [gemm, grads]
        never = torch.cuda.CUDAGraph()
        with torch.cuda.graph(never, stream=stream):
            _call(v, *rest)
        _equal(_call(v, *rest), _fresh(v, *rest))
    torch.cuda.current_stream().wait_stream(stream)
