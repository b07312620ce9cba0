"""eg_split_f16 + eg_gemm_f16x3 (fp32 accuracy from three products on the fp16
matrix cores) against float64 products of the same fp32 operands.

Bar: |C - C64| <= ((k + 2) 2^-24 + 3 2^-22) (|A| |B|^T): an fp32 sum of k
products in any order, plus what the split drops of each product (lo*lo and
the two lo planes' rounding, 2^-22 each at most).  Rows spread over less than
2^18 are within the planes' 22 bits everywhere; marked rows (a share of the values far
below the largest, tiny, infinite, NaN) are computed in fp32, where the other row
does not make up for it, and held to the same bar."""
from __future__ import annotations

import sys

import pytest
import torch

from oracle import ple as P

pytestmark = pytest.mark.gpu


def _say(msg: str) -> None:
    print(f"[gpu-test] {msg}", file=sys.stderr, flush=True)


def _check(got, a, b):
    exp = sum(x.double() @ y.double().T for x, y in zip(a, b))
    mag = sum(x.double().abs() @ y.double().abs().T for x, y in zip(a, b))
    k = sum(x.shape[1] for x in a)
    torch.cuda.synchronize()
    fin = torch.isfinite(exp)
    assert torch.equal(torch.isfinite(got), fin)
    err = (got.double() - exp).abs()[fin]
    tol = (k + 2) * 2.0 ** -24 + 3 * 2.0 ** -22
    assert bool((err <= tol * mag[fin] + 1e-36).all()), float((err / (mag[fin] + 1e-300)).max())


def _matrix(rows, k, g, dev, layout):
    """[rows, k] values over 2^12 in magnitude: row-major, transposed, or a column slice (odd row stride)."""
    def val(*shape):
        x = torch.rand(shape, generator=g, device=dev) * 2 - 1
        return torch.where(x == 0, 1.0, x.sign()) * torch.exp2(x.abs() * 12 - 6)
    if layout == "t":
        return val(k, rows).T
    if layout == "slice":
        return val(rows, k + 3)[:, 1:k + 1]
    return val(rows, k)


# edges of the 256 x 256 tiles, 32-row blocks and 32-wide K steps; K ranges of the last round
@pytest.mark.parametrize("m,n,n2,ks,layout", [
    (1, 1, 0, (1,), "r"), (65, 33, 31, (31,), "r"), (256, 256, 256, (32,), "slice"), (257, 255, 0, (33, 65), "r"),
    (300, 513, 1, (2560,), "r"), (31, 260, 40, (2561,), "slice"), (130, 200, 0, (2048,), "t"),
    (70, 300, 0, (2049,), "t"), (96, 100, 64, (40, 2600), "t"), (2048, 2048, 512, (640,), "r")])
def test_gemm_h3_against_float64(cuda, m, n, n2, ks, layout):
    from engraft_ngram_amd.ple import gemm_h3
    _say(f"gemm_h3 m={m} n={n} n2={n2} k={ks} {layout}")
    g = torch.Generator(device=cuda).manual_seed(m + n + sum(ks))
    a, b = (tuple(_matrix(r, k, g, cuda, layout) for k in ks) for r in (m, n))
    b2 = tuple(_matrix(n2, k, g, cuda, layout) for k in ks) if n2 else None
    got = gemm_h3(a, b, b2)
    for o, y in zip(got if n2 else (got,), (b, b2)):
        _check(o, a, y)


# the split keeps a row's values in registers up to 2,560 of them (80 steps of 32), a column's up
# to 1,536 (48 steps), and reads longer ones again: the last of each form and the first past it
@pytest.mark.parametrize("layout,ks", [("r", (2529,)), ("r", (2560,)), ("r", (2561,)), ("slice", (2560,)),
                                       ("r", (2500, 40)), ("r", (2530, 40)), ("t", (1505,)), ("t", (1536,)),
                                       ("t", (1537,)), ("t", (1568,)), ("t", (1500, 20)), ("t", (1500, 40))])
def test_gemm_h3_split_in_registers_and_read_again(cuda, layout, ks):
    from engraft_ngram_amd.ple import gemm_h3
    _say(f"gemm_h3 split forms {layout} k={ks}")
    g = torch.Generator(device=cuda).manual_seed(sum(ks))
    a, b = (tuple(_matrix(r, k, g, cuda, layout) for k in ks) for r in (41, 67))
    _check(gemm_h3(a, b), a, b)


@pytest.mark.parametrize("layout", ["r", "t"])
def test_gemm_h3_marked_rows(cuda, layout):
    """Rows the planes cannot hold on either side, beside ordinary ones of the same tiles."""
    from engraft_ngram_amd.ple import gemm_h3
    _say(f"gemm_h3 marked rows {layout}")
    g = torch.Generator(device=cuda).manual_seed(5)
    a, b = (_matrix(r, 96, g, cuda, layout) for r in (200, 330))
    a[3, 5] = 1e30  # a wide row whose other elements meet a zero column of b
    b[:, 5] = 0.0
    a[70] *= 1e-30
    a[129, 1] = float("nan")
    a[10] = 0.0
    b[77, 0] = 1e12
    b[150, 7] = float("inf")
    _check(gemm_h3((a,), (b,)), (a,), (b,))


def test_gemm_h3_repeats_bitwise_and_in_a_graph(cuda):
    from engraft_ngram_amd.ple import gemm_h3
    _say("gemm_h3 repeated and captured")
    g = torch.Generator(device=cuda).manual_seed(6)
    a, b = _matrix(1500, 320, g, cuda, "r"), _matrix(700, 320, g, cuda, "t")
    first = gemm_h3((a,), (b,))
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream):
        assert torch.equal(gemm_h3((a,), (b,)), first)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream):
            out = gemm_h3((a,), (b,))
    for i in range(3):
        a[i, i] = 1e30 * i  # ordinary, then marked
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, gemm_h3((a,), (b,)))


def _rel(got, exp):
    return float((got.double() - exp).norm() / exp.norm())


@pytest.mark.parametrize("layout", ["r", "t"])
@pytest.mark.parametrize("p", [0, 12, 24, -24, 30, 36, -36, 37, 40, 60])
def test_gemm_h3_sources_of_different_size(cuda, p, layout):
    """a1 2^-p of a2 where b1 is 2^p of b2: both products count alike, so both
    keep an fp32 product's accuracy.  2-norm bar, no K in it but the sums': 3 2^-22
    for what the split drops of each product, and 2^-24 times the square root
    of the number of fp32 additions (three products a 16-wide step)."""
    from engraft_ngram_amd.ple import gemm_h3
    _say(f"gemm_h3 two sources p={p} {layout}")
    g = torch.Generator(device=cuda).manual_seed(100 + p)
    m, n, ks = 300, 270, (320, 96)

    def rnd(rows, k):
        return torch.randn((rows, k) if layout == "r" else (k, rows), generator=g, device=cuda)
    a, b = ([rnd(r, k) for k in ks] for r in (m, n))
    a[0] *= 2.0 ** -p
    b[0] *= 2.0 ** p
    if layout == "t":
        a, b = [x.T for x in a], [x.T for x in b]
    a[0][5], a[1][7], b[0][9], b[1][11] = 0.0, 0.0, 0.0, 0.0  # rows with one source, of zeros in the other
    got = gemm_h3(tuple(a), tuple(b))
    exp = sum(x.double() @ y.double().T for x, y in zip(a, b))
    bar = 3 * 2.0 ** -22 + (3 * sum(ks) / 16) ** 0.5 * 2.0 ** -24
    assert _rel(got, exp) <= bar
    for i in (5, 7):
        assert _rel(got[i], exp[i]) <= bar
    for j in (9, 11):
        assert _rel(got[:, j], exp[:, j]) <= bar


@pytest.mark.parametrize("wide", [1e-7, 1e-11])
def test_ple_backward_with_a_value_projection_near_zero(cuda, wide):
    """A block added with its value projection near zero: d_emb's two sources
    (d_key w_key and d_value w_value) differ by its factor each, one up and one
    down.  Against float64 autograd of the block; the bar allows each of its dozen
    fp32 stages 2^-20 (the key's rounding enters through the gate's slope)."""
    from engraft_ngram_amd import ple

    class HP:
        hc_mult, n_embd, f_norm_rms_eps, ple_ngram_size = 2, 256, 1e-30, 3
    _say(f"ple backward with w_value times {wide}")
    g = torch.Generator(device=cuda).manual_seed(8)
    rnd = lambda *s: torch.randn(s, generator=g, device=cuda)
    hc, n, t = 2, 256, 96
    emb = rnd(t, n)
    hidden = rnd(t, hc, n) * 0.1 + 0.5 * emb.unsqueeze(1)
    wk, wv = rnd(hc * n, n) / 16, rnd(n, n) / 16 * wide
    wk.view(hc, n, n).diagonal(dim1=1, dim2=2).add_(0.5)  # scores away from zero
    w = ple.PleWeights(wk, wv, *(1 + 0.1 * rnd(hc * n) for _ in range(3)), rnd(hc * n, 4) / 2)
    r = rnd(t, hc, n)
    e = emb.clone().requires_grad_(True)
    out, _ = ple.ple_forward(e, hidden, w, hidden.new_zeros((0, hc, n)), HP)
    got, = torch.autograd.grad(out, e, r)
    e64 = emb.cpu().double().requires_grad_(True)
    w64 = {k: v.cpu().double() for k, v in vars(w).items()}
    out64 = P.ple_forward(e64, hidden.cpu().double(), w64, torch.zeros((0, hc, n), dtype=torch.float64), hc, n,
                          HP.f_norm_rms_eps, 3)[0]
    exp, = torch.autograd.grad(out64, e64, r.cpu().double())
    _say(f"d_emb off by {_rel(got.cpu(), exp):.2e}")
    assert _rel(got.cpu(), exp) <= 1e-5


def _sums_bar(k: int) -> float:
    """2-norm: 3 2^-22 for what the split drops, 2^-24 times the root of the fp32 additions of a marked row's
    output (one a k; the planes' three products take fewer)."""
    return 3 * 2.0 ** -22 + k ** 0.5 * 2.0 ** -24


@pytest.mark.parametrize("layout", ["r", "t"])
@pytest.mark.parametrize("p", [17, 19, 22, 24, 30, 50, 100])
def test_gemm_h3_one_column_far_above_the_rest(cuda, p, layout):
    """Rows of values in [1, 2) with one 2^p above them that meets weights 2^-p, or
    zeros: most values lie below the planes' 22 bits, on either side."""
    from engraft_ngram_amd.ple import gemm_h3
    _say(f"gemm_h3 outlier column p={p} {layout}")
    g = torch.Generator(device=cuda).manual_seed(p)
    m, n, k = 150, 140, 1536
    a = 1 + torch.rand((m, k), generator=g, device=cuda)
    b = torch.randn((n, k), generator=g, device=cuda)
    a[:, 700] *= 2.0 ** p
    b[:, 700] *= 2.0 ** -p
    b[::3, 700] = 0.0
    if layout == "t":
        a, b = (x.T.contiguous().T for x in (a, b))
    exp = a.double() @ b.double().T
    for got in (gemm_h3((a,), (b,)), gemm_h3((b,), (a,)).T):
        assert _rel(got, exp) <= _sums_bar(k)
        assert _rel(got[::3], exp[::3]) <= _sums_bar(k)
        assert _rel(got[:, ::3], exp[:, ::3]) <= _sums_bar(k)


@pytest.mark.parametrize("k,low,p", [(32, 31, 23), (1536, 90, 30), (1536, 90, 50), (1536, 1500, 20), (160, 2, 30)])
def test_gemm_h3_low_values_among_zeros(cuda, k, low, p):
    """One value 1, `low` values around 2^-p and zeros (a gradient over positions of
    which few have a loss), against columns that are zero at the 1: the low values are
    counted among the nonzero ones."""
    from engraft_ngram_amd.ple import gemm_h3
    _say(f"gemm_h3 low values k={k} low={low} p={p}")
    g = torch.Generator(device=cuda).manual_seed(k + low + p)
    m, n = 140, 130
    a = torch.zeros((m, k), device=cuda)
    a[:, 0] = 1.0
    a[:, 1:1 + low] = torch.randn((m, low), generator=g, device=cuda) * 2.0 ** -p
    a = a[:, torch.randperm(k, generator=g, device=cuda)]
    b = torch.randn((n, k), generator=g, device=cuda)
    b[:, (a[0] == 1.0).nonzero()[0, 0]] = 0.0
    exp = a.double() @ b.double().T
    for x, y in ((a, b), (a.T.contiguous().T, b.T.contiguous().T)):
        assert _rel(gemm_h3((x,), (y,)), exp) <= _sums_bar(k)
        assert _rel(gemm_h3((y,), (x,)).T, exp) <= _sums_bar(k)


def test_gemm_h3_outputs_beside_a_marked_row(cuda):
    """An output takes the fp32 path for its own rows' marks alone: its neighbours' bits stay."""
    from engraft_ngram_amd.ple import gemm_h3
    _say("gemm_h3 neighbours of marked rows")
    g = torch.Generator(device=cuda).manual_seed(12)
    a, b = _matrix(300, 100, g, cuda, "r"), _matrix(270, 100, g, cuda, "t")
    first = gemm_h3((a,), (b,))
    a[129, 3], b[77, 9], b[269, 0] = 1e30, float("inf"), 1e20
    got = gemm_h3((a,), (b,))
    _check(got, (a,), (b,))
    keep = torch.ones_like(first, dtype=torch.bool)
    keep[129], keep[:, 77], keep[:, 269] = False, False, False
    assert torch.equal(got[keep], first[keep])


def test_gemm_h3_converts_other_dtypes(cuda):
    from engraft_ngram_amd.ple import gemm_h3
    _say("gemm_h3 of bf16 and float64 operands")
    g = torch.Generator(device=cuda).manual_seed(13)
    a, b = (torch.randn((r, 70), generator=g, device=cuda).bfloat16() for r in (40, 33))
    exp = gemm_h3((a.float(),), (b.float(),))
    assert torch.equal(gemm_h3((a,), (b.double(),)), exp)


@pytest.mark.parametrize("ks", [(1024,), (512, 160), (2624,), (96,)])
@pytest.mark.parametrize("p", [15, 22, 30, 60])
def test_gemm_h3_rows_small_outside_a_part(cuda, ks, p):
    """Rows of which a quarter is 2^p above the rest (a stream with a steep gradient): what their
    planes lose counts for columns that are small there, alone.  Those are computed in fp32; the
    columns that are not keep the planes' bits (those of the rows without what is lost: at
    p 60 nothing is left of it).  At the rule's line too: of K / 4 large values, K / 16 of a column's
    are large as well, or one fewer."""
    from engraft_ngram_amd.ple import gemm_h3
    _say(f"gemm_h3 rows small outside a part k={ks} p={p}")
    g = torch.Generator(device=cuda).manual_seed(sum(ks) + p)
    m, n = 70, 96

    def near(*shape):  # within 2^-6 of the largest, which is below 2: all of them near
        x = torch.rand(shape, generator=g, device=cuda) * 1.9 - 0.95
        return x + 0.05 * x.sign()
    a, b, a0 = [], [], []
    for k in ks:
        x, y = near(m, k), near(n, k)
        q = k // 4
        x[:, q:] *= 2.0 ** -p
        x[:35, 0], y[:, 0] = 1.0, 1.0  # the largest of each row in the part
        y[0::4, :q] = 0.0                     # nothing of the part
        y[1::4, (k + 15) // 16:q] = 0.0        # exactly enough of it
        y[2::4, (k + 15) // 16 - 1:q] = 0.0     # one too few
        x[40] = 0.0                           # a row of zeros
        a.append(x), b.append(y)
        a0.append(torch.where(torch.arange(k, device=cuda) < q, x, 0.0))
    k = sum(ks)
    exp = sum(x.double() @ y.double().T for x, y in zip(a, b))
    for flip in (False, True):
        got = gemm_h3(tuple(b), tuple(a)).T if flip else gemm_h3(tuple(a), tuple(b))
        without = gemm_h3(tuple(b), tuple(a0)).T if flip else gemm_h3(tuple(a0), tuple(b))
        for c in range(4):
            assert _rel(got[:, c::4], exp[:, c::4]) <= _sums_bar(k), (c, flip)
        assert not got[40].any()
        if p == 60:
            for c in (1, 3):
                assert torch.equal(got[:, c::4], without[:, c::4]), (c, flip)
            assert _rel(got[:, 0::4], exp[:, 0::4]) <= _sums_bar(k) and not without[:, 0::4].any()


@pytest.mark.parametrize("steps", [9, 32])
def test_gemm_h3_second_source_from_every_step_on(cuda, steps):
    """A tile's K is cut into ranges; the second source begins at every step of them (the first,
    inside, the last, past the last), 2^24 from the first in size."""
    from engraft_ngram_amd.ple import gemm_h3
    _say(f"gemm_h3 second source from every of {steps} steps")
    g = torch.Generator(device=cuda).manual_seed(steps)
    m, n, k = 70, 260, 32 * steps
    a, b = (torch.randn((r, k), generator=g, device=cuda) for r in (m, n))
    for q in range(32, k, 32):
        x, y = (a[:, :q] * 2.0 ** -24, a[:, q:]), (b[:, :q] * 2.0 ** 24, b[:, q:])
        got = gemm_h3(x, y)
        exp = a.double() @ b.double().T
        assert _rel(got, exp) <= 3 * 2.0 ** -22 + (3 * k / 16) ** 0.5 * 2.0 ** -24, q
