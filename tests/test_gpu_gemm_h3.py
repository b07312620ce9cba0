"""eg_split_f16 + eg_gemm_f16x3 (fp32 accuracy from three products on the fp16
matrix cores) against float64 products of the same fp32 operands.

Bar: |C - C64| <= ((k + 2) 2^-24 + 3 2^-22) (|A| |B|^T): an fp32 sum of k
products in any order, plus what the split drops of each product (lo*lo and
the two lo planes' rounding, 2^-22 each at most).  Rows spread over less than
2^18 are within the planes' 22 bits everywhere; marked rows (most values 2^24
below the largest, tiny, infinite, NaN) are computed in fp32 and held to the
same bar."""
from __future__ import annotations

import sys

import pytest
import torch

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


# edges of the 256 x 256 tiles, 32-row blocks and 32-wide K steps; the register and the
# re-reading forms of the split (rows of 2560 / columns of 2048 values); K ranges of the last round
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
