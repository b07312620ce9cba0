"""eg_gemm_f32_rows (up to 4 rows on the vector units, up to 8 and up to 32 on
the matrix cores) against float64:
the fp32 GEMM's bar |C - C64| <= (k + 2) 2^-24 (|A| |B|^T), single products
exact, at the edges of its 32-column blocks, its wavefronts' K steps and its
two segments; 33 rows are refused."""
from __future__ import annotations

import sys

import pytest
import torch

pytestmark = pytest.mark.gpu


# k in steps of 32: fewer steps than wavefronts, one turn of three and its remainders; more than 256 column blocks
@pytest.mark.parametrize("m,n,n2,ks", [(1, 1, 0, (32,)), (1, 10240, 2560, (2560,)), (32, 33, 31, (512, 32)),
                                       (31, 64, 0, (160, 2560)), (7, 8225, 40, (800,)), (2, 100, 0, (10240, 2560)),
                                       (5, 2560, 0, (1536,)), (1, 10241, 3, (288, 32)),
                                       (3, 10300, 2, (256,)), (4, 37, 1, (2592,)), (2, 10240, 0, (544,))])
@pytest.mark.parametrize("accumulate", [False, True])
def test_few_rows_against_float64(cuda, m, n, n2, ks, accumulate):
    from engraft_ngram_amd.ple import gemm_f32
    print(f"[gpu-test] gemm_f32 rows m={m} n={n} n2={n2} k={ks} acc={accumulate}", file=sys.stderr, flush=True)
    g = torch.Generator(device=cuda).manual_seed(m + n + sum(ks))
    rnd = lambda *s: torch.randn(s, generator=g, device=cuda)
    a = [rnd(m, k) for k in ks]
    b, b2 = ([rnd(r, k) for k in ks] for r in (n, n2))
    outs = [rnd(m, n), rnd(m, n2)] if accumulate else [None, None]
    base = [None if o is None else o.clone() for o in outs]
    got = gemm_f32(a[0], b[0], *((a[1], b[1]) if len(ks) > 1 else ()), b_n2=b2[0] if n2 else None,
                   b2_n2=b2[1] if n2 and len(ks) > 1 else None, out=outs[0], out2=outs[1] if n2 else None,
                   accumulate=accumulate, few_rows=True)
    torch.cuda.synchronize()
    for o, y, c in zip(got if n2 else (got,), (b, b2), base):
        exp = sum(p.double() @ q.double().T for p, q in zip(a, y))
        mag = sum(p.double().abs() @ q.double().abs().T for p, q in zip(a, y))
        if c is not None:
            exp, mag = exp + c.double(), mag + c.double().abs()
        assert bool(((o.double() - exp).abs() <= (sum(ks) + 2) * 2.0 ** -24 * mag).all())


def test_few_rows_single_products_exact(cuda):
    from engraft_ngram_amd.ple import gemm_f32
    g = torch.Generator(device=cuda).manual_seed(3)
    a = torch.randn((32, 96), generator=g, device=cuda)
    b = torch.zeros((96, 96), device=cuda)
    perm = torch.randperm(96, generator=g, device=cuda)
    b[torch.arange(96, device=cuda), perm] = 0.5
    for m in (1, 2, 3, 4, 5, 8, 9, 32):
        assert torch.equal(gemm_f32(a[:m], b, few_rows=True), a[:m, perm] * 0.5)


def test_more_rows_are_refused(cuda):
    from engraft_ngram_amd import _lib
    from engraft_ngram_amd.ple import gemm_f32
    with pytest.raises(_lib.EgError, match="33 rows"):
        gemm_f32(torch.zeros((33, 32), device=cuda), torch.zeros((8, 32), device=cuda), few_rows=True)
