"""The damage scan of blocks cut into several pieces (the first of 2^18 tokens)
against the oracle: hits, counts and statistics at the pieces' and blocks'
edges, where a position's n-grams reach into the tokens of the piece or block
before it.  Ids and counts exact, dnorm_sum within 1e-6 (16 fp32 additions)."""
from __future__ import annotations

import sys

import numpy as np
import pytest

from oracle import damage as DM
from oracle import hash as H
from tests import gpu_util as G
from tests.params import fake_table_spec

pytestmark = pytest.mark.gpu

FIRST = 1 << 18
N = 5 * FIRST + 77


@pytest.fixture(scope="module")
def scan_case():
    spec = fake_table_spec(7)
    rng = np.random.default_rng(21)
    tokens = rng.integers(0, 3_000, N, dtype=np.int64)
    edges = np.unique([FIRST, 2 * FIRST, 4 * FIRST, 700_001, FIRST + 1, 2 * (FIRST + 1)])
    for i, e in enumerate(edges):  # an EOS on, before and after an edge, or none
        if i % 4:
            tokens[e - 2 + i % 4] = spec.eos_token_id
    rows = H.ngram_rows_np(spec, tokens)
    near = np.concatenate([np.arange(e - 4, e + 4) for e in edges])
    ov = np.unique(np.concatenate([rows[near].reshape(-1), rows[::9_001].reshape(-1)]))
    dn = np.linspace(0.5, 2.0, ov.size).astype(np.float32)
    return spec, tokens, ov, dn, DM.scan_hits(spec, tokens, ov, dn, block=N), near


# one block of four pieces; three blocks of two or more pieces; blocks of one whole piece and one of a single token
@pytest.mark.parametrize("block", [8_000_000, 700_001, FIRST + 1])
@pytest.mark.parametrize("dtype", [np.int32, np.int64])
def test_scan_pieces_against_oracle(cuda, scan_case, block, dtype):
    from engraft_ngram_amd import damage
    print(f"[gpu-test] damage scan in pieces block={block} {dtype.__name__}", file=sys.stderr, flush=True)
    spec, tokens, ov, dn, exp, near = scan_case
    tab, _ = G.f32_table(spec, 32, seed=53)
    assert len(damage._pieces(min(block, N))) > 1 and np.isin(near, exp["pos"]).all()
    for _ in range(2):  # again with the pinned buffers of the first call
        got = damage.scan_hits(tokens.astype(dtype), tab, ov, dn, block=block)
        for k in ("pos", "n_hit_rows", "dnorm_max", "read_count"):
            assert np.array_equal(got[k], exp[k]), k
        np.testing.assert_allclose(got["dnorm_sum"], exp["dnorm_sum"], rtol=1e-6)
