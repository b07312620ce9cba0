"""The measured cases of the n-gram table path: what a user of this package has
it do, through its public entry points, with seeded inputs.

Kinds of case (``kind``):

* ``forward``  -- a prompt's positions: hash, gather, dequantise, overlay,
                  residual add (``table.forward``), in each table format;
* ``decode``   -- one new token of many sequences over an overlaid table
                  (``table.forward_decode``);
* ``descent``  -- one optimizer step of the overlay rows
                  (``DescentState.step``), sparse with requantised rows or
                  dense in fp32 with the pull term;
* ``emb``      -- the differentiable overlay of one packed sequence, built and
                  differentiated (``OverlayEmb.build`` and its backward);
* ``scan``     -- the damage scan of a host token array (``damage.scan_hits``);
* ``ple``      -- the PLE block (``ple.ple_forward``): forward alone, forward
                  and backward to its inputs, or with every weight's gradient.

Sizes are the benchmark's configurations and the reference's real table
format and PLE block.  Tables repeat a pool of seeded rows: a row's bytes do
not matter to the path, which row is read does.
"""
from __future__ import annotations

import math
import types

import numpy as np
import torch

import __graft_entry__

__graft_entry__.load_package()

from engraft_ngram_amd import damage, ple  # noqa: E402
from engraft_ngram_amd import table as tables  # noqa: E402
from engraft_ngram_amd.descent import DescentState  # noqa: E402
from engraft_ngram_amd.overlay import DeviceOverlay  # noqa: E402
from engraft_ngram_amd.seq import OverlayEmb  # noqa: E402

DEV = "cuda"
EOS = 151_643
VOCAB = 151_936
POOL = 1 << 20  # distinct payload rows of a table
SCALE_POOL = (1 << 20) - 3  # distinct scale rows (another period, so rows differ beyond the pool)
IQ4_CODEBOOK = (-127, -104, -83, -65, -49, -35, -22, -10, 1, 13, 25, 38, 53, 69, 89, 113)
ROW_BYTES = {"q8_0": lambda d: d + d // 16, "mxfp8": lambda d: d + d // 32, "bf16": lambda d: 2 * d,
             "iq4_nl": lambda d: d // 32 * 18, "f32": lambda d: 4 * d}
TAPS, DILATION, RMS_EPS = 4, 3, 1e-6


def listed() -> list[dict]:
    full = 320_000_000
    return [
        # one new token of each of 256 served sequences, the table under a 500,000-row overlay
        dict(name="decode_q8_overlay", kind="decode", fmt="q8_0", rows=full, dim=128, ngram=3, heads=8, layers=1,
             seqs=256, overlay=500_000),
        # a batch of eight prompts over the full-size int8 table
        dict(name="prompt_q8", kind="forward", fmt="q8_0", rows=full, dim=128, ngram=3, heads=8, layers=1, batch=8,
             seq=2048, overlay=0, shared=False),
        # one short prompt over the small bf16 table a CPU replica also runs
        dict(name="prompt_bf16_short", kind="forward", fmt="bf16", rows=4_194_304, dim=128, ngram=3, heads=8,
             layers=1, batch=1, seq=2048, overlay=0, shared=False),
        # the model's real row format under a fact overlay (fp32 rows, as its files hold them), prompts of odd length
        dict(name="prompt_iq4_overlay", kind="forward", fmt="iq4_nl", rows=full, dim=160, ngram=3, heads=8, layers=1,
             batch=3, seq=2731, overlay=14_032, shared=True),
        # a long prompt over two MXFP8 table layers with 4-grams
        dict(name="prompt_mxfp8_two_layers", kind="forward", fmt="mxfp8", rows=160_000_000, dim=128, ngram=4, heads=8,
             layers=2, batch=1, seq=32_768, overlay=0, shared=False),
        # a descent step over a batch: the rows it reads (about 226,000) and some more are variables, requantised as
        # the table
        dict(name="descent_sparse_q8", kind="descent", rows=full, seqs=8, seq=2048, variables=235_000, dense=False,
             quant=True, grad="bf16"),
        # the fact descent: one packed sequence, a fact's rows as fp32 variables, dense Adam and the pull term
        dict(name="descent_dense_fact", kind="descent", rows=full, seqs=1, seq=2048, variables=14_032, dense=True,
             quant=False, grad="f32"),
        # the same descent's embedding of its packed sequence and that embedding's gradient
        dict(name="overlay_emb_packed", kind="emb", rows=full, seq=2048, fragments=7, variables=14_032),
        # which positions of a corpus block read an overlaid row
        dict(name="scan_block", kind="scan", rows=full, tokens=8_000_000, overlay=500_000),
        # the PLE block: one decoded token, a prompt, and the descent through it
        dict(name="ple_decode_token", kind="ple", n=2560, hc=4, t=1, history=9, mode="forward", gemm="bf16x6"),
        dict(name="ple_prompt", kind="ple", n=2560, hc=4, t=2048, history=0, mode="forward", gemm="bf16x6"),
        dict(name="ple_descent_weights", kind="ple", n=2560, hc=4, t=1531, history=9, mode="weights", gemm="bf16x6"),
    ]


def draw(rng) -> dict:
    def span(lo: int, hi: int) -> int:  # log-uniform, odd sizes among them
        return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))

    kind = rng.choice(["decode", "forward", "forward", "descent", "emb", "scan", "ple", "ple", "ple"])
    rows = span(4_000_000, 320_000_000)
    if kind == "decode":
        return dict(kind=kind, fmt=rng.choice(["q8_0", "bf16", "mxfp8"]), rows=min(rows, 160_000_000), dim=128,
                    ngram=3, heads=8, layers=1, seqs=span(1, 1024), overlay=rng.choice([0, span(1000, 500_000)]))
    if kind == "forward":
        fmt = rng.choice(["q8_0", "bf16", "mxfp8", "iq4_nl"])
        two = fmt == "mxfp8" and rng.random() < 0.5
        return dict(kind=kind, fmt=fmt, rows=min(rows, 160_000_000 if fmt in ("bf16", "mxfp8") else rows),
                    dim=160 if fmt == "iq4_nl" else 128, ngram=4 if two else 3, heads=8, layers=2 if two else 1,
                    batch=span(1, 8), seq=span(17, 4096), overlay=rng.choice([0, 0, span(1000, 200_000)]),
                    shared=fmt == "iq4_nl")
    if kind == "descent":
        dense = rng.random() < 0.5
        seqs, seq = 1 if dense else span(1, 8), span(64, 2048)
        return dict(kind=kind, rows=rows, seqs=seqs, seq=seq,
                    variables=span(500, 30_000) if dense else seqs * seq * 14, dense=dense, quant=not dense,
                    grad="f32" if dense else "bf16")
    if kind == "emb":
        return dict(kind=kind, rows=rows, seq=span(64, 4096), fragments=span(1, 12), variables=span(500, 30_000))
    if kind == "scan":
        return dict(kind=kind, rows=rows, tokens=span(50_000, 8_000_000), overlay=min(span(1000, 500_000), rows // 64))
    mode = rng.choice(["forward", "forward", "descent", "weights"])
    t = span(1, 2048) if mode == "forward" else span(64, 1531)
    return dict(kind="ple", n=2560, hc=4, t=t, history=rng.choice([0, 9]), mode=mode,
                gemm=rng.choice(["bf16x6", "bf16x6", "bf16x6", "fp32", "bf16x3"]))


# ---- inputs -----------------------------------------------------------------------------------

def _gen(seed: int, salt: int) -> torch.Generator:
    return torch.Generator(device=DEV).manual_seed((seed * 1_000_003 + salt) % (1 << 62))


def _pools(fmt: str, dim: int, seed: int, layer: int):
    """The distinct payload and scale rows of a table layer (values about N(0, 0.02))."""
    g = _gen(seed, 11 + layer)
    if fmt == "iq4_nl":
        p = torch.randint(0, 256, (POOL, 128 * -(-(dim // 32 * 18) // 128)), generator=g, device=DEV,
                          dtype=torch.uint8)
        d = (torch.rand((POOL, dim // 32), generator=g, device=DEV) * 4e-4 + 1e-4).to(torch.float16)
        blocks = p[:, :dim // 32 * 18].view(POOL, dim // 32, 18)
        blocks[:, :, :2] = d.view(torch.uint8).view(POOL, dim // 32, 2)
        return p, None
    x = torch.randn((POOL, dim), generator=g, device=DEV)
    if fmt == "bf16":
        return (x * 0.02).to(torch.bfloat16), None
    if fmt == "f32":
        return x * 0.02, None
    if fmt == "q8_0":
        p = (x * 42).round().clamp(-127, 127).to(torch.int8).view(torch.uint8)
        s = (torch.rand((SCALE_POOL, dim // 32), generator=g, device=DEV) * 4e-4 + 2.5e-4).to(torch.float16)
        return p, s
    p = (x * 90).clamp(-400, 400).to(torch.float8_e4m3fn).view(torch.uint8)
    s = torch.randint(113, 117, (SCALE_POOL, dim // 32), generator=g, device=DEV, dtype=torch.uint8)
    return p, s


def _tile(pool: torch.Tensor, n: int) -> torch.Tensor:
    out = torch.empty((n, pool.shape[1]), dtype=pool.dtype, device=DEV)
    for r in range(0, n, pool.shape[0]):
        m = min(pool.shape[0], n - r)
        out[r:r + m] = pool[:m]
    return out


def _rows64(fmt: str, dim: int, pools, ids: torch.Tensor) -> torch.Tensor:
    """The values of table rows ``ids`` in float64, from the pools alone."""
    p, s = pools
    raw = p[ids % POOL]
    if fmt in ("bf16", "f32"):
        return raw.double()
    if fmt == "iq4_nl":
        b = raw[:, :dim // 32 * 18].reshape(-1, dim // 32, 18)
        d = b[:, :, :2].contiguous().view(torch.float16).double()
        q = torch.cat([b[:, :, 2:] & 15, b[:, :, 2:] >> 4], dim=2).long()
        code = torch.tensor(IQ4_CODEBOOK, dtype=torch.float64, device=DEV)
        return (code[q] * d).reshape(-1, dim)
    sc = s[ids % SCALE_POOL]
    if fmt == "q8_0":
        return (raw.view(torch.int8).double().view(-1, dim // 32, 32) * sc.double().unsqueeze(-1)).view(-1, dim)
    lut = torch.arange(256, dtype=torch.uint8).view(torch.float8_e4m3fn).double().to(DEV)
    return (lut[raw.long()].view(-1, dim // 32, 32) * torch.exp2(sc.double() - 127).unsqueeze(-1)).view(-1, dim)


def _hash(rows: int, ngram: int, heads: int, seed: int, shared: bool) -> dict:
    """Addressing of a table layer: rows split evenly over the heads, odd 64-bit multipliers."""
    n_heads = (ngram - 1) * heads
    rng = np.random.default_rng([seed, 29])
    mult = (rng.integers(1, 2 ** 62, size=(n_heads, ngram)) * 2 + 1).tolist()
    per = rows // n_heads
    return dict(eos_token_id=EOS, ngram_size=ngram, heads_per_ngram=heads, layer_multipliers=mult[0],
                head_vocab_sizes=[per] * n_heads, head_offsets=[h * per for h in range(n_heads)],
                head_multipliers=None if shared else mult)


def _hash64(hp: dict, tokens: torch.Tensor, start: torch.Tensor) -> torch.Tensor:
    """Global row ids [n, n_heads] in plain torch: products wrap modulo 2^64, the modulus is unsigned."""
    idx = torch.arange(tokens.numel(), device=DEV)
    ctx, cut = [tokens], torch.zeros_like(tokens, dtype=torch.bool)
    for s in range(1, hp["ngram_size"]):
        prev = torch.where(idx - s >= start, tokens[(idx - s).clamp_min(0)], EOS)
        cut = cut | (prev == EOS)
        ctx.append(torch.where(cut, EOS, prev))
    cols = []
    for h, (p, off) in enumerate(zip(hp["head_vocab_sizes"], hp["head_offsets"])):
        m = hp["layer_multipliers"] if hp["head_multipliers"] is None else hp["head_multipliers"][h]
        mixed = torch.zeros_like(tokens)
        for j in range(h // hp["heads_per_ngram"] + 2):
            mixed = mixed ^ (ctx[j] * (m[j] - (1 << 64) if m[j] >= 1 << 63 else m[j]))
        local = torch.where(mixed < 0, (mixed.remainder(p) + (1 << 64) % p) % p, mixed.remainder(p))
        cols.append(local + off)
    return torch.stack(cols, dim=1)


def _tokens(n: int, seed: int) -> torch.Tensor:
    """Zipf(1.1) token ids with a document end about every 700 tokens."""
    g = _gen(seed, 5)
    # summed on the host: the device's parallel sum may round differently from run to run
    cdf = torch.cumsum(torch.arange(1, VOCAB + 1, dtype=torch.float64) ** -1.1, 0).to(DEV)
    u = torch.rand(n, generator=g, device=DEV, dtype=torch.float64) * cdf[-1]
    rank = torch.searchsorted(cdf, u).clamp_max(VOCAB - 1)
    tok = torch.randperm(VOCAB, generator=g, device=DEV)[rank]
    return torch.where(torch.rand(n, generator=g, device=DEV) < 1 / 700, EOS, tok)


def _starts(n: int, seq: int) -> torch.Tensor:
    i = torch.arange(n, device=DEV)
    return i // seq * seq


def _table(fmt: str, rows: int, dim: int, hp: dict, seed: int, layer: int = 0):
    p, s = _pools(fmt, dim, seed, layer)
    store = tables.RowStore(fmt, dim, _tile(p, rows), None if s is None else _tile(s, rows))
    return tables.DeviceTable(store, **hp)


def _pick(read: torch.Tensor, of_read: int, k: int, n_rows: int, g: torch.Generator) -> torch.Tensor:
    """``k`` sorted distinct rows: up to ``of_read`` of those read, the rest of the table's others."""
    uniq = torch.unique(read)
    some = uniq[torch.randperm(uniq.numel(), generator=g, device=DEV)[:of_read]]
    other = torch.arange(2 * k + uniq.numel(), device=DEV) * (n_rows // (2 * k + uniq.numel()))
    other = other[~torch.isin(other, uniq)]
    other = other[torch.randperm(other.numel(), generator=g, device=DEV)[:k - some.numel()]]
    return torch.cat([some, other]).sort().values


def _overlay_ids(case: dict, seed: int, read: torch.Tensor) -> torch.Tensor:
    """Overlay ids, up to half of them among the rows read."""
    return _pick(read, case["overlay"] // 2, case["overlay"], case["rows"], _gen(seed, 7)).to(torch.int32)


def _read_inputs(case: dict, seed: int):
    """Of ``forward`` and ``decode``: the layers' addressing, tokens, segment starts and residual."""
    hps = [_hash(case["rows"], case["ngram"], case["heads"], 10 * seed + layer, case.get("shared", False))
           for layer in range(case["layers"])]
    if case["kind"] == "decode":
        n, per = case["seqs"], case["ngram"]
    else:
        n, per = case["batch"] * case["seq"], case["seq"]
    tok = _tokens(case["seqs"] * per if case["kind"] == "decode" else n, seed)
    width = (case["ngram"] - 1) * case["heads"] * case["dim"]
    res = torch.randn((n, width), generator=_gen(seed, 3), device=DEV).to(torch.bfloat16)
    return hps, tok, _starts(tok.numel(), per), res


def _read_rows(case: dict, hps, tok, start):
    rows = [_hash64(hp, tok, start) for hp in hps]
    return [r[case["ngram"] - 1::case["ngram"]] for r in rows] if case["kind"] == "decode" else rows


def _overlay_fmt(case: dict) -> str:
    return "f32" if case["fmt"] == "iq4_nl" else case["fmt"]


def _prepare_read(case: dict, seed: int) -> dict:
    hps, tok, start, res = _read_inputs(case, seed)
    tabs = [_table(case["fmt"], case["rows"], case["dim"], hp, seed, i) for i, hp in enumerate(hps)]
    overlays = None
    if case["overlay"]:
        ids = _overlay_ids(case, seed, _read_rows(case, hps, tok, start)[0])
        p, s = _pools(_overlay_fmt(case), case["dim"], seed, 100)
        store = tables.RowStore(_overlay_fmt(case), case["dim"], p[:ids.numel()].contiguous(),
                                None if s is None else s[:ids.numel()].contiguous())
        ov = DeviceOverlay(ids, store)
        overlays = [ov.with_bitmap(case["rows"]) if case["kind"] == "decode" else ov] + [None] * (len(tabs) - 1)
    if case["kind"] == "decode":
        tok = tok.view(case["seqs"], case["ngram"])
    return dict(case=case, tabs=tabs, tok=tok, res=res, overlays=overlays)


def _exact_read(case: dict, seed: int):
    hps, tok, start, res = _read_inputs(case, seed)
    out = res.double().view(res.shape[0], -1, case["dim"])
    for layer, rows in enumerate(_read_rows(case, hps, tok, start)):
        pools = _pools(case["fmt"], case["dim"], seed, layer)
        ids = None
        if case["overlay"] and layer == 0:
            ids = _overlay_ids(case, seed, rows).long()
            over = _pools(_overlay_fmt(case), case["dim"], seed, 100)
        for h in range(rows.shape[1]):
            emb = _rows64(case["fmt"], case["dim"], pools, rows[:, h])
            if ids is not None:
                at = torch.searchsorted(ids, rows[:, h].contiguous()).clamp_max(ids.numel() - 1)
                hit = ids[at] == rows[:, h]
                emb[hit] = _rows64(_overlay_fmt(case), case["dim"], over, at[hit])
            out[:, h] += emb
    return out.view(res.shape)


def _descent_inputs(case: dict, seed: int):
    hp = _hash(case["rows"], 3, 8, 10 * seed, False)
    n = case["seqs"] * case["seq"]
    tok = _tokens(n, seed)
    rows = _hash64(hp, tok, _starts(n, case["seq"]))
    g = _gen(seed, 9)
    ids = _pick(rows, case["variables"], case["variables"], case["rows"], g)
    d_out = torch.randn((n, 2048), generator=g, device=DEV) * 1e-3
    d_out = d_out.to(torch.bfloat16) if case["grad"] == "bf16" else d_out
    # a descent under way: moments of earlier steps, rows moved off the table's
    m = torch.randn((ids.numel(), 128), generator=g, device=DEV) * 1e-4
    v = torch.rand((ids.numel(), 128), generator=g, device=DEV) * 1e-6
    moved = torch.randn((ids.numel(), 128), generator=g, device=DEV) * 2e-3
    return hp, rows, ids, d_out, m, v, moved


LR, MU, STEPS_BEFORE = 1e-3, 1e-3, 10


def _prepare_descent(case: dict, seed: int) -> dict:
    hp, rows, ids, d_out, m, v, moved = _descent_inputs(case, seed)
    tab = _table("q8_0", case["rows"], 128, hp, seed)
    start = tab.gather(ids.to(torch.int32).reshape(-1, 1)) + moved
    st = DescentState(ids.to(torch.int32), start, quant_fmt="q8_0" if case["quant"] else None, base=tab)
    st.m.copy_(m)
    st.v.copy_(v)
    st.step_count = STEPS_BEFORE
    return dict(case=case, st=st, rows=rows.to(torch.int32), d_out=d_out)


def _run_descent(s: dict):
    case, st = s["case"], s["st"]
    st.step(s["d_out"], s["rows"], lr=LR, dense=case["dense"], mu=MU if case["dense"] else 0.0)
    out = {"rows": st.master, "m": st.m, "v": st.v}
    if case["quant"]:
        out["payload"], out["scales"] = st.quant.payload, st.quant.scales
    return out


def _exact_descent(case: dict, seed: int):
    hp, rows, ids, d_out, m, v, moved = _descent_inputs(case, seed)
    rows0 = _rows64("q8_0", 128, _pools("q8_0", 128, seed, 0), ids)
    p0 = (rows0.float() + moved).double()  # the start is the float32 sum
    m0, v0 = m.double(), v.double()
    flat = rows.reshape(-1)
    at = torch.searchsorted(ids, flat).clamp_max(ids.numel() - 1)
    hit = ids[at] == flat
    grad = torch.zeros_like(p0).index_add_(0, at[hit], d_out.reshape(-1, 128)[hit].double())
    steps = torch.zeros((ids.numel(), 1), dtype=torch.bool, device=DEV)
    steps[at[hit]] = True  # a sparse step moves the rows read alone
    if case["dense"]:
        grad += MU / float(rows0.pow(2).sum()) * 2 * (p0 - rows0)
        steps[:] = True
    b1, b2, eps, t = 0.9, 0.999, 1e-8, STEPS_BEFORE + 1
    m = m0 + (1 - b1) * (grad - m0)
    v = v0 * b2 + (1 - b2) * grad * grad
    p = p0 - LR / (1 - b1 ** t) * m / (v.sqrt() / math.sqrt(1 - b2 ** t) + eps)
    out = {"rows": torch.where(steps, p, p0), "m": torch.where(steps, m, m0), "v": torch.where(steps, v, v0)}
    if case["quant"]:
        out["payload"] = out["scales"] = None
    return out


def _emb_inputs(case: dict, seed: int):
    hp = _hash(case["rows"], 3, 8, 10 * seed, False)
    n = case["seq"]
    tok = _tokens(n, seed)
    g = _gen(seed, 13)
    cuts = torch.randint(1, n, (case["fragments"] - 1,), generator=g, device=DEV).unique()
    seg = torch.searchsorted(cuts, torch.arange(n, device=DEV), right=True)
    start = torch.cat([torch.zeros(1, dtype=torch.int64, device=DEV), cuts])[seg]
    rows = _hash64(hp, tok, start)
    ids = _pick(rows, case["variables"], case["variables"], case["rows"], g)
    moved = torch.randn((ids.numel(), 128), generator=g, device=DEV) * 2e-3
    d_out = torch.randn((n, 2048), generator=g, device=DEV) * 1e-3
    return hp, tok, seg, rows, ids, moved, d_out


def _prepare_emb(case: dict, seed: int) -> dict:
    hp, tok, seg, _, ids, moved, d_out = _emb_inputs(case, seed)
    tab = _table("q8_0", case["rows"], 128, hp, seed)
    var = (tab.gather(ids.to(torch.int32).reshape(-1, 1)) + moved).requires_grad_(True)
    emb = OverlayEmb(tab, tok.tolist(), var, {r: i for i, r in enumerate(ids.tolist())}, segment_ids=seg.cpu())
    return dict(case=case, emb=emb, var=var, d_out=d_out)


def _run_emb(s: dict):
    out = s["emb"].build(s["case"]["seq"])
    (grad,) = torch.autograd.grad(out, s["var"], s["d_out"])
    return {"emb": out.detach(), "grad": grad}


def _exact_emb(case: dict, seed: int):
    _, _, _, rows, ids, moved, d_out = _emb_inputs(case, seed)
    pools = _pools("q8_0", 128, seed, 0)
    flat = rows.reshape(-1)
    at = torch.searchsorted(ids, flat).clamp_max(ids.numel() - 1)
    hit = ids[at] == flat
    var = (_rows64("q8_0", 128, pools, ids).float() + moved).double()
    emb = _rows64("q8_0", 128, pools, flat)
    emb[hit] = var[at[hit]]
    grad = torch.zeros_like(var).index_add_(0, at[hit], d_out.reshape(-1, 128)[hit].double())
    return {"emb": emb.view(case["seq"], -1), "grad": grad}


def _scan_inputs(case: dict, seed: int):
    hp = _hash(case["rows"], 3, 8, 10 * seed, False)
    g = _gen(seed, 17)
    step = case["rows"] // case["overlay"]
    ids = torch.arange(case["overlay"], device=DEV) * step
    ids = ids + torch.randint(0, step, (case["overlay"],), generator=g, device=DEV)
    dnorm = torch.rand(ids.numel(), generator=g, device=DEV)
    return hp, _tokens(case["tokens"], seed), ids, dnorm


def _prepare_scan(case: dict, seed: int) -> dict:
    hp, tok, ids, dnorm = _scan_inputs(case, seed)
    tab = _table("q8_0", case["rows"], 128, hp, seed)
    return dict(case=case, tab=tab, tok=tok.to(torch.int32).cpu().numpy(), ids=ids.to(torch.int32).cpu().numpy(),
                dnorm=dnorm.cpu().numpy())


SCAN_KEYS = ("pos", "n_hit_rows", "dnorm_max", "dnorm_sum", "read_count")


def _whole_scan(case: dict, hits: dict) -> dict:
    """The scan's arrays; those of the hits in zero-filled ones of a length that only the case sets."""
    cap = case["tokens"] // 8 + case["tokens"] * 64 * case["overlay"] // case["rows"]
    out = {"read_count": hits["read_count"], "hits": np.array([hits["pos"].size])}
    for k in SCAN_KEYS[:4]:
        out[k] = np.zeros(cap, dtype=hits[k].dtype)
        out[k][:hits[k].size] = hits[k]
    return out


def _run_scan(s: dict):
    return _whole_scan(s["case"], damage.scan_hits(s["tok"], s["tab"], s["ids"], s["dnorm"]))


def _exact_scan(case: dict, seed: int):
    hp, tok, ids, dnorm = _scan_inputs(case, seed)
    n = tok.numel()
    rows = _hash64(hp, tok, torch.zeros_like(tok))
    count = torch.zeros(ids.numel(), dtype=torch.int64, device=DEV)
    hits = torch.zeros(n, dtype=torch.int64, device=DEV)
    top, total = (torch.zeros(n, dtype=torch.float64, device=DEV) for _ in range(2))
    for h in range(rows.shape[1]):
        col = rows[:, h].contiguous()
        at = torch.searchsorted(ids, col).clamp_max(ids.numel() - 1)
        hit = ids[at] == col
        count += torch.bincount(at[hit], minlength=ids.numel())
        d = torch.where(hit, dnorm[at].double(), 0.0)
        hits += hit
        top, total = torch.maximum(top, d), total + d
    pos = torch.nonzero(hits[:n - 1]).reshape(-1)
    vals = (pos, hits[pos], top[pos], total[pos], count)
    return _whole_scan(case, {k: v.cpu().numpy() for k, v in zip(SCAN_KEYS, vals)})


def _ple_inputs(case: dict, seed: int):
    n, hc, t = case["n"], case["hc"], case["t"]
    g = _gen(seed, 19)

    def rnd(*shape, scale=1.0, mean=0.0):
        return torch.randn(shape, generator=g, device=DEV) * scale + mean

    w = [rnd(hc * n, n, scale=n ** -0.5), rnd(n, n, scale=n ** -0.5), rnd(hc * n, scale=0.1, mean=1.0),
         rnd(hc * n, scale=0.1, mean=1.0), rnd(hc * n, scale=0.1, mean=1.0), rnd(hc * n, TAPS, scale=0.5)]
    # a trained block's scores keep away from zero, where the gate's slope is infinite: the residual
    # stream carries some of the embedding, and so does the key (a score of 4, give or take 1)
    emb = rnd(t, n, scale=0.1)
    hidden = rnd(t, hc, n, scale=0.1) + 0.3 * emb.unsqueeze(1)
    w[0].view(hc, n, n).diagonal(dim1=1, dim2=2).add_(0.3)
    hist = rnd(case["history"], hc, n)
    return w, emb, hidden, hist, rnd(t, hc, n, scale=1e-3)


def _prepare_ple(case: dict, seed: int) -> dict:
    w, emb, hidden, hist, d_out = _ple_inputs(case, seed)
    if case["mode"] != "forward":
        emb.requires_grad_(True)
        hidden.requires_grad_(True)
    if case["mode"] == "weights":
        w = [x.requires_grad_(True) for x in w]
    hp = types.SimpleNamespace(hc_mult=case["hc"], n_embd=case["n"], f_norm_rms_eps=RMS_EPS,
                               ple_ngram_size=DILATION)
    return dict(case=case, w=ple.PleWeights(*w), wrt=[emb, hidden] + (w if case["mode"] == "weights" else []),
                emb=emb, hidden=hidden, hist=hist, d_out=d_out, hp=hp)


def _run_ple(s: dict):
    def call():
        return ple.ple_forward(s["emb"], s["hidden"], s["w"], s["hist"], s["hp"], gemm=s["case"]["gemm"])

    if s["case"]["mode"] == "forward":
        with torch.no_grad():
            out, hist = call()
        return [out, hist]
    out, hist = call()
    return [out.detach(), hist.detach(), *torch.autograd.grad(out, s["wrt"], s["d_out"])]


def _exact_ple(case: dict, seed: int):
    w, emb, hidden, hist, d_out = _ple_inputs(case, seed)
    n, hc, t = case["n"], case["hc"], case["t"]
    w, emb, hidden, hist, d_out = [x.double() for x in w], emb.double(), hidden.double(), hist.double(), d_out.double()
    grads = case["mode"] != "forward"
    wrt = [emb, hidden] + (w if case["mode"] == "weights" else [])
    for x in wrt:
        x.requires_grad_(grads)
    w_key, w_value, nk, nq, nc, conv = w

    def rms(x, weight):
        return x * torch.rsqrt(x.pow(2).mean(dim=-1, keepdim=True) + RMS_EPS) * weight.view(hc, n)

    s = (rms((emb @ w_key.T).view(t, hc, n), nk) * rms(hidden, nq)).sum(dim=-1) / math.sqrt(n)
    gate = torch.sigmoid(torch.sign(s) * torch.sqrt(s.abs().clamp_min(1e-6)))
    gated = (emb @ w_value.T).unsqueeze(1) * gate.unsqueeze(-1)
    full = torch.cat([hist, rms(gated, nc)]).view(-1, hc * n)
    pad = torch.cat([full.new_zeros(((TAPS - 1) * DILATION, hc * n)), full])[case["history"]:]
    acc = sum(pad[k * DILATION:k * DILATION + t] * conv[:, k] for k in range(TAPS))
    out = hidden + gated + torch.nn.functional.silu(acc).view(t, hc, n)
    new_hist = full[-(TAPS - 1) * DILATION:].view(-1, hc, n)
    res = [out.detach(), new_hist.detach()]
    return res + list(torch.autograd.grad(out, wrt, d_out)) if grads else res


# ---- the interface ----------------------------------------------------------------------------

_PREPARE = {"forward": _prepare_read, "decode": _prepare_read, "descent": _prepare_descent, "emb": _prepare_emb,
            "scan": _prepare_scan, "ple": _prepare_ple}
_EXACT = {"forward": _exact_read, "decode": _exact_read, "descent": _exact_descent, "emb": _exact_emb,
          "scan": _exact_scan, "ple": _exact_ple}


def prepare(case: dict, seed: int) -> dict:
    return _PREPARE[case["kind"]](case, seed)


def run(state: dict):
    kind = state["case"]["kind"]
    if kind == "forward":
        return tables.forward(state["tabs"], state["tok"], state["res"], overlays=state["overlays"],
                              seq_len=state["case"]["seq"])
    if kind == "decode":
        return tables.forward_decode(state["tabs"], state["tok"], state["res"], overlays=state["overlays"])
    return {"descent": _run_descent, "emb": _run_emb, "scan": _run_scan, "ple": _run_ple}[kind](state)


def exact(case: dict, seed: int):
    return _EXACT[case["kind"]](case, seed)


def work(case: dict) -> dict:
    kind = case["kind"]
    if kind in ("forward", "decode"):
        heads = (case["ngram"] - 1) * case["heads"]
        n = case["seqs"] if kind == "decode" else case["batch"] * case["seq"]
        tok = 8 * n * (case["ngram"] if kind == "decode" else 1)
        row = ROW_BYTES[case["fmt"]](case["dim"])
        return {"bytes": n * heads * (case["layers"] * row + 4 * case["dim"]) + tok,
                "flops": n * heads * case["dim"] * 2 * case["layers"]}
    if kind == "descent":
        slots = case["seqs"] * case["seq"] * 16
        # a sparse step touches the rows read: Zipf streams repeat about one slot in seven
        var = case["variables"] if case["dense"] else int(slots * 0.86)
        d_out = slots * 128 * (2 if case["grad"] == "bf16" else 4)
        return {"bytes": d_out + 4 * slots + var * (6 * 512 + (136 if case["quant"] or case["dense"] else 0)),
                "flops": slots * 128 + var * 128 * 12}
    if kind == "emb":
        slots = case["seq"] * 16
        return {"bytes": slots * (136 + 512 + 8 + 512) + case["variables"] * 2 * 512, "flops": slots * 128 * 2}
    if kind == "scan":
        # int32 tokens, each read once, an int64 read count a row, about one position in forty a hit
        return {"bytes": 4 * case["tokens"] + case["overlay"] * 16 + case["tokens"] // 40 * 20,
                "flops": case["tokens"] * 16 * 6}
    n, hc, t = case["n"], case["hc"], case["t"]
    gemm = 2 * t * n * (hc + 1) * n
    weights = 4 * (hc + 1) * n * n
    acts = 4 * t * n * (2 * hc + 1) + 8 * case["history"] * hc * n
    if case["mode"] == "forward":
        return {"bytes": weights + acts, "flops": gemm + 20 * t * hc * n}
    back = 4 * t * n * (2 * hc + 1)
    if case["mode"] == "descent":
        return {"bytes": weights + acts + back, "flops": 2 * gemm + 60 * t * hc * n}
    return {"bytes": 2 * weights + acts + back, "flops": 3 * gemm + 80 * t * hc * n}


def tolerance(case: dict):
    kind = case["kind"]
    if kind in ("forward", "decode"):
        return {"rel": 6e-3}  # one rounding to bf16
    if kind == "descent":
        # float32 sums and one Adam step; a row's requantisation may round a tie the other way
        return {"rel": 1e-6, "differ": 1e-3}
    if kind == "emb":
        return {"rel": 1e-6}
    if kind == "scan":
        return {"rel": 1e-6, "differ": 0.0}
    # float32 products (16 significand bits with bf16x3); the gate's slope amplifies a rounding in the gradients
    if case["gemm"] == "bf16x3":
        return {"rel": 1e-4 if case["mode"] == "forward" else 5e-4}
    return {"rel": 3e-6 if case["mode"] == "forward" else 1.2e-5}
