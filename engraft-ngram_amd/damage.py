"""The damage plan's table half on the device: the drop-in for
``ngram_rows`` / ``iter_blocks`` / ``scan_hits`` / ``compute_rows_delta``
(``engraft/damage.py:68-224``).

``scan_hits`` runs one fused launch per corpus block (``eg_scan_overlay``):
every position hashes its ``n_heads`` rows (the whole block as one sequence,
so every position sees its real predecessors), looks each up in the sorted
overlay ids, counts the reads of every overlay row and reduces per position
the number of overlay rows read and the max / sum of their ``dnorm``.  Blocks
overlap by ``ngram_size - 1`` tokens, whose positions are dropped, so the
result equals a scan of the whole corpus as one sequence.
"""
from __future__ import annotations

import ctypes
import time
from concurrent.futures import wait
from typing import Iterator

import numpy as np
import torch

from . import _lib
from .descent import _read_true_rows

BLOCK_TOKENS = 8_000_000  # engraft/damage.py:60


def ngram_rows(tokens: np.ndarray, table) -> tuple[np.ndarray, ...]:
    """Global rows of every position of ``tokens``, one int64 ``[n,
    heads_per_ngram]`` array per n-gram order (bigram, trigram, ...;
    ``engraft/damage.py:68-104`` returns the bigram and trigram arrays of an
    ``ngram_size = 3`` table)."""
    tok = np.asarray(tokens).reshape(-1)
    if tok.size == 0:
        return tuple(np.zeros((0, table.heads_per_ngram), dtype=np.int64) for _ in range(table.ngram_size - 1))
    rows = table.rows(torch.as_tensor(tok.astype(np.int64))).cpu().numpy().astype(np.int64)
    k = table.heads_per_ngram
    return tuple(rows[:, o * k:(o + 1) * k] for o in range(table.ngram_size - 1))


def iter_blocks(tokens: np.ndarray, block: int = BLOCK_TOKENS, overlap: int = 2) -> Iterator[tuple[int, np.ndarray]]:
    """``(offset, tokens[offset-overlap : offset+block])`` -- ``overlap``
    tokens of history (none on the first block; ``engraft/damage.py:107-118``
    uses 2, the context of a trigram table)."""
    n = len(tokens)
    offset = 0
    first = True
    while offset < n:
        this_block = min(block, n - offset)
        start = offset if first else offset - overlap
        yield offset, tokens[start:offset + this_block]
        offset += this_block
        first = False


def compute_rows_delta(table, rows_global: np.ndarray, data: np.ndarray) -> dict:
    """``(dnorm, ratio, cos)`` of every overlay row against its true row
    (``engraft/damage.py:126-151``); the true rows come from the device
    gather."""
    true = _read_true_rows(table, np.asarray(rows_global).tolist())
    data = np.asarray(data, dtype=np.float32)
    diff = data.astype(np.float64) - true.astype(np.float64)
    dnorm = np.linalg.norm(diff, axis=1).astype(np.float32)
    norm_true = np.linalg.norm(true, axis=1).astype(np.float64)
    norm_ov = np.linalg.norm(data, axis=1).astype(np.float64)
    ratio = np.where(norm_true > 0, norm_ov / np.maximum(norm_true, 1e-30), np.nan).astype(np.float32)
    denom = norm_ov * norm_true
    dot = np.sum(data.astype(np.float64) * true.astype(np.float64), axis=1)
    cos = np.where(denom > 0, dot / np.maximum(denom, 1e-30), np.nan).astype(np.float32)
    return {"rows_global": np.asarray(rows_global, dtype=np.int32), "dnorm": dnorm, "ratio": ratio, "cos": cos,
            "true": true}


_FILL_POOL = None


def _pieces(n: int) -> list[tuple[int, int]]:
    """``[a, b)`` ranges of an n-token block: a quarter of a million tokens first,
    so that the first piece is soon on its way to the device, a million once
    the copies, the transfers and the scans run side by side."""
    out, a, size = [], 0, 1 << 18
    while a < n:
        b = min(a + size, n)
        out.append((a, b))
        size = min(2 * size, 1 << 20) if len(out) > 1 else size
        a = b
    return out


def _fill(dst: np.ndarray, src: np.ndarray, pieces: list[tuple[int, int]]):
    """Futures of ``dst[a:b] = src[a:b]`` (converting to dst's type) for every
    piece, in order, over four threads: numpy's copy releases the GIL, and one
    thread moves an 8M-token block at well under the host's memory bandwidth."""
    global _FILL_POOL
    if _FILL_POOL is None:
        from concurrent.futures import ThreadPoolExecutor
        _FILL_POOL = ThreadPoolExecutor(4, thread_name_prefix="eg-fill")
    return [_FILL_POOL.submit(np.copyto, dst[a:b], src[a:b], casting="unsafe") for a, b in pieces]


def scan_hits(tokens: np.ndarray, table, overlay_sorted: np.ndarray, dnorm_sorted: np.ndarray,
              block: int = BLOCK_TOKENS) -> dict:
    """Positions of ``tokens`` that read at least one row of the sorted overlay
    ids (``engraft/damage.py:159-224``): ``pos`` / ``n_hit_rows`` /
    ``dnorm_max`` / ``dnorm_sum`` per hit position (the corpus's last
    position excluded), and ``read_count`` per overlay row."""
    tokens = np.asarray(tokens).reshape(-1)
    n = int(tokens.shape[0])
    dev = table.device
    ov = np.asarray(overlay_sorted, dtype=np.int64).reshape(-1)
    n_ov = int(ov.shape[0])
    if n_ov > 1 and np.any(ov[1:] <= ov[:-1]):
        raise ValueError("scan_hits: overlay_sorted must be strictly ascending")
    if n_ov and (ov[0] < 0 or ov[-1] > np.iinfo(np.int32).max):
        raise ValueError("scan_hits: overlay ids must be global rows in [0, 2^31)")
    dnorm = np.asarray(dnorm_sorted, dtype=np.float32).reshape(-1)
    if dnorm.shape[0] != n_ov:
        raise ValueError("scan_hits: dnorm_sorted must match overlay_sorted")
    hist = table.ngram_size - 1
    if block < max(hist, 1):
        # a later block's history would start before the corpus (the
        # reference's loop reads a wrapped-around slice there)
        raise ValueError(f"scan_hits: block ({block}) must be at least the n-gram history ({hist})")
    t0 = time.time()
    spec = table.c_spec
    # int32 token arrays (a tokenized corpus file) go to the device as they are
    # (4 bytes a token); any other integer type as int64.  A block is cut into
    # pieces: threads copy them into pinned memory, a second stream takes each
    # across PCIe when it is there, and the main stream scans it when it has
    # arrived, so that copies, transfers and scans overlap within a block as the
    # blocks do (a scan of one 8M-token block and its caller's result arrays 4.4 ms
    # one after the other, 3.4 ms so).
    narrow = tokens.dtype == np.int32
    tdt = torch.int32 if narrow else torch.int64
    main = torch.cuda.current_stream(dev)
    upload_stream = torch.cuda.Stream(device=dev)
    blocks = list(iter_blocks(tokens, block=block, overlap=hist)) if n_ov else []
    # two pinned host buffers (torch's host allocator keeps them for the next
    # call): one is filled while the other's copies to the device are in flight
    cap = max((len(b) for _, b in blocks), default=0)
    staging = [torch.empty(max(cap, 1), dtype=tdt, pin_memory=True) for _ in range(min(2, len(blocks)))]
    copied = [None, None]  # the last copy out of each pinned buffer

    def start_fill(j):
        blk = blocks[j][1]
        if copied[j % 2] is not None:
            copied[j % 2].synchronize()  # that buffer's previous block has left it
        host = staging[j % 2][:len(blk)]
        pieces = _pieces(len(blk))
        return host, pieces, _fill(host.numpy(), blk, pieces)

    filling = start_fill(0) if blocks else None
    try:
        # while the first pieces are copied: the overlay's arrays, and the membership bitmap over the
        # table's rows (almost every lookup is a miss, settled by one bit instead of the binary search)
        ids = torch.as_tensor(ov.astype(np.int32), device=dev)
        dn = torch.as_tensor(dnorm, device=dev)
        counts = torch.zeros(max(n_ov, 1), dtype=torch.int64, device=dev)
        n_bits = max(int(table.n_rows), 1)
        bitmap = torch.empty(int(_lib.load().eg_id_bitmap_words(n_bits)), dtype=torch.int32, device=dev)
        if n_ov:
            _lib.call("eg_build_id_bitmap", _lib.ptr(ids), n_ov, _lib.ptr(bitmap), n_bits, _lib.stream_ptr(dev))
        parts = []  # per block with hits: their positions and [3, hits] results
        for i, (offset, blk) in enumerate(blocks):
            host, pieces, fills = filling
            with torch.cuda.stream(upload_stream):
                tok = torch.empty(len(blk), dtype=tdt, device=dev)
            tok.record_stream(main)  # allocated on the upload stream, read on this one
            start_local = 0 if offset == 0 else hist
            m, size = tok.numel() - start_local, tok.element_size()
            # one fused launch a piece: hash, membership, per-position reductions, read counts;
            # n_hit / dnorm_max / dnorm_sum land in the rows of one [3, m] buffer so the hits leave
            # the device in one gather.  A piece's positions read the hist tokens before it.
            out = torch.empty((3, max(m, 0)), dtype=torch.int32, device=dev)
            for (a, b), done in zip(pieces, fills):
                done.result()
                with torch.cuda.stream(upload_stream):
                    tok[a:b].copy_(host[a:b], non_blocking=True)
                    ready = upload_stream.record_event()
                copied[i % 2] = ready
                first = max(a, start_local)  # the piece's first position
                if b <= first:
                    continue
                main.wait_event(ready)
                back = min(first, hist)
                o = _lib.ptr(out) + 4 * (first - start_local)
                _lib.call("eg_scan_overlay", ctypes.byref(spec), _lib.ptr(tok) + size * (first - back), size,
                          b - first + back, back, _lib.ptr(ids), n_ov, _lib.ptr(bitmap), n_bits, _lib.ptr(dn), o,
                          o + 4 * m, o + 8 * m, _lib.ptr(counts), _lib.stream_ptr(dev))
            filling = start_fill(i + 1) if i + 1 < len(blocks) else None  # while the scans run
            lim = min(m, n - 1 - offset)  # the corpus's last position is not a hit
            if lim <= 0:
                continue
            hit_local = torch.nonzero(out[0, :lim] > 0).reshape(-1)
            if hit_local.numel():
                parts.append(((hit_local + offset).cpu().numpy(), out[:, hit_local].cpu().numpy()))
    finally:
        if filling is not None:  # an error above: no thread may write into the buffers once they are let go
            wait(filling[2])
    # through pinned memory: the copy to pageable memory took as long as the scan
    counted = torch.empty(n_ov, dtype=torch.int64, pin_memory=True).copy_(counts[:n_ov]) if n_ov else counts[:0].cpu()
    read_count = counted.numpy().copy()
    dt = time.time() - t0

    def _cat(parts, dtype):
        return np.concatenate(parts) if len(parts) > 1 else parts[0] if parts else np.zeros(0, dtype=dtype)

    return {"pos": _cat([p for p, _ in parts], np.int64), "n_hit_rows": _cat([v[0] for _, v in parts], np.int32),
            "dnorm_max": _cat([v[1].view(np.float32) for _, v in parts], np.float32),
            "dnorm_sum": _cat([v[2].view(np.float32) for _, v in parts], np.float32),
            "read_count": read_count, "scan_time_s": dt, "n_tokens": n}
