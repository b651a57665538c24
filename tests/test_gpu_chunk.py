"""Calls of many rows per request (csrc/chunk.hip) against the CPU oracle: both
head dims, page sizes and modes, with and without means and rotations, row
counts at the edges of its 32-row waves and 256-row tiles, requests without
history or rows, several history splits, and value and output rows that are
only 2-byte aligned.  Bars and rounding as in test_gpu_multirow.py."""

from __future__ import annotations

import numpy as np
import pytest
import torch

import residualquant_amd as rq

from .cases import OURO_G16, OURO_G32, make_decode
from .test_gpu_multirow import ADJACENT_G16, ADJACENT_G32, MAX_ABS, MEAN_ABS, _bf16, _oracle, _run

pytestmark = pytest.mark.gpu

CASES = [
    # lengths (incl. the new rows), rows per request, heads, records, page tokens, mean, rotation, dim, mode
    ([900, 65], [48, 48], 2, OURO_G32, 16, True, True, 128, "anchor"),
    ([257], [257], 2, OURO_G32, 32, False, True, 128, "anchor"),             # no history, two tiles
    ([1300, 300], [256, 33], 2, OURO_G16, 16, True, False, 128, "anchor"),   # no rotation
    ([140, 700, 90], [130, 97, 0], 3, OURO_G32, 32, True, True, 96, "anchor"),
    ([2100], [64], 1, ((2, 16), (4, 16), (2, 32), (4, 32)), 16, False, True, 96, "anchor"),  # eight splits
    ([600, 129], [100, 64], 2, ADJACENT_G32, 16, True, True, 128, "adjacent"),
    ([333], [289], 2, ADJACENT_G16, 32, False, False, 96, "adjacent"),
    # row tiles of many depths, at the edges of 32 rows; the most requests
    ([9, 40, 31, 90, 33, 200, 65, 420, 70, 96, 300], [0, 1, 31, 32, 33, 64, 65, 300, 0, 96, 129], 3, OURO_G32, 16, True,
     True, 128, "anchor"),
    ([60 + i for i in range(64)], [48] * 63 + [49], 1, OURO_G32, 16, True, True, 128, "anchor"),
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: f"n{sum(c[1])}-d{c[7]}-pt{c[4]}-{c[8]}")
@pytest.mark.parametrize("causal", [True, False], ids=["prefill", "decode"])
def test_chunk_matches_oracle(oracle, device, case, causal):
    lengths, rows, heads, records, pt, mean, rotation, dim, mode = case
    print(f"[case] chunk causal={causal} {case}", flush=True)
    d = make_decode(lengths, heads, dim, records, seed=sum(lengths) + len(rows), page_tokens=pt, mean=mean,
                    rotation=rotation, rows_per_request=rows, mode=mode, anchor=0 if mode == "adjacent" else None)
    cache_np = d.group.oracle_cache(oracle)
    cache = torch.from_numpy(cache_np).to(device)
    for loop in range(len(records)):
        expected = _bf16(_oracle(oracle, d, cache_np, loop, causal))
        err = np.abs(_run(d, device, cache, loop, causal) - expected)
        print(f"[case]   loop {loop}: max {err.max():.3g} mean {err.mean():.3g}", flush=True)
        # Both sides are BF16, so values that round apart differ by an ulp (at
        # most 2^-7 of the value), which exceeds the bar from 4 up: a chunk's
        # first rows average few values.
        bar = np.maximum(MAX_ABS, np.abs(expected) * 2.0 ** -7)
        assert (err <= bar).all() and err.mean() <= MEAN_ABS, (loop, err.max(), err.mean())


def test_chunk_unaligned_rows(device):
    """Value and output views that start on an odd element, padded token
    strides and a workspace of any content: the bytes of the plain call."""
    d = make_decode([500, 210], 2, 128, OURO_G32, seed=3, rows_per_request=[130, 60])
    g = d.group
    cache = torch.zeros(g.cache_shape, dtype=torch.uint8, device=device)
    kr, vr, km = g.device_args(device)
    rq.quantize([(a.to(device), b.to(device)) for a, b in g.pairs], cache, g.slots.to(device), kr, vr, km, g.records,
                g.mode, g.anchor, g.coefficient)
    starts, lens, table = (t.to(device) for t in (d.query_start_loc, d.seq_lens, d.table))

    def padded(t, offset, pad):
        rows, heads, dim = t.shape
        flat = torch.zeros(offset + rows * (heads * dim + pad), dtype=t.dtype, device=device)
        view = flat[offset:].as_strided((rows, heads, dim), (heads * dim + pad, dim, 1))
        return view.copy_(t.to(device))

    for causal in (True, False):
        call = rq.packed_prefill_attention if causal else rq.attention
        for loop in (0, 3):
            plain = torch.empty_like(d.query, device=device)
            call(d.query.to(device), d.key.to(device), d.value.to(device), cache, plain, starts, lens, table, kr, vr,
                 km, g.records, g.mode, g.anchor, loop)
            out = padded(torch.full_like(d.query, float("nan")), 1, 3)
            size = rq.ops.attention_workspace_bytes(d.query.size(0), 2, 128, table.size(1), 16)
            workspace = torch.full((size,), 0xFF, dtype=torch.uint8, device=device)
            call(padded(d.query, 4, 4), padded(d.key, 4, 12), padded(d.value, 1, 5), cache, out, starts, lens, table,
                 kr, vr, km, g.records, g.mode, g.anchor, loop, workspace=workspace)
            assert torch.equal(out.contiguous().view(torch.int16), plain.view(torch.int16)), (causal, loop)
