"""Calls whose work is planned on the device from the request lengths
(csrc/rq_plan.h), one row per request and several: requests of very different lengths, several rows of one
request among single ones, requests without rows, more requests than one
64-lane register set or than the plan covers, against the FP64 oracle with
the attention bars."""

from __future__ import annotations

import numpy as np
import pytest
import torch

import residualquant_amd as rq

from .cases import OURO_G32, make_decode, oracle_attention
from .test_gpu_multirow import _bf16, _oracle, _run

pytestmark = pytest.mark.gpu

MAX_ABS, MEAN_ABS = 2e-2, 1e-3
ADJACENT = ((4, 32), (2, 32), (2, 32), (2, 32))

CASES = [
    # lengths, rows per request, heads, dim, page tokens, mode, split target (0: default)
    ([4097, 1, 257, 258, 33], None, 2, 128, 16, "anchor", 0),
    ([2900, 513, 2, 1030], [1, 3, 0, 1], 2, 128, 32, "anchor", 0),
    ([1700, 300, 16, 17], None, 3, 96, 16, "anchor", 64),
    ([2600, 1, 600], None, 2, 128, 16, "adjacent", 0),
    ([2100, 2050, 2090], None, 2, 96, 32, "adjacent", 0),   # near-equal chains: as many splits as fit
    ([34] * 58, None, 9, 96, 16, "adjacent", 0),            # 522 of them: more than two per compute unit
    ([1400] + [3] * 64 + [700], None, 1, 128, 16, "anchor", 9),
    ([600] + [2, 35] * 130, None, 1, 128, 16, "anchor", 600),
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: f"{len(c[0])}x{c[0][0]}-d{c[3]}-pt{c[4]}-{c[5]}-t{c[6]}")
def test_planned_decode_matches_oracle(oracle, device, case):
    print(f"[case] planned decode {str(case)[:120]}", flush=True)
    lengths, rows, heads, dim, pt, mode, target = case
    records = ADJACENT if mode == "adjacent" else OURO_G32
    d = make_decode(lengths, heads, dim, records, seed=len(lengths) + dim, page_tokens=pt, mode=mode,
                    anchor=0 if mode == "adjacent" else 3, rows_per_request=rows)
    g = d.group
    cache_np = g.oracle_cache(oracle)
    cache = torch.from_numpy(cache_np).to(device)
    kr, vr, km = g.device_args(device)
    q, k, v = (t.to(device) for t in (d.query, d.key, d.value))
    starts, lens, table = (t.to(device) for t in (d.query_start_loc, d.seq_lens, d.table))
    # The arrival words of split rows lie in a workspace of any content.
    size = rq.ops.attention_workspace_bytes(q.size(0), heads, dim, table.size(1), pt)
    workspace = torch.full((size,), 0xFF, dtype=torch.uint8, device=device)
    try:
        rq.ops.set_split_target(target)
        for loop in (0, 1, 3):
            out = torch.full_like(q, float("nan"))
            for _ in range(2):  # the second call finds the words as the first left them
                rq.attention(q, k, v, cache, out, starts, lens, table, kr, vr, km, g.records, g.mode, g.anchor, loop,
                             workspace=workspace)
            expected = oracle_attention(oracle, d, cache_np, loop)
            err = np.abs(out.float().cpu().numpy() - expected)
            print(f"[case]   loop {loop}: max {err.max():.3g} mean {err.mean():.3g}", flush=True)
            # Histories of a token or two leave outputs near 1 in magnitude,
            # whose BF16 rounding alone averages up to 2^-9 of them (a quarter
            # of an ulp, the ulp at most 2^-7 of the value).
            bar = MEAN_ABS + np.abs(expected).mean() * 2.0 ** -9
            assert err.max() <= MAX_ABS and err.mean() <= bar, (loop, err.max(), err.mean(), bar)
    finally:
        rq.ops.set_split_target(0)


MULTIROW_CASES = [
    # lengths (incl. the new rows), rows per request, heads, dim, page tokens, mode
    ([2500, 40, 300, 9, 700], [3, 2, 20, 4, 0], 16, 128, 16, "anchor"),
    ([1900, 400, 150], [40, 3, 70], 3, 96, 32, "anchor"),
    ([1300, 70], [4, 2], 16, 128, 16, "adjacent"),
    ([40] * 64 + [900], [2] * 65, 1, 128, 16, "anchor"),  # more requests than the plan covers
    # near-equal requests: whole (10 tiles), split (22 tiles; chains from 8 tiles)
    ([310, 300, 318], [20, 20, 20], 2, 128, 16, "anchor"),
    ([700, 690], [20, 20], 2, 96, 32, "anchor"),
    ([262, 262], [3, 3], 2, 128, 16, "adjacent"),
]


@pytest.mark.parametrize("case", MULTIROW_CASES, ids=lambda c: f"{len(c[0])}x{c[0][0]}-d{c[3]}-pt{c[4]}-{c[5]}")
@pytest.mark.parametrize("causal", [True, False], ids=["prefill", "decode"])
def test_planned_multirow_matches_oracle(oracle, device, case, causal):
    print(f"[case] planned multirow causal={causal} {str(case)[:120]}", flush=True)
    lengths, rows, heads, dim, pt, mode = case
    records = ADJACENT if mode == "adjacent" else OURO_G32
    d = make_decode(lengths, heads, dim, records, seed=len(lengths) + dim, page_tokens=pt, mode=mode,
                    anchor=0 if mode == "adjacent" else 3, rows_per_request=rows)
    cache_np = d.group.oracle_cache(oracle)
    cache = torch.from_numpy(cache_np).to(device)
    for loop in (1, 3):
        err = np.abs(_run(d, device, cache, loop, causal) - _bf16(_oracle(oracle, d, cache_np, loop, causal)))
        print(f"[case]   loop {loop}: max {err.max():.3g} mean {err.mean():.3g}", flush=True)
        assert err.max() <= MAX_ABS and err.mean() <= MEAN_ABS, (loop, err.max(), err.mean())


def test_planned_decode_replays(device):
    """A captured call repeats its tag: every replay, with other lengths in
    place of the captured ones, equals the eager call."""
    d = make_decode([3000, 400, 50], 2, 128, OURO_G32, seed=5)
    g = d.group
    cache = torch.zeros(g.cache_shape, dtype=torch.uint8, device=device)
    kr, vr, km = g.device_args(device)
    rq.quantize([(a.to(device), b.to(device)) for a, b in g.pairs], cache, g.slots.to(device), kr, vr, km, g.records,
                g.mode, g.anchor, g.coefficient)
    q, k, v = (t.to(device) for t in (d.query, d.key, d.value))
    starts, lens, table = (t.to(device) for t in (d.query_start_loc, d.seq_lens, d.table))
    out, want = torch.empty_like(q), torch.empty_like(q)

    def call(to):
        rq.attention(q, k, v, cache, to, starts, lens, table, kr, vr, km, g.records, g.mode, g.anchor, 1)

    call(out)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        call(out)
    for lengths in ([3000, 400, 50], [257, 400, 50], [2800, 1, 33], [3000, 399, 2]):
        lens.copy_(torch.tensor(lengths, dtype=torch.int32))
        call(want)
        for _ in range(3):
            out.fill_(float("nan"))
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(out.view(torch.int16), want.view(torch.int16)), lengths


@pytest.mark.parametrize("rows", [[3, 5, 2], [60, 50, 40]], ids=["rows", "chunks"])
def test_captured_rows_replay(device, rows):
    """Several rows per request, captured: every replay, with other lengths in
    place of the captured ones, equals the eager call."""
    d = make_decode([2800, 400, 130], 2, 128, OURO_G32, seed=6, rows_per_request=rows)
    g = d.group
    cache = torch.zeros(g.cache_shape, dtype=torch.uint8, device=device)
    kr, vr, km = g.device_args(device)
    rq.quantize([(a.to(device), b.to(device)) for a, b in g.pairs], cache, g.slots.to(device), kr, vr, km, g.records,
                g.mode, g.anchor, g.coefficient)
    q, k, v = (t.to(device) for t in (d.query, d.key, d.value))
    starts, lens, table = (t.to(device) for t in (d.query_start_loc, d.seq_lens, d.table))
    out, want = torch.empty_like(q), torch.empty_like(q)

    def call(to):
        rq.packed_prefill_attention(q, k, v, cache, to, starts, lens, table, kr, vr, km, g.records, g.mode, g.anchor, 1)

    call(out)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        call(out)
    captured = lens.tolist()
    for lengths in (captured, [700, captured[1], rows[2]], [captured[0], rows[1] + 1, captured[2]]):
        lens.copy_(torch.tensor(lengths, dtype=torch.int32))
        call(want)
        for _ in range(3):
            out.fill_(float("nan"))
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(out.view(torch.int16), want.view(torch.int16)), lengths


@pytest.mark.parametrize("lengths,rows,mode", [([3000, 700, 90], None, "anchor"), ([2600, 1, 600], None, "adjacent"),
                                               ([4000, 300, 600], [3, 20, 4], "anchor"),
                                               ([3000, 400, 700], [300, 50, 110], "anchor"),
                                               ([90] * 70, [2] * 70, "anchor")],
                         ids=["decode", "adjacent", "rows", "chunk", "past-the-plan"])
def test_workspace_of_the_required_size(oracle, device, lengths, rows, mode):
    """The smallest workspace that a call takes, at any address: right results,
    nothing written around it."""
    print(f"[case] required workspace {lengths[:3]} {rows and rows[:3]} {mode}", flush=True)
    d = make_decode(lengths, 2, 128, ADJACENT if mode == "adjacent" else OURO_G32, seed=8, mode=mode,
                    anchor=0 if mode == "adjacent" else 3, rows_per_request=rows)
    g = d.group
    cache_np = g.oracle_cache(oracle)
    cache = torch.from_numpy(cache_np).to(device)
    kr, vr, km = g.device_args(device)
    q, k, v = (t.to(device) for t in (d.query, d.key, d.value))
    starts, lens, table = (t.to(device) for t in (d.query_start_loc, d.seq_lens, d.table))
    out = torch.full_like(q, float("nan"))

    def call(workspace):
        rq.attention(q, k, v, cache, out, starts, lens, table, kr, vr, km, g.records, g.mode, g.anchor, 1,
                     workspace=workspace)

    with pytest.raises(RuntimeError, match=r"Attention workspace of \d+ bytes required") as refused:
        call(torch.empty(16, dtype=torch.uint8, device=device))
    required = int(str(refused.value).split("workspace of ")[1].split()[0])
    full = rq.ops.attention_workspace_bytes(q.size(0), 2, 128, table.size(1), 16)
    assert required < full if rows and max(rows) > 100 else required <= full
    with pytest.raises(RuntimeError, match="Attention workspace"):
        call(torch.empty(required - 1, dtype=torch.uint8, device=device))
    buffer = torch.full((required + 65536,), 0xA5, dtype=torch.uint8, device=device)
    want = _bf16(_oracle(oracle, d, cache_np, 1, False))
    for offset in (0, 0, 4, 264, 4097, 31):
        print(f"[case]   workspace at + {offset}", flush=True)
        out.fill_(float("nan"))
        buffer.fill_(0xA5)
        call(buffer[offset:offset + required])
        err = np.abs(out.float().cpu().numpy() - want)
        bar = MEAN_ABS + np.abs(want).mean() * 2.0 ** -9  # (as in test_planned_decode_matches_oracle)
        assert err.max() <= MAX_ABS and err.mean() <= bar, (err.max(), err.mean())
        assert bool((buffer[:offset] == 0xA5).all()) and bool((buffer[offset + required:] == 0xA5).all())
