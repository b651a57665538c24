"""The work that programs built on this package have it do, as cases that can be timed and compared.

Five kinds, each through the package's public entry points:

- ``decode``: one layer's attention calls of every loop, one new token per
  request, over the packed cache (``attention``);
- ``rows``: the same for several new rows per request, either draft rows to
  verify (``attention``) or a prompt chunk over a packed prefix
  (``packed_prefill_attention``, causal among the new rows);
- ``prompt``: full prompts over their raw K/V (``flash_attn_varlen_func``);
- ``write``: quantize-on-write of one loop group (``quantize``);
- ``step``: a decode step of a whole looped model, replayed from its graph
  (``LoopedDecoder``).

``exact`` restates each in float64 torch: the page format, the BF16 restore
of the values, the unrounded keys, the softmax and the rotations.
"""

from __future__ import annotations

import math
import random

import torch

from residualquant_amd import (attention, flash_attn_varlen_func, packed_prefill_attention, page_width, quantize,
                               workloads)
from residualquant_amd.layout import staged_bytes
from residualquant_amd.looped_decode import LoopedConfig, LoopedDecoder

DEVICE = torch.device("cuda:0")
LOOPS = 4
WRITE_CHUNK = 16384  # history tokens quantized per call while a cache is filled


def listed():
    return [
        # One user's next token on a short conversation: launches and latency.
        {"name": "decode_single", "kind": "decode", "batch": 1, "shortest": 2047, "longest": 2047, "mix": 0,
         "heads": 16, "dim": 128, "group": 32, "page": 16, "mode": "anchor", "mean": False},
        # The headline batch: 32 requests of 8192 tokens at the Ouro geometry.
        {"name": "decode_batch", "kind": "decode", "batch": 32, "shortest": 8192, "longest": 8192, "mix": 0,
         "heads": 16, "dim": 128, "group": 32, "page": 16, "mode": "anchor", "mean": False},
        # A serving batch as it really is: conversations of very different lengths, calibrated key means.
        {"name": "decode_mixed", "kind": "decode", "batch": 32, "shortest": 61, "longest": 8000, "mix": 1,
         "heads": 16, "dim": 128, "group": 32, "page": 32, "mode": "anchor", "mean": True},
        # The Huginn geometry: 55 heads of 96 channels, groups of 16, ragged lengths.
        {"name": "decode_huginn", "kind": "decode", "batch": 8, "shortest": 1001, "longest": 4096, "mix": 2,
         "heads": 55, "dim": 96, "group": 16, "page": 16, "mode": "anchor", "mean": False},
        # Records chained from loop to loop instead of against one anchor.
        {"name": "decode_adjacent", "kind": "decode", "batch": 8, "shortest": 500, "longest": 4096, "mix": 3,
         "heads": 16, "dim": 128, "group": 32, "page": 16, "mode": "adjacent", "mean": False},
        # Four draft rows per request verified in one call.
        {"name": "rows_verify", "kind": "rows", "causal": False, "rows": 4, "batch": 16, "shortest": 700,
         "longest": 8192, "mix": 4, "heads": 16, "dim": 128, "group": 32, "page": 16, "mode": "anchor",
         "mean": False},
        # The next chunk of two long prompts over their packed prefixes.
        {"name": "rows_chunk", "kind": "rows", "causal": True, "rows": 509, "batch": 2, "shortest": 2000,
         "longest": 6000, "mix": 5, "heads": 16, "dim": 128, "group": 32, "page": 16, "mode": "anchor",
         "mean": False},
        # One long prompt.
        {"name": "prompt_long", "kind": "prompt", "batch": 1, "shortest": 4096, "longest": 4096, "mix": 0,
         "heads": 16, "dim": 128},
        # A prefill batch of chat prompts.
        {"name": "prompt_mixed", "kind": "prompt", "batch": 12, "shortest": 17, "longest": 1500, "mix": 6,
         "heads": 16, "dim": 128},
        # The records of a whole prompt written at once.
        {"name": "write_prompt", "kind": "write", "tokens": 4096, "heads": 16, "dim": 128, "group": 32, "page": 16,
         "mode": "anchor", "mean": False, "coefficient": "ls"},
        # The records of one decode step's new tokens.
        {"name": "write_step", "kind": "write", "tokens": 32, "heads": 16, "dim": 128, "group": 32, "page": 16,
         "mode": "anchor", "mean": False, "coefficient": "ls"},
        # A looped model's decode step, graph replay: Ouro widths, one physical
        # layer (four layer passes; more of them amplify one rounding's
        # difference past any useful tolerance on the logits).
        {"name": "step_model", "kind": "step", "batch": 4, "context": 2048, "layers": 1},
    ]


def _log_uniform(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "rows", "rows", "prompt", "write", "step"])
    if kind == "step":
        return {"kind": kind, "batch": rng.randint(1, 16), "context": _log_uniform(rng, 256, 3000), "layers": 1}
    heads, dim = rng.choice([(16, 128), (16, 128), (55, 96)])
    geometry = {"heads": heads, "dim": dim}
    mix = rng.randrange(1 << 20)
    if kind == "prompt":
        longest = _log_uniform(rng, 40, 4096 if heads == 16 else 2048)
        batch = rng.randint(1, max(1, min(24, 4096 // longest)))
        return {"kind": kind, "batch": batch, "shortest": rng.randint(1, longest), "longest": longest, "mix": mix,
                **geometry}
    packed = {"group": rng.choice([16, 32]), "page": rng.choice([16, 32]),
              "mode": rng.choice(["anchor", "anchor", "adjacent"])}
    packed["mean"] = packed["mode"] == "anchor" and rng.random() < 0.5
    if kind == "write":
        return {"kind": kind, "tokens": _log_uniform(rng, 1, 4096 if heads == 16 else 1200), **geometry, **packed,
                "coefficient": rng.choice(["ls", "ls", "norm", "unit"])}
    longest = _log_uniform(rng, 128, 8192)
    most = max(1, (80_000 if heads == 16 else 30_000) // longest)  # history tokens of the whole batch
    case = {"kind": kind, "batch": min(most, _log_uniform(rng, 1, 48)), "shortest": rng.randint(1, longest),
            "longest": longest, "mix": mix, **geometry, **packed}
    if kind == "rows":
        case["causal"] = rng.random() < 0.6
        case["rows"] = _log_uniform(rng, 16, 768) if case["causal"] else _log_uniform(rng, 2, 16)
        case["batch"] = max(1, min(case["batch"], (1024 if heads == 16 else 384) // case["rows"]))
    return case


def _lengths(case):
    """History (or prompt) tokens per request: log-uniform, the longest among them."""
    rng = random.Random(case["mix"])
    lengths = [_log_uniform(rng, case["shortest"], case["longest"]) for _ in range(case["batch"])]
    lengths[rng.randrange(case["batch"])] = case["longest"]
    return lengths


def _records(case):
    """Three INT2 residual records and the INT4 anchor, which is first in adjacent mode."""
    residual, anchor = (2, case["group"]), (4, 32)
    if case["mode"] == "adjacent":
        return (anchor, residual, residual, residual), 0
    return (residual, residual, residual, anchor), LOOPS - 1


def _rotations(case, seed):
    return (workloads.random_sign_rotation(case["heads"], case["dim"], seed + 1, device=DEVICE),
            workloads.random_sign_rotation(case["heads"], case["dim"], seed + 2, device=DEVICE))


# ---------------------------------------------------------------- prepare


def _prepare_packed(case, seed):
    heads, dim, page = case["heads"], case["dim"], case["page"]
    records, anchor = _records(case)
    lengths = _lengths(case)
    rows = case.get("rows", 1)
    causal = case.get("causal", False)
    # Rows of a chunk are the request's last tokens; every other row counts itself alone.
    seq_lens = [n + (rows if causal else 1) for n in lengths]
    pages = (max(seq_lens) + page - 1) // page
    table = workloads.block_tables(case["batch"], pages, seed + 3, device=DEVICE)
    cache = torch.zeros((2, case["batch"] * pages, heads, page, page_width(dim, records)), dtype=torch.uint8,
                        device=DEVICE)
    key_rotation, value_rotation = _rotations(case, seed)
    mean = workloads.key_means(LOOPS, heads, dim, seed + 4, device=DEVICE) if case["mean"] else None
    slots = workloads.history_slots(table, lengths, page)
    for start in range(0, slots.numel(), WRITE_CHUNK):
        part = slots[start:start + WRITE_CHUNK]
        pairs = workloads.loop_kv(part.numel(), heads, dim, LOOPS, seed + 5 + start, device=DEVICE,
                                  anchor_index=anchor)
        quantize(pairs, cache, part, key_rotation, value_rotation, mean, records, case["mode"], anchor, "ls")
    generator = torch.Generator(device=DEVICE).manual_seed(seed)
    total = case["batch"] * rows
    shape = (total, heads, dim)
    query = torch.randn(shape, generator=generator, device=DEVICE).to(torch.bfloat16)
    live = workloads.loop_kv(total, heads, dim, LOOPS, seed + 6, device=DEVICE, anchor_index=anchor)
    return {
        "case": case, "records": records, "anchor": anchor, "query": query, "live": live, "cache": cache,
        "table": table, "outputs": [torch.empty(shape, dtype=torch.bfloat16, device=DEVICE) for _ in range(LOOPS)],
        "starts": torch.arange(0, total + 1, rows, dtype=torch.int32, device=DEVICE),
        "seq_lens": torch.tensor(seq_lens, dtype=torch.int32, device=DEVICE),
        "key_rotation": key_rotation, "value_rotation": value_rotation, "mean": mean, "lengths": lengths,
    }


def _prepare_prompt(case, seed):
    lengths = _lengths(case)
    generator = torch.Generator(device=DEVICE).manual_seed(seed)
    shape = (sum(lengths), case["heads"], case["dim"])
    query, key, value = (torch.randn(shape, generator=generator, device=DEVICE).to(torch.bfloat16) for _ in range(3))
    starts = [0]
    for n in lengths:
        starts.append(starts[-1] + n)
    return {"case": case, "query": query, "key": key, "value": value, "lengths": lengths,
            "output": torch.empty_like(query),
            "starts": torch.tensor(starts, dtype=torch.int32, device=DEVICE)}


def _prepare_write(case, seed):
    heads, dim, page, tokens = case["heads"], case["dim"], case["page"], case["tokens"]
    records, anchor = _records(case)
    blocks = (tokens + page - 1) // page + 32
    key_rotation, value_rotation = _rotations(case, seed)
    generator = torch.Generator().manual_seed(seed)
    slots = torch.randperm(blocks * page, generator=generator)[:tokens]
    if tokens > 1024:  # a prompt fills its pages in order
        slots = workloads.history_slots(workloads.block_tables(1, blocks, seed), [tokens], page)
    return {"case": case, "records": records, "anchor": anchor, "slots": slots.to(DEVICE),
            "pairs": workloads.loop_kv(tokens, heads, dim, LOOPS, seed + 5, device=DEVICE, anchor_index=anchor),
            "cache": torch.zeros((2, blocks, heads, page, page_width(dim, records)), dtype=torch.uint8,
                                 device=DEVICE),
            "key_rotation": key_rotation, "value_rotation": value_rotation,
            "mean": workloads.key_means(LOOPS, heads, dim, seed + 4, device=DEVICE) if case["mean"] else None}


NEW_TOKENS = 256


def _prepare_step(case, seed):
    decoder = LoopedDecoder(LoopedConfig(layers=case["layers"]), case["batch"], case["context"], NEW_TOKENS, DEVICE,
                            seed=seed)
    decoder.build_history(seed=seed)
    decoder.capture()
    generator = torch.Generator(device=DEVICE).manual_seed(seed + 8)
    tokens = torch.randint(0, decoder.config.vocab, (NEW_TOKENS, case["batch"]), generator=generator, device=DEVICE)
    return {"case": case, "decoder": decoder, "tokens": tokens}


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("decode", "rows"):
        return _prepare_packed(case, seed)
    return {"prompt": _prepare_prompt, "write": _prepare_write, "step": _prepare_step}[kind](case, seed)


# ---------------------------------------------------------------- run


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind in ("decode", "rows"):
        call = packed_prefill_attention if case.get("causal") else attention
        for loop in range(LOOPS):
            key, value = state["live"][loop]
            call(state["query"], key, value, state["cache"], state["outputs"][loop], state["starts"],
                 state["seq_lens"], state["table"], state["key_rotation"], state["value_rotation"], state["mean"],
                 state["records"], case["mode"], state["anchor"], loop)
        return state["outputs"]
    if kind == "prompt":
        longest = max(state["lengths"])
        return flash_attn_varlen_func(q=state["query"], k=state["key"], v=state["value"], out=state["output"],
                                      cu_seqlens_q=state["starts"], cu_seqlens_k=state["starts"],
                                      max_seqlen_q=longest, max_seqlen_k=longest,
                                      softmax_scale=case["dim"] ** -0.5, causal=True)
    if kind == "write":
        quantize(state["pairs"], state["cache"], state["slots"], state["key_rotation"], state["value_rotation"],
                 state["mean"], state["records"], case["mode"], state["anchor"], case["coefficient"])
        return state["cache"]
    # One token of a given continuation; a finished one starts over.
    decoder = state["decoder"]
    if decoder.next_position >= decoder.max_tokens:
        decoder.positions.fill_(decoder.context)
        decoder.seq_lens.fill_(decoder.context + 1)
        decoder.slots.copy_(decoder.block_table[:, decoder.context // decoder.config.page_tokens].long()
                            * decoder.config.page_tokens + decoder.context % decoder.config.page_tokens)
        decoder.next_position = decoder.context
    decoder.tokens.copy_(state["tokens"][decoder.next_position - decoder.context])
    return decoder.replay()


# ---------------------------------------------------------------- work


def work(case):
    kind = case["kind"]
    if kind == "step":
        c = LoopedConfig(layers=case["layers"])
        layer = c.hidden * (4 * c.heads * c.head_dim + 3 * c.intermediate)
        pages = case["context"] // c.page_tokens
        history = sum(2 * pages * c.heads * staged_bytes(c.head_dim, c.schedule, c.page_tokens, "anchor", c.anchor, r)
                      for r in range(c.loops))
        weights = c.layers * layer * c.loops + c.vocab * c.hidden
        return {"bytes": 2 * weights + case["batch"] * c.layers * history,
                "flops": 2 * case["batch"] * (weights + 2 * c.layers * c.loops * c.heads * c.head_dim * case["context"])}
    heads, dim = case["heads"], case["dim"]
    if kind == "write":
        records, _ = _records(case)
        tokens = case["tokens"]
        return {"bytes": tokens * heads * (2 * LOOPS * 2 * dim + 2 * page_width(dim, records)) + 4 * heads * dim * dim,
                "flops": 2 * 2 * LOOPS * tokens * heads * dim * dim}
    lengths = _lengths(case)
    if kind == "prompt":
        return {"bytes": 4 * 2 * sum(lengths) * heads * dim,
                "flops": sum(4 * dim * heads * n * (n + 1) // 2 for n in lengths)}
    records, anchor = _records(case)
    rows = case.get("rows", 1)
    history_bytes = sum(2 * heads * staged_bytes(dim, records, 1, case["mode"], anchor, loop) * sum(lengths)
                        for loop in range(LOOPS))
    live = rows * (rows + 1) // 2 if case.get("causal") else rows
    return {"bytes": history_bytes + LOOPS * 4 * 2 * case["batch"] * rows * heads * dim + LOOPS * 4 * heads * dim * dim,
            "flops": LOOPS * 4 * dim * heads * sum(rows * n + live for n in lengths)}


def tolerance(case):
    if case["kind"] == "write":
        return "exact"  # bytes
    # BF16 outputs and, in the matrix-core paths, BF16 probabilities (2e-3
    # against float64); a model's logits carry the rounding of its four layer
    # passes, which every softmax and norm after it amplifies (the projections
    # summed in another order: 0.012, and 0.08 at most).
    return {"rel": 0.03, "max": 0.4} if case["kind"] == "step" else {"rel": 8e-3, "max": 0.1}


# ---------------------------------------------------------------- exact


def _bf16(x):
    """Float64 values rounded once to BF16, ties to even."""
    _, exponent = torch.frexp(x)
    quantum = torch.ldexp(torch.ones_like(x), exponent.clamp(min=-125) - 8)
    return torch.round(x / quantum) * quantum


def _read_record(pages, dim, records, index):
    """(code x scale + offset [pages, heads, PT, D], alpha [pages, heads, PT, 1]) of pages [pages, heads, PT, width]."""
    count, heads, page, _ = pages.shape
    sizes = [(dim * bits // 8, dim // group) for bits, group in records]
    begin = page * sum(code + 2 * groups + 2 for code, groups in sizes[:index])
    (bits, group), (code, groups) = records[index], sizes[index]
    flat = pages.reshape(count, heads, -1)[..., begin:begin + page * (code + 2 * groups + 2)]
    codes, scale, offset, alpha = torch.split(flat, [page * code, page * groups, page * groups, page * 2], dim=-1)
    shifts = torch.arange(0, 8, bits, dtype=torch.uint8, device=pages.device)
    values = ((codes[..., None] >> shifts) & (2 ** bits - 1)).reshape(count, heads, page, groups, group).double()
    as_fp8 = lambda raw: raw.contiguous().view(torch.float8_e4m3fn).reshape(  # noqa: E731
        count, heads, page, groups, 1).to(torch.float32).double()
    restored = (values * as_fp8(scale) + as_fp8(offset)).reshape(count, heads, page, dim)
    return restored, alpha.contiguous().view(torch.bfloat16).reshape(count, heads, page, 1).double()


def _history(cache, blocks, length, dim, records, anchor, mode, loop, mean):
    """Float64 keys and values [heads, length, D] of a request's cached tokens."""
    key_pages, value_pages = cache[0, blocks], cache[1, blocks]
    per_head = lambda m: m.double()[None, :, None, :]  # noqa: E731
    key, _ = _read_record(key_pages, dim, records, anchor)
    value = _bf16(_read_record(value_pages, dim, records, anchor)[0])
    if mode == "adjacent" and loop > 0:
        key = _bf16(key)
        for link in range(1, loop + 1):
            for plane, pages in (("key", key_pages), ("value", value_pages)):
                step, alpha = _read_record(pages, dim, records, link)
                if plane == "key":
                    key = _bf16(alpha * key + _bf16(step))
                else:
                    value = _bf16(alpha * value + _bf16(step))
    elif loop != anchor:
        if mean is not None:
            key = key + per_head(mean[anchor].to(torch.bfloat16))
        step, alpha = _read_record(key_pages, dim, records, loop)
        key = alpha * key + step
        step, alpha = _read_record(value_pages, dim, records, loop)
        value = _bf16(alpha * value + _bf16(step))
    if mean is not None:
        key = key + per_head(mean[loop])
    heads = cache.size(2)
    return tuple(x.permute(1, 0, 2, 3).reshape(heads, -1, dim)[:, :length] for x in (key, value))


def _attend(query, key, value, keys, values, key_rotation, value_rotation, causal):
    """Float64 [rows, heads, D]: rows of one request over its history and their own new tokens."""
    rows, _, dim = query.shape
    q, k, v = (x.double().transpose(0, 1) for x in (query, key, value))
    rotated = torch.matmul(q, key_rotation.double()) / math.sqrt(dim)
    history = torch.matmul(rotated, keys.transpose(1, 2).contiguous())
    live = torch.matmul(q, k.transpose(1, 2).contiguous()) / math.sqrt(dim)
    index = torch.arange(rows, device=query.device)
    visible = index[None, :] <= index[:, None] if causal else index[None, :] == index[:, None]
    live = live.masked_fill(~visible, -math.inf)
    weights = torch.softmax(torch.cat((history, live), dim=-1), dim=-1)
    old, new = weights[..., :keys.size(1)], weights[..., keys.size(1):]
    out = torch.matmul(torch.matmul(old, values), value_rotation.double().transpose(1, 2).contiguous())
    return (out + torch.matmul(new, v)).transpose(0, 1)


def _exact_packed(case, seed):
    s = _prepare_packed(case, seed)
    rows = case.get("rows", 1)
    outputs = []
    for loop in range(LOOPS):
        key, value = s["live"][loop]
        parts = []
        for b, length in enumerate(s["lengths"]):
            blocks = s["table"][b, :(length + case["page"] - 1) // case["page"]].long()
            keys, values = _history(s["cache"], blocks, length, case["dim"], s["records"], s["anchor"], case["mode"],
                                    loop, s["mean"])
            at = slice(b * rows, (b + 1) * rows)
            parts.append(_attend(s["query"][at], key[at], value[at], keys, values, s["key_rotation"],
                                 s["value_rotation"], case.get("causal", False)))
        outputs.append(torch.cat(parts))
    return outputs


def _exact_prompt(case, seed):
    s = _prepare_prompt(case, seed)
    parts, start = [], 0
    for n in s["lengths"]:
        heads = []
        for head in range(case["heads"]):  # one head's scores at a time
            q, k, v = (x[start:start + n, head].double() for x in (s["query"], s["key"], s["value"]))
            scores = torch.matmul(q, k.t().contiguous()) * case["dim"] ** -0.5
            scores.masked_fill_(torch.ones_like(scores, dtype=torch.bool).triu_(1), -math.inf)
            heads.append(torch.matmul(torch.softmax(scores, dim=-1), v))
        parts.append(torch.stack(heads, dim=1))
        start += n
    return torch.cat(parts)


def _exact_step(case, seed):
    """The step's logits with no rounding between its operations."""
    s = _prepare_step(case, seed)
    d = s["decoder"]
    c = d.config
    batch, context = case["batch"], case["context"]

    def norm(x, weight):
        return x * torch.rsqrt(x.square().mean(dim=-1, keepdim=True) + c.rms_eps) * weight.double()

    def rope(x):
        low, high = x.chunk(2, dim=-1)
        cos, sin = d.cos[context].double(), d.sin[context].double()
        return torch.cat((low * cos - high * sin, high * cos + low * sin), dim=-1)

    blocks = [d.block_table[b, :(context + c.page_tokens - 1) // c.page_tokens].long() for b in range(batch)]
    hidden = d.embed[s["tokens"][0]].double()
    for loop in range(c.loops):
        residual = None
        for layer in range(c.layers):
            residual = hidden if residual is None else residual + hidden
            qkv = torch.matmul(norm(residual, d.norms[layer][0]), d.qkv[layer].double().t().contiguous())
            q, k, v = (x.reshape(batch, c.heads, c.head_dim) for x in qkv.chunk(3, dim=-1))
            q, k = rope(q), rope(k)
            rows = []
            for b in range(batch):
                keys, values = _history(d.caches[layer], blocks[b], context, c.head_dim, c.schedule, c.anchor,
                                        "anchor", loop, None)
                at = slice(b, b + 1)
                rows.append(_attend(q[at], k[at], v[at], keys, values, d.key_rotation[layer], d.value_rotation[layer],
                                    False))
            out = torch.matmul(torch.cat(rows).reshape(batch, -1), d.o[layer].double().t().contiguous())
            residual = residual + norm(out, d.norms[layer][1])
            mlp = torch.matmul(norm(residual, d.norms[layer][2]), d.gate_up[layer].double().t().contiguous())
            gate, up = mlp.chunk(2, dim=-1)
            out = torch.matmul(torch.nn.functional.silu(gate) * up, d.down[layer].double().t().contiguous())
            hidden = norm(out, d.norms[layer][3])
        hidden = norm(residual + hidden, d.final_norm)
    return torch.matmul(hidden, d.lm_head.double().t().contiguous())


def exact(case, seed):
    kind = case["kind"]
    if kind in ("decode", "rows"):
        return _exact_packed(case, seed)
    if kind == "write":
        return None  # bytes only
    return _exact_prompt(case, seed) if kind == "prompt" else _exact_step(case, seed)
