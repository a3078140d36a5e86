"""Performance cases of the link step: what one user's call costs.

Four kinds of call, each through a public entry point:

* ``operator``: the fused link operator on token maps that the caller holds,
  for one layer (``fused_kv_link_inplace``, how the reference's runtime calls
  it) or for every layer at once (``fused_kv_link_layers_inplace``);
* ``link``: a request's link (or a batch's) through the executor, from its
  link plan: preparation, link kernels and the write-back of the repaired
  rows;
* ``repair``: the repair pass's attention of one layer, with the plan that a
  program builds once per repair batch and keeps for every layer.

Sizes follow the workloads of ``legolink_amd.workloads`` (c1 to c5) and the
head shapes of the tests.  A case fixes everything that the amount of work
depends on (block lengths, spans, which blocks a batch shares); the seed
draws the slots, the positions and the values.
"""

from __future__ import annotations

import functools
import math
import sys
from pathlib import Path

import numpy as np
import torch

_PACKAGE = str(Path.cwd() / "sglang-legolink_amd")
if _PACKAGE not in sys.path:
    sys.path.insert(0, _PACKAGE)

from legolink_amd import kv_link  # noqa: E402
from legolink_amd.link_runtime import KVLinkExecutor, KVPool  # noqa: E402
from legolink_amd.registry import LegoLinkBlockRegistry  # noqa: E402
from legolink_amd.repair_attention import RepairAttentionPlan  # noqa: E402
from legolink_amd.rope import RotarySpec, build_cos_sin_cache  # noqa: E402

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32,
          "int32": torch.int32, "int64": torch.int64}


def _operator(**options):
    case = {"kind": "operator", "layers": 28, "tokens": 8192, "heads": 4, "key_dim": 128, "value_dim": 128,
            "rotary": 128, "kv": "bf16", "table": "fp32", "neox": True, "index": "int64", "mask": False, "prefix": 0}
    return {**case, **options}


def _link(**options):
    case = {"kind": "link", "requests": 1, "tokens": 32768, "blocks": 16, "catalogue": 0, "seam": 16,
            "layers": 28, "heads": 4, "dim": 128, "kv": "bf16", "shifted": False, "mode": "required"}
    return {**case, **options}


def _repair(**options):
    case = {"kind": "repair", "requests": 1, "tokens": 32768, "spans": 15, "rows": 16, "q_heads": 28,
            "kv_heads": 4, "dim": 128, "kv": "bf16", "index": "int64"}
    return {**case, **options}


def listed():
    return [
        # One layer of a small request through the drop-in operator: the smallest call a
        # runtime makes, once per layer, where the host path and the launch are the cost.
        _operator(name="operator_one_layer_tokens", layers=1, tokens=2048, mask=True, prefix=512),
        # A model whose keys rotate a quarter of their dims (GPT-NeoX, Phi style).
        _operator(name="operator_quarter_rotary", rotary=32),
        # A model whose value heads are narrower than its key heads.
        _operator(name="operator_narrow_values", heads=8, value_dim=64),
        # A short chat's link (c1) with the reference's default rounding: latency of the
        # whole call, host preparation included.
        _link(name="link_2k_tokens", tokens=2048, blocks=4, seam=8, shifted=True, mode="disabled"),
        # The headline: a 32k-token request of 16 blocks (c2).
        _link(name="link_32k_tokens"),
        # The same length from many small blocks, half of it repair rows (c5).
        _link(name="link_512_blocks", blocks=512, seam=32, shifted=True),
        # A batch of requests that share catalogue blocks (c3): the largest link.
        _link(name="link_batch_of_24", requests=24, tokens=4096, blocks=8, catalogue=64, seam=8),
        # One layer's repair attention of c1's, c2's and c5's spans ...
        _repair(name="repair_2k_tokens", tokens=2048, spans=3, rows=8),
        _repair(name="repair_32k_tokens"),
        _repair(name="repair_512_blocks", spans=511, rows=32),
        # ... of a batch of requests like c3's ...
        _repair(name="repair_batch_of_24", requests=24, tokens=8192, spans=7, rows=8, index="int32"),
        # ... and of a model with wide heads in fp16.
        _repair(name="repair_head_dim_256", dim=256, tokens=16384, kv="fp16", q_heads=8),
    ]


# The most work that a drawn case may have, so that it costs no more than the listed ones.
_MOST_LINK_BYTES = 24 * 4096 * 28 * 4 * 128 * 2 * 2 * 2
_MOST_REPAIR_FLOPS = 3.0e12


def _log(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    kind = rng.choice(["operator", "link", "link", "repair", "repair"])
    while True:
        if kind == "operator":
            key, value, rotary = rng.choice([(128, 128, 128), (128, 128, 64), (128, 128, 32), (64, 64, 64),
                                             (256, 256, 256), (256, 256, 128), (32, 32, 32), (128, 64, 128),
                                             (40, 24, 16)])
            tokens = _log(rng, 16, 16384)
            case = _operator(layers=rng.choice([1, 1, 28, 64]), tokens=tokens, heads=rng.choice([1, 2, 3, 4, 8]),
                             key_dim=key, value_dim=value, rotary=rotary, kv=rng.choice(["bf16", "bf16", "fp16"]),
                             table=rng.choice(["fp32", "fp32", "bf16"]), neox=rng.random() < 0.8,
                             index=rng.choice(["int64", "int32"]), mask=rng.random() < 0.5,
                             prefix=rng.choice([0, tokens // 3]))
        elif kind == "link":
            requests = rng.choice([1, 1, _log(rng, 2, 24)])
            blocks = _log(rng, 2, 16) if requests > 1 else _log(rng, 2, 512)
            tokens = max(blocks * 33, _log(rng, 512, 32768))
            case = _link(requests=requests, tokens=tokens, blocks=blocks,
                         catalogue=0 if requests == 1 else blocks * rng.choice([2, 4, 8]),
                         seam=rng.choice([8, 16, 32]), layers=rng.choice([28, 64]), heads=rng.choice([1, 2, 4, 8]),
                         dim=rng.choice([64, 128, 128, 256]), kv=rng.choice(["bf16", "bf16", "fp16"]),
                         shifted=rng.random() < 0.5, mode=rng.choice(["required", "disabled"]))
        else:
            q_heads, kv_heads = rng.choice([(28, 4), (28, 4), (64, 8), (14, 2), (7, 1), (8, 8), (16, 2), (32, 1)])
            requests = rng.choice([1, 1, _log(rng, 2, 24)])
            tokens = _log(rng, 512, 32768)
            rows = rng.choice([1, 8, 16, 32])
            case = _repair(requests=requests, tokens=tokens, spans=_log(rng, 1, max(1, min(511, tokens // 33))),
                           rows=rows, q_heads=q_heads, kv_heads=kv_heads, dim=rng.choice([64, 128, 128, 256]),
                           kv=rng.choice(["bf16", "bf16", "fp16"]), index=rng.choice(["int64", "int32"]))
        cost = work(case)
        if cost["bytes"] <= _MOST_LINK_BYTES and cost["flops"] <= _MOST_REPAIR_FLOPS:
            return case


# -- what the cases hold ----------------------------------------------------


def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


@functools.lru_cache(maxsize=8)
def _table(rows, rotary, dtype):
    """The model's cos/sin table, built once per program."""

    return build_cos_sin_cache(rows, rotary, dtype=DTYPES[dtype]).cuda()


def _pool(generator, layers, slots, heads, dim, dtype):
    """[layers, slots, heads, dim] rows as a model's keys are distributed: channels of different scale."""

    rows = torch.randn(layers, slots, heads, dim, dtype=dtype, device="cuda", generator=generator)
    return rows.mul_(torch.linspace(0.25, 4.0, dim, device="cuda").to(dtype))


def _block_lengths(case):
    """Token counts of a request's blocks: uneven, at least 33 each (a batch's
    catalogue blocks are all alike); the same for every seed."""

    tokens, blocks = case["tokens"], case["blocks"]
    if case["requests"] > 1 or tokens == 64 * blocks:
        return [tokens // blocks] * blocks
    rng = np.random.default_rng([tokens, blocks])
    shares = rng.uniform(0.25, 1.75, blocks)
    lengths = 33 + np.floor((tokens - 33 * blocks) * shares / shares.sum()).astype(np.int64)
    lengths[0] += tokens - int(lengths.sum())
    return lengths.tolist()


def _chosen_blocks(case):
    """Which catalogue blocks each request links: popular ones in many requests."""

    if case["requests"] == 1:
        return [list(range(case["blocks"]))]
    rng = np.random.default_rng([case["requests"], case["tokens"], case["blocks"]])
    weights = 1.0 / np.arange(1, case["catalogue"] + 1) ** 1.1
    return [rng.choice(case["catalogue"], case["blocks"], replace=False, p=weights / weights.sum()).tolist()
            for _ in range(case["requests"])]


def _seam_rows(case):
    """Repair rows of one request: the first rows of every block after the first."""

    return sum(min(case["seam"], n) for n in _block_lengths(case)[1:])


def _span_ranges(case):
    """The repair spans of one request: evenly spread seams of ``rows`` rows."""

    tokens, spans, rows = case["tokens"], case["spans"], case["rows"]
    step = tokens / (spans + 1)
    starts = [min(int(step * (i + 1)), tokens - rows) for i in range(spans)]
    return [(max(s, 0), max(s, 0) + rows) for s in starts]


def prepare(case, seed):
    return {"operator": _prepare_operator, "link": _prepare_link, "repair": _prepare_repair}[case["kind"]](case, seed)


def _prepare_operator(case, seed):
    generator = _generator(seed)
    tokens, dtype, index = case["tokens"], DTYPES[case["kv"]], DTYPES[case["index"]]
    slots = 4 * tokens + 7
    keys = _pool(generator, case["layers"], slots, case["heads"], case["key_dim"], dtype)
    values = _pool(generator, case["layers"], slots, case["heads"], case["value_dim"], dtype)
    perm = torch.randperm(slots, device="cuda", generator=generator)
    # A block at local positions 0 .. n - 1, linked somewhere in a 32k context.
    local = torch.arange(tokens, device="cuda")
    shift = torch.randint(1, 32768 - 16384 + 1, (1,), device="cuda", generator=generator)
    position = local + shift
    mask = (torch.rand(tokens, device="cuda", generator=generator) < 0.02).to(torch.uint8) if case["mask"] else None
    arguments = dict(
        source_slots=perm[:tokens].to(index).contiguous(),
        destination_slots=perm[tokens:2 * tokens].to(index).contiguous(),
        local_positions=local.to(index), global_positions=position.to(index),
        cos_sin_cache=_table(32768, case["rotary"], case["table"]), prefix_token_count=case["prefix"],
        rotary_dim=case["rotary"], is_neox_style=case["neox"], repair_mask=mask)
    return {"kind": "operator", "keys": keys, "values": values, "arguments": arguments,
            "key_buffers": list(keys.unbind(0)), "value_buffers": list(values.unbind(0))}


def _prepare_link(case, seed):
    generator = _generator(seed)
    rng = np.random.default_rng(seed)
    dtype, layers, tokens = DTYPES[case["kv"]], case["layers"], case["tokens"]
    lengths = _block_lengths(case)
    catalogue = lengths if case["requests"] == 1 else [lengths[0]] * case["catalogue"]
    own = sum(lengths)
    registered = sum(catalogue)
    slots = registered + case["requests"] * own + 1024
    keys = _pool(generator, layers, slots, case["heads"], case["dim"], dtype)
    values = _pool(generator, layers, slots, case["heads"], case["dim"], dtype)
    perm = torch.randperm(slots, device="cuda", generator=generator)
    pool = KVPool(list(keys.unbind(0)), list(values.unbind(0)))
    registry = LegoLinkBlockRegistry()
    offsets = np.concatenate(([0], np.cumsum(catalogue)))
    first_positions = []
    for block, count in enumerate(catalogue):
        # Shifted blocks were compiled behind another prefix; a request's first block never moves then.
        first = int(rng.integers(0, 16384)) if case["shifted"] and block else 0
        first_positions.append(first)
        registry.register_legolink_block(f"block-{block}", range(count), perm[offsets[block]:offsets[block + 1]],
                                         compile_local_positions=range(first, first + count))
    requests, taken = [], registered
    for chosen in _chosen_blocks(case):
        destination = perm[taken:taken + own].clone()
        taken += own
        ranges, repair, start = [], [], 0
        for place, block in enumerate(chosen):
            count = catalogue[block]
            ranges.append({"start_token": start, "end_token": start + count})
            if place:
                repair.extend(range(start, start + min(case["seam"], count)))
            start += count
        requests.append((destination, {"cache_keys": [f"block-{b}" for b in chosen], "block_ranges": ranges,
                                       "imp_indices": repair}))
    rows = _seam_rows(case) * case["requests"]
    repaired_keys = _pool(generator, layers, rows, case["heads"], case["dim"], dtype)
    repaired_values = _pool(generator, layers, rows, case["heads"], case["dim"], dtype)
    rotary = RotarySpec(cos_sin_cache=_table(49152, case["dim"], "fp32"), rotary_dim=case["dim"], is_neox_style=True)
    executor = KVLinkExecutor(registry, rotary, end_layer=layers, fused_mode=case["mode"])
    return {"kind": "link", "keys": keys, "values": values, "pool": pool, "executor": executor,
            "requests": requests, "repaired_keys": repaired_keys, "repaired_values": repaired_values,
            "sources": [perm[offsets[b]:offsets[b + 1]] for b in range(len(catalogue))],
            "first_positions": first_positions}


def _prepare_repair(case, seed):
    generator = _generator(seed)
    dtype, index, tokens = DTYPES[case["kv"]], DTYPES[case["index"]], case["tokens"]
    slots = 2 * tokens * case["requests"] if case["requests"] < 4 else tokens * case["requests"] + 512
    keys = torch.randn(slots, case["kv_heads"], case["dim"], dtype=dtype, device="cuda", generator=generator)
    values = torch.randn(slots, case["kv_heads"], case["dim"], dtype=dtype, device="cuda", generator=generator)
    perm = torch.randperm(slots, device="cuda", generator=generator)
    spans = []
    for request in range(case["requests"]):
        own = perm[request * tokens:(request + 1) * tokens].to(index).contiguous()
        spans += [(own, start, end) for start, end in _span_ranges(case)]
    plan = RepairAttentionPlan(spans, num_q_heads=case["q_heads"], num_kv_heads=case["kv_heads"],
                               head_dim=case["dim"], pool_size=slots)
    query = 1.5 * torch.randn(plan.num_queries, case["q_heads"], case["dim"], device="cuda", generator=generator)
    return {"kind": "repair", "plan": plan, "query": query.to(dtype), "keys": keys, "values": values, "spans": spans}


def run(state):
    if state["kind"] == "operator":
        keys, values = state["key_buffers"], state["value_buffers"]
        if len(keys) == 1:
            kv_link.fused_kv_link_inplace(key_buffer=keys[0], value_buffer=values[0], **state["arguments"])
        else:
            kv_link.fused_kv_link_layers_inplace(key_buffers=keys, value_buffers=values, **state["arguments"])
        return {"keys": state["keys"], "values": state["values"]}
    if state["kind"] == "link":
        executor, pool, requests = state["executor"], state["pool"], state["requests"]
        if len(requests) == 1:
            link = executor.prepare_link(pool, *requests[0], boundary_repair_aware=True)
        else:
            link = executor.prepare_links(pool, requests, boundary_repair_aware=True)
        link.launch()
        link.write_repaired(state["repaired_keys"], state["repaired_values"])
        return {"keys": state["keys"], "values": state["values"]}
    return state["plan"].run(state["query"], state["keys"], state["values"])


def work(case):
    if case["kind"] == "operator":
        row = case["heads"] * (case["key_dim"] + case["value_dim"]) * 2
        index = 4 if case["index"] == "int32" else 8
        copied = case["tokens"] * (0.98 if case["mask"] else 1.0)
        return {"bytes": copied * case["layers"] * row * 2 + case["tokens"] * 4 * index,
                "flops": (case["tokens"] - case["prefix"]) * case["layers"] * case["heads"] * case["rotary"] * 3}
    if case["kind"] == "link":
        row = 2 * case["heads"] * case["dim"] * 2 * case["layers"]
        lengths = _block_lengths(case)
        if case["requests"] == 1:
            read = sum(lengths) - _seam_rows(case)
        else:
            # A shared block is read once; its first rows where some request has it first.
            chosen = _chosen_blocks(case)
            first = {blocks[0] for blocks in chosen}
            read = sum(lengths[0] - (0 if block in first else min(case["seam"], lengths[0]))
                       for block in set().union(*chosen))
        repaired = _seam_rows(case) * case["requests"]
        written = case["requests"] * sum(lengths)
        return {"bytes": (read + repaired + written) * row + written * 8,
                "flops": (written - repaired) * case["layers"] * case["heads"] * case["dim"] * 3}
    ranges = _span_ranges(case)
    pairs = case["requests"] * sum((end - start) * (start + end + 1) // 2 for start, end in ranges)
    queries = case["requests"] * case["spans"] * case["rows"]
    keys = case["requests"] * max(end for _, end in ranges)
    return {"bytes": keys * (2 * case["kv_heads"] * case["dim"] * 2 + (4 if case["index"] == "int32" else 8))
            + 2 * queries * case["q_heads"] * case["dim"] * 2,
            "flops": 4 * case["dim"] * case["q_heads"] * pairs}


def tolerance(case):
    if case["kind"] != "repair":
        return "exact"  # copied rows are bit copies, rotated ones have fixed rounding points
    # The output's and the probabilities' rounding to the 16-bit type (measured
    # against 64 bits: 2.1e-3 to 2.8e-3 in bf16, 3.5e-4 in fp16; about four times that here).
    return {"rel": 1e-2, "max": 0.1} if case["kv"] == "bf16" else {"rel": 1.5e-3, "max": 0.015}


# -- the same in 64 bits, with torch alone ----------------------------------


def _rotated(rows, local, position, table, rotary, neox):
    """Key rows [n, heads, dim] in float64 turned from ``local`` to ``position``."""

    half = rotary // 2
    table = table.double()
    lc, ls = table[local, :half][:, None], table[local, half:rotary][:, None]
    gc, gs = table[position, :half][:, None], table[position, half:rotary][:, None]
    dc, ds = gc * lc + gs * ls, gs * lc - gc * ls
    out = rows.clone()
    if neox:
        a, b = rows[..., :half], rows[..., half:rotary]
        out[..., :half], out[..., half:rotary] = a * dc - b * ds, b * dc + a * ds
    else:
        a, b = rows[..., 0:rotary:2], rows[..., 1:rotary:2]
        out[..., 0:rotary:2], out[..., 1:rotary:2] = a * dc - b * ds, b * dc + a * ds
    return out


def exact(case, seed):
    return {"operator": _exact_operator, "link": _exact_link, "repair": _exact_repair}[case["kind"]](case, seed)


def _exact_operator(case, seed):
    state = _prepare_operator(case, seed)
    arguments = state["arguments"]
    keys, values = state["keys"].double(), state["values"].double()
    kept = slice(None) if arguments["repair_mask"] is None else arguments["repair_mask"] == 0
    source, destination = arguments["source_slots"].long(), arguments["destination_slots"].long()
    local, position = arguments["local_positions"].long(), arguments["global_positions"].long()
    prefix = case["prefix"]
    for layer in range(case["layers"]):
        rows = keys[layer][source]
        rows[prefix:] = _rotated(rows[prefix:], local[prefix:], position[prefix:], arguments["cos_sin_cache"],
                                 case["rotary"], case["neox"])
        keys[layer][destination[kept]] = rows[kept]
        values[layer][destination[kept]] = values[layer][source][kept]
    return {"keys": keys, "values": values}


def _exact_link(case, seed):
    state = _prepare_link(case, seed)
    keys, values = state["keys"].double(), state["values"].double()
    table = state["executor"].rotary_by_layer[0].cos_sin_cache
    taken = 0
    for destination, plan in state["requests"]:
        source, local = [], []
        for key, bounds in zip(plan["cache_keys"], plan["block_ranges"]):
            block = int(key.split("-")[1])
            count, first = bounds["end_token"] - bounds["start_token"], state["first_positions"][block]
            source.append(state["sources"][block])
            local.append(torch.arange(first, first + count, device="cuda"))
        source, local = torch.cat(source), torch.cat(local)
        position = torch.arange(source.numel(), device="cuda")
        repair = torch.tensor(plan["imp_indices"], device="cuda", dtype=torch.int64)
        for layer in range(case["layers"]):
            keys[layer][destination] = _rotated(keys[layer][source], local, position, table, case["dim"], True)
            values[layer][destination] = values[layer][source]
            part = slice(taken, taken + repair.numel())
            keys[layer][destination[repair]] = state["repaired_keys"][layer, part].double()
            values[layer][destination[repair]] = state["repaired_values"][layer, part].double()
        taken += repair.numel()
    return {"keys": keys, "values": values}


def _exact_repair(case, seed):
    state = _prepare_repair(case, seed)
    query, group = state["query"].double(), case["q_heads"] // case["kv_heads"]
    out = torch.empty_like(query)
    per_request = case["spans"] * case["rows"]
    for request in range(case["requests"]):
        spans = state["spans"][request * case["spans"]:(request + 1) * case["spans"]]
        slots = spans[0][0].long()
        positions = torch.cat([torch.arange(start, end, device="cuda") for _, start, end in spans])
        for head in range(case["kv_heads"]):
            key, value = state["keys"][slots, head].double(), state["values"][slots, head].double()
            for begin in range(0, per_request, 1024):
                rows = slice(request * per_request + begin, request * per_request + min(begin + 1024, per_request))
                heads = slice(head * group, (head + 1) * group)
                at = positions[begin:begin + 1024]
                part = query[rows, heads].reshape(-1, case["dim"])
                seen = int(at.max()) + 1
                scores = part @ key[:seen].t() / math.sqrt(case["dim"])
                hidden = torch.arange(seen, device="cuda")[None] > at.repeat_interleave(group)[:, None]
                weights = torch.softmax(scores.masked_fill_(hidden, -math.inf), dim=-1)
                out[rows, heads] = (weights @ value[:seen]).view(-1, group, case["dim"])
    return out
