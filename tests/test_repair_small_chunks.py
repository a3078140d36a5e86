"""Plans that know the head dim: chunks below 512 keys, wide (fp32) partials,
the workspace limit, and the two workgroups per window of head dim 256."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from legolink_amd import _native
from legolink_amd.repair_attention import RepairAttentionPlan

WIDE = 0x100


def _rows(context, spans, rows):
    step = context // (spans + 1)
    starts = [min(step * (i + 1), context - rows) for i in range(spans)]
    return np.array([(i * rows, s, rows, 0) for i, s in enumerate(starts)], dtype=np.int64)


def _slot_bytes(heads, dim):
    return heads * (16 * dim * 2 + 128)


@pytest.mark.parametrize("context,spans,rows,heads,dim", [
    (2048, 3, 8, (28, 4), 128), (2000, 2, 16, (16, 2), 64), (1000, 5, 16, (64, 8), 256), (1500, 2, 16, (32, 1), 128),
])
def test_short_chunks_fill_idle_compute_units_with_wide_partials(context, spans, rows, heads, dim):
    table = _rows(context, spans, rows)
    items, combine, positions, info = _native.repair_attention_plan(table, *heads, 0, head_dim=dim)
    assert info.split_tokens < 512 and info.split_tokens % 64 == 0 and info.num_combine > 0
    assert (items[:, 5] & WIDE).all() and (combine[:, 1] & WIDE).all()
    # Every (tile, chunk) has an even slot of its own, two slots wide, inside the workspace.
    expected = set()
    for first, count in combine[:, 2:].tolist():
        expected |= set(range(first, first + 2 * count, 2))
    assert len(expected) == int(combine[:, 3].sum()) and info.workspace_items == 2 * len(expected)
    H, T = _native.REPAIR_ITEM_HEADER, _native.REPAIR_TILE_INTS
    used = set()
    for item in items.tolist():
        used |= {item[H + T * t + 3] for t in range(item[3]) if item[H + T * t + 2] > 0} - {-1}
    assert used == expected
    # The same plan again with the chosen length given, and the plain entry's
    # plan (head dim not known): at least 512 keys per chunk, no flag.
    again = _native.repair_attention_plan(table, *heads, int(info.split_tokens), head_dim=dim)
    assert np.array_equal(again[0], items) and np.array_equal(again[1], combine)
    plain = _native.repair_attention_plan(table, *heads, 0)
    assert plain[3].split_tokens >= 512 and not (plain[0][:, 5] & WIDE).any()


def test_chunks_stay_at_512_where_they_fill_the_device():
    table = _rows(32768, 15, 16)
    assert _native.repair_attention_plan(table, 28, 4, 0, head_dim=128)[3].split_tokens >= 512


def test_the_combine_is_priced_in_the_head_dims_own_tiles():
    """A key tile of head dim 64 takes 0.8 times that of 128, one of 256 1.5 times
    (not half and twice): shapes where the difference decides."""

    plan = _native.repair_attention_plan(_rows(15838, 5, 8), 14, 2, 0, head_dim=256)[3]
    assert plan.split_tokens >= 512 and plan.num_items <= 40  # 39 us; in 73 items of 256 keys 51 us
    plan = _native.repair_attention_plan(_batch(8, 850, 9, 1), 16, 2, 0, head_dim=64)[3]
    assert plan.num_items > 16  # 12.3 us in 48 items; in 8 whole ranges 19.3 us


@pytest.mark.parametrize("context,spans,rows", [(16384, 15, 16), (8192, 7, 16)])
def test_head_dim_256_plans_one_round_of_its_two_workgroups_per_window(context, spans, rows):
    items, _, _, info = _native.repair_attention_plan(_rows(context, spans, rows), 8, 4, 0, head_dim=256)
    assert info.num_items * 4 * 2 <= 256


def _batch(requests, context, spans, rows):
    """The rows of `requests` requests of `context` keys with `spans` spans each."""

    one = _rows(context, spans, rows)
    table = np.concatenate([one] * requests)
    table[:, 0] = np.arange(len(table)) * rows
    table[:, 3] = np.repeat(np.arange(requests) * context, spans)
    return table


def _check_splits_are_wide(table, heads, dim, limit=0):
    """A tile that the plan made without the head dim keeps whole, in fp32 from
    end to end, is whole here too, or its partials are fp32.  Returns whether
    the plan splits such a tile."""

    blind = _native.repair_attention_plan(table, *heads, 0)[1]
    items, combine, _, info = _native.repair_attention_plan(table, *heads, 0, head_dim=dim, workspace_limit=limit)
    newly_split = set(combine[:, 0].tolist()) - set(blind[:, 0].tolist())
    if newly_split:
        assert (combine[:, 1] & WIDE).all() and (items[:, 5] & WIDE).all(), (heads, dim, info.split_tokens)
        assert info.workspace_items == 2 * int(combine[:, 3].sum())
    assert limit == 0 or info.workspace_items * _slot_bytes(heads[0], dim) <= limit
    return bool(newly_split)


NEWLY_SPLIT = [(6, 938, 10, 32, (28, 4)), (12, 875, 4, 32, (32, 1)), (14, 1727, 2, 32, (64, 8))]


@pytest.mark.parametrize("requests,context,spans,rows,heads", NEWLY_SPLIT)
def test_ranges_that_stayed_whole_split_into_wide_partials(requests, context, spans, rows, heads):
    table = _batch(requests, context, spans, rows)
    for limit in (0, 64 << 20, 1 << 20):
        _check_splits_are_wide(table, heads, 256, limit)
    # A chunk length that the caller gives (512 keys and more) keeps its 16-bit
    # partials, whatever was planned before on this thread.
    chosen = _native.repair_attention_plan(table, *heads, 0, head_dim=256)
    given = _native.repair_attention_plan(table, *heads, max(512, int(chosen[3].split_tokens)), head_dim=256)
    assert not (given[1][:, 1] & WIDE).any()


def test_drawn_plans_never_lose_the_partials_precision():
    rng = np.random.default_rng(7)
    split = 0
    for _ in range(400):
        dim = int(rng.choice([64, 128, 256, 256]))
        heads = [(28, 4), (64, 8), (14, 2), (7, 1), (8, 8), (16, 2), (32, 1)][rng.integers(7)]
        context = int(np.exp(rng.uniform(np.log(512), np.log(32768))))
        rows = int(rng.choice([1, 8, 16, 32]))
        spans = int(np.exp(rng.uniform(0, np.log(max(1, min(64, context // 33))))))
        split += _check_splits_are_wide(_batch(int(rng.integers(1, 25)), context, spans, rows), heads, dim)
    assert split > 0


def test_a_workspace_limit_bounds_the_partials():
    """Whatever the limit, the plan's partials fit it; the limit of the
    allocation-free entry is the library's scratch array."""

    table = _rows(32768, 3, 16)
    for limit in (0, 64 << 20, 8 << 20, 1 << 20, 1):
        info = _native.repair_attention_plan(table, 64, 8, 0, head_dim=256, workspace_limit=limit)[3]
        assert limit == 0 or info.workspace_items * _slot_bytes(64, 256) <= limit
    slots = torch.arange(32768)
    plan = RepairAttentionPlan([(slots, 32000, 32016)], num_q_heads=512, num_kv_heads=2, head_dim=256,
                               allocation_free=True)
    assert plan.info["workspace_items"] * _slot_bytes(512, 256) <= _native.repair_scratch_bytes()
    # A given length whose 16-bit partials fit the limit is not widened past it.
    limit = 48 << 20
    narrow = _native.repair_attention_plan(_rows(16384, 2, 16), 28, 4, 64, head_dim=128, workspace_limit=limit)[3]
    wide = _native.repair_attention_plan(_rows(16384, 2, 16), 28, 4, 64, head_dim=128)[3]
    assert narrow.workspace_items * 2 == wide.workspace_items
    assert narrow.workspace_items * _slot_bytes(28, 128) <= limit < wide.workspace_items * _slot_bytes(28, 128)


def test_bad_head_dims_and_limits_are_refused():
    table = _rows(1000, 1, 8)
    with pytest.raises(_native.NativeCallError):
        _native.repair_attention_plan(table, 8, 4, 0, head_dim=96)
    with pytest.raises(_native.NativeCallError):
        _native.repair_attention_plan(table, 8, 4, 0, head_dim=128, workspace_limit=-1)
    # A plan object still takes any head dim (run() refuses it).
    RepairAttentionPlan([(torch.arange(1000), 1, 9)], num_q_heads=8, num_kv_heads=4, head_dim=96)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("context,spans,rows,heads,dim", [
    (2048, 3, 8, (28, 4), 128), (2113, 2, 17, (8, 8), 64), (1000, 5, 1, (12, 4), 256), (2500, 1, 33, (32, 1), 128),
    (4100, 6, 16, (7, 1), 64), (1471, 4, 16, (64, 8), 256),
])
def test_short_chunks_are_as_exact_as_whole_ranges(gpu_device, context, spans, rows, heads, dim, dtype):
    """Against fp64: within the bound of the probabilities' rounding (half an
    ulp of each, 2^-8 of weighted |V| with its sum) and the output's (2^-9);
    wide partials add fp32 terms only.  The error is that of the same run with
    every range whole (the 5 % are the probabilities' other rounding, drawn
    anew by each chunk's own maximum)."""

    generator = torch.Generator(device=gpu_device).manual_seed(context)
    pool, (hq, hkv) = context + 100, heads
    key, value = (torch.randn(pool, hkv, dim, device=gpu_device, generator=generator).to(dtype) for _ in range(2))
    slots = torch.randperm(pool, device=gpu_device, generator=generator)[:context]
    slots[context // 3] = -1  # an invisible key
    table = _rows(context, spans, rows)
    plan_spans = [(slots, int(s), int(s + n)) for _, s, n, _ in table.tolist()]
    common = dict(num_q_heads=hq, num_kv_heads=hkv, head_dim=dim)
    short = RepairAttentionPlan(plan_spans, **common)
    assert short.info["split_tokens"] < 512 and short.info["num_combine"] > 0
    whole = RepairAttentionPlan(plan_spans, split_tokens=8192, **common)
    free = RepairAttentionPlan(plan_spans, allocation_free=True, **common)
    query = (1.5 * torch.randn(short.num_queries, hq, dim, device=gpu_device, generator=generator)).to(dtype)
    positions = torch.cat([torch.arange(s, e, device=gpu_device) for _, s, e in plan_spans])
    hidden = torch.arange(context, device=gpu_device)[None] > positions[:, None]
    hidden[:, context // 3] = True
    safe = slots.clamp(min=0)
    errors = []
    for plan in (short, whole, free):
        got = plan.run(query, key, value).double()
        total = 0.0
        for head in range(hq):
            k, v = key[safe, head // (hq // hkv)].double(), value[safe, head // (hq // hkv)].double()
            scores = (query[:, head].double() @ k.t()) / dim ** 0.5
            weights = torch.softmax(scores.masked_fill(hidden, float("-inf")), dim=-1)
            want, size = weights @ v, weights @ v.abs()
            error = (got[:, head] - want).abs()
            assert (error <= 2.0 ** -8 * size + 2.0 ** -9 * want.abs() + 1e-5).all()
            total += float((error ** 2).sum())
        errors.append(total ** 0.5)
    assert errors[0] <= 1.05 * errors[1] and errors[2] == errors[0], errors


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("requests,context,spans,rows,heads", NEWLY_SPLIT)
def test_newly_split_ranges_are_as_exact_as_whole_ones(gpu_device, requests, context, spans, rows, heads, dtype):
    """Against fp64, as test_short_chunks_are_as_exact_as_whole_ranges: the chosen
    plan's error is that of every range whole."""

    dim, (hq, hkv) = 256, heads
    generator = torch.Generator(device=gpu_device).manual_seed(context)
    pool = requests * context + 100
    key, value = (torch.randn(pool, hkv, dim, device=gpu_device, generator=generator).to(dtype) for _ in range(2))
    perm = torch.randperm(pool, device=gpu_device, generator=generator)
    table = _rows(context, spans, rows).tolist()
    lists = [perm[r * context:(r + 1) * context].contiguous() for r in range(requests)]
    plan_spans = [(slots, int(s), int(s + n)) for slots in lists for _, s, n, _ in table]
    common = dict(num_q_heads=hq, num_kv_heads=hkv, head_dim=dim)
    chosen = RepairAttentionPlan(plan_spans, **common)
    whole = RepairAttentionPlan(plan_spans, split_tokens=8192, **common)
    query = (1.5 * torch.randn(chosen.num_queries, hq, dim, device=gpu_device, generator=generator)).to(dtype)
    positions = torch.cat([torch.arange(s, s + n, device=gpu_device) for _, s, n, _ in table])
    hidden = torch.arange(context, device=gpu_device)[None] > positions[:, None]
    errors = []
    for plan in (chosen, whole):
        got = plan.run(query, key, value).double().view(requests, -1, hq, dim)
        total = 0.0
        for request, slots in enumerate(lists):
            for head in range(hq):
                k, v = key[slots, head // (hq // hkv)].double(), value[slots, head // (hq // hkv)].double()
                q = query.view(requests, -1, hq, dim)[request, :, head].double()
                weights = torch.softmax((q @ k.t() / dim ** 0.5).masked_fill(hidden, float("-inf")), dim=-1)
                total += float(((got[request, :, head] - weights @ v) ** 2).sum())
        errors.append(total ** 0.5)
    assert errors[0] <= 1.05 * errors[1], errors


@pytest.mark.gpu
@pytest.mark.parametrize("requests,context,spans,rows,heads,dim", [
    (1, 32768, 1, 1, (28, 4), 128), (1, 8192, 2, 16, (28, 4), 256), (1, 8192, 2, 3, (64, 8), 64),
    (2, 32768, 5, 32, (28, 4), 128), (12, 12000, 3, 32, (28, 4), 256), (14, 12000, 3, 16, (64, 8), 64),
])
def test_the_combine_depends_on_the_plan_alone(gpu_device, requests, context, spans, rows, heads, dim):
    """Launches of few and of many workgroups (one and two groups of threads
    each): the same bits with a larger workspace than the plan's, and the whole
    ranges' result.  Probabilities, partials and outputs are each rounded to
    2^-9 of themselves, independently per key as the output's own terms are, in
    either run: 2^-7 of the output's norm for all four."""

    generator = torch.Generator(device=gpu_device).manual_seed(context + dim)
    pool, (hq, hkv) = requests * context + 64, heads
    key, value = (torch.randn(pool, hkv, dim, device=gpu_device, generator=generator).bfloat16() for _ in range(2))
    perm = torch.randperm(pool, device=gpu_device, generator=generator)
    plan_spans = [(perm[r * context:(r + 1) * context].contiguous(), int(s), int(s + n))
                  for r in range(requests) for _, s, n, _ in _rows(context, spans, rows).tolist()]
    common = dict(num_q_heads=hq, num_kv_heads=hkv, head_dim=dim)
    plan = RepairAttentionPlan(plan_spans, split_tokens=640, **common)
    query = torch.randn(plan.num_queries, hq, dim, device=gpu_device, generator=generator).bfloat16()
    assert plan.info["num_combine"] > 0 and int(plan.combine[3::4].max()) > 8
    got = plan.run(query, key, value)
    plan.info["workspace_items"] *= 9
    plan.workspace = torch.empty(9 * plan.workspace.numel(), device=gpu_device)
    assert torch.equal(plan.run(query, key, value), got)
    whole = RepairAttentionPlan(plan_spans, split_tokens=32768, **common).run(query, key, value)
    assert float((got.double() - whole.double()).norm()) <= 2.0 ** -7 * float(whole.double().norm())


@pytest.mark.gpu
def test_counts_with_other_bits_than_the_wide_flag_are_refused(gpu_device):
    """An item or combine item whose count is none (negative, or with bits above
    the flag) is skipped, as without the flag: its output stays as it was."""

    slots = torch.randperm(2000, device=gpu_device)
    key, value = (torch.randn(2000, 4, 128, device=gpu_device).bfloat16() for _ in range(2))
    plan = RepairAttentionPlan([(slots, 1900, 1916)], num_q_heads=28, num_kv_heads=4, head_dim=128)
    query = torch.randn(16, 28, 128, device=gpu_device).bfloat16()
    good = plan.run(query, key, value)
    assert plan.info["num_combine"] == 1 and int(plan.combine[1]) == 16 | WIDE
    for change in (1 << 9, 1 << 20, -1 << 31):
        plan.combine[1] ^= change
        untouched = torch.full_like(good, 7.0)
        plan.run(query, key, value, output=untouched)
        assert bool((untouched == 7.0).all())
        plan.combine[1] ^= change
    whole = RepairAttentionPlan([(slots, 100, 116)], num_q_heads=28, num_kv_heads=4, head_dim=128, split_tokens=512)
    assert whole.info["num_combine"] == 0
    counts = whole.items.view(-1, _native.REPAIR_ITEM_INTS)[:, 5]
    for change in (1 << 9, 1 << 20, -1 << 31):
        counts ^= change
        untouched = torch.full_like(good, 7.0)
        whole.run(query, key, value, output=untouched)
        assert bool((untouched == 7.0).all())
        counts ^= change
    assert torch.equal(plan.run(query, key, value), good)
