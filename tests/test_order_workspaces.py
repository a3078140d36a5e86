"""The visit order's workspaces: one per stream, never shared by calls that may
overlap, and made only where an order needs one."""

from __future__ import annotations

import threading
import time

import pytest
import torch

from legolink_amd import _native, link_maps
from legolink_amd.link_runtime import KVLinkExecutor, KVPool, RotarySpec
from legolink_amd.registry import LegoLinkBlockRegistry

OPTIONS = dict(key_row=1, prefix=0, num_slots=10)


def _fake(monkeypatch, streams, seen, hold=0.0):
    """An order that records (stream, workspace) of each call and whether another
    call on that workspace was under way; it fails for a prefix of -1."""

    busy = {}

    def order(maps, mask, key_row, prefix, num_slots, workspace, handle, stream, exact):
        key = workspace.data_ptr()
        seen.append((streams(), key, busy.get(key, False)))
        busy[key] = True
        time.sleep(hold)
        busy[key] = False
        if prefix < 0:
            raise _native.NativeCallError(-1, "hip_error", "launch failed")
        return maps, mask

    monkeypatch.setattr(link_maps, "_order", order)
    monkeypatch.setattr(_native, "stream_handle", lambda stream, device: streams())
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)


def test_streams_do_not_share_a_workspace(monkeypatch):
    seen, stream = [], [1]
    _fake(monkeypatch, lambda: stream[0], seen)
    workspaces, maps = link_maps.OrderWorkspaces(), torch.zeros(4, 3, dtype=torch.int64)
    for stream[0] in (1, 2, 1, 3, 2):
        workspaces.order(maps, None, **OPTIONS)
    used = {}
    for handle, key, _ in seen:
        assert used.setdefault(handle, key) == key
    assert len(set(used.values())) == 3


def test_threads_on_one_stream_take_turns(monkeypatch):
    seen = []
    _fake(monkeypatch, lambda: 7, seen, hold=0.01)
    workspaces, maps = link_maps.OrderWorkspaces(), torch.zeros(4, 3, dtype=torch.int64)
    threads = [threading.Thread(target=workspaces.order, args=(maps, None), kwargs=OPTIONS) for _ in range(8)]
    for thread in threads:
        thread.start()
    for thread in threads:
        thread.join()
    assert len(seen) == 8 and not any(overlapped for _, _, overlapped in seen)


def test_a_capture_and_a_failed_call_leave_no_shared_workspace(monkeypatch):
    seen = []
    _fake(monkeypatch, lambda: 7, seen)
    workspaces, maps = link_maps.OrderWorkspaces(), torch.zeros(4, 3, dtype=torch.int64)
    workspaces.order(maps, None, **OPTIONS)
    kept = workspaces._kept[None, 7]
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: True)
    workspaces.order(maps, None, **OPTIONS)
    assert seen[1][1] != kept.data_ptr() and workspaces._kept[None, 7] is kept
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
    with pytest.raises(_native.NativeCallError):
        workspaces.order(maps, None, **{**OPTIONS, "prefix": -1})
    assert not workspaces._kept  # its counters may be left half-way
    for handle in range(link_maps.OrderWorkspaces.LIMIT + 5):
        monkeypatch.setattr(_native, "stream_handle", lambda stream, device, handle=handle: handle)
        workspaces.order(maps, None, **OPTIONS)
    assert len(workspaces._kept) == link_maps.OrderWorkspaces.LIMIT


def _setup(device, slots, tokens):
    pool = KVPool.allocate(num_slots=slots, num_layers=2, num_heads=1, head_dim=32, device=device)
    for buffer in pool.k_buffer + pool.v_buffer:
        buffer.normal_()
    registry = LegoLinkBlockRegistry()
    perm = torch.randperm(slots, device=device)
    for name, first in (("a", 0), ("b", tokens)):
        registry.register_legolink_block(name, range(tokens), perm[first:first + tokens],
                                         compile_local_positions=range(tokens))
    executor = KVLinkExecutor(registry, RotarySpec.for_theta(4 * tokens, 32), end_layer=2, fused_mode="required")
    plan = {"cache_keys": ["a", "b"], "block_ranges": [{"start_token": 0, "end_token": tokens},
                                                       {"start_token": tokens, "end_token": 2 * tokens}]}
    return pool, executor, perm, plan


@pytest.mark.gpu
@pytest.mark.parametrize("requests", [1, 2])
def test_links_prepared_on_two_streams_keep_apart(gpu_device, requests):
    """Two links prepared in turn on two streams, both on the way at once, equal
    the same links prepared alone; a batch over a pool too large for the exact
    order makes no workspace."""

    tokens, slots = 30000, 300000
    pool, executor, perm, plan = _setup(gpu_device, slots, tokens)
    starts = [buffer.clone() for buffer in pool.k_buffer + pool.v_buffer]
    batches = [[(perm[tokens * (2 + 2 * (requests * k + r)):][:2 * tokens].clone(), plan) for r in range(requests)]
               for k in range(2)]

    def prepare(batch):
        if requests == 1:
            return executor.prepare_link(pool, *batch[0])
        return executor.prepare_links(pool, batch)

    def restore():
        torch.cuda.synchronize(gpu_device)
        for buffer, start in zip(pool.k_buffer + pool.v_buffer, starts):
            buffer.copy_(start)
        torch.cuda.synchronize(gpu_device)

    for batch in batches:
        prepare(batch).launch()
    torch.cuda.synchronize(gpu_device)
    want = [buffer.clone() for buffer in pool.k_buffer + pool.v_buffer]
    for _ in range(5):
        restore()
        streams = [torch.cuda.Stream(gpu_device) for _ in range(2)]
        links = []
        for stream, batch in zip(streams, batches):
            with torch.cuda.stream(stream):
                links.append(prepare(batch))
                links[-1].launch()
        torch.cuda.synchronize(gpu_device)
        for buffer, expected in zip(pool.k_buffer + pool.v_buffer, want):
            assert torch.equal(buffer, expected)
    assert len(executor._order_workspaces._kept) >= 2


@pytest.mark.gpu
def test_an_order_without_buckets_makes_no_workspace(gpu_device, monkeypatch):
    tokens = 100
    pool, executor, perm, plan = _setup(gpu_device, 3000, tokens)
    monkeypatch.setattr(_native, "ORDER_EXACT_SLOTS", 2000)  # as for a pool beyond the exact order's
    batch = [(perm[tokens * (2 + 2 * r):][:2 * tokens].clone(), plan) for r in range(2)]
    executor.prepare_links(pool, batch).launch()
    executor.prepare_links(pool, batch, order_by_source=False).launch()
    torch.cuda.synchronize(gpu_device)
    assert not executor._order_workspaces._kept
