"""The exact visit order (ll_order_link_maps_exact): a permutation that keeps
the identity prefix and lists the rest by slot, at pool sizes with one, two and
64 slots per bucket, entries piled on few slots, and out-of-range slots; and the
bucketed order of small maps, which one workgroup makes."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from legolink_amd import _native, link_maps

CASES = [
    # entries, prefix, pool rows, distinct slots (0: any), outside
    (5000, 0, 12000, 0, False),            # one slot per bucket
    (40000, 64, 16385, 0, False),          # two
    (98304, 0, 164864, 65536, False),      # a batch's pool, shared rows
    (60000, 1000, 1 << 20, 700, False),    # 64 slots per bucket, piled up
    (30000, 1, 1 << 20, 1, False),         # every entry on one slot
    (20000, 0, 262144, 0, True),
    (3000, 3000, 100000, 0, False),        # all prefix
    (2, 1, 1 << 20, 0, False),
    (63, 0, 1 << 20, 0, False),
    (1, 0, 1 << 20, 0, False),
]


@pytest.mark.gpu
@pytest.mark.parametrize("with_mask", [False, True])
@pytest.mark.parametrize("num_slots", [1, 16384, 70000, 1 << 22])
@pytest.mark.parametrize("n,prefix", [(1, 0), (63, 0), (1025, 1), (2047, 64), (2048, 2048), (2048, 0), (2049, 0)])
def test_small_maps_order_in_one_workgroup_as_in_three_launches(gpu_device, n, prefix, num_slots, with_mask):
    """Sizes on both sides of the one-workgroup line: bucket order, the prefix and the masks kept."""

    rng = np.random.default_rng([n, num_slots])
    host = np.stack([rng.integers(0, 1 << 40, n), rng.integers(-2, num_slots + 2, n), rng.integers(0, 99, n),
                     np.arange(n) * 5 + 1]).astype(np.int64)
    mask_host = rng.integers(0, 2, n).astype(np.uint8)
    mask = torch.from_numpy(mask_host).to(gpu_device) if with_mask else None
    workspace = torch.zeros(_native.ORDER_WORKSPACE_BYTES, dtype=torch.uint8, device=gpu_device)
    out, out_mask = link_maps.order_link_maps(torch.from_numpy(host).to(gpu_device), mask, key_row=1, prefix=prefix,
                                              num_slots=num_slots, workspace=workspace)
    got = out.cpu().numpy()
    assert np.array_equal(got[:, :prefix], host[:, :prefix])
    assert np.array_equal(got[:, np.argsort(got[3])], host)
    shift = max(0, int(num_slots - 1).bit_length() - 14)
    buckets = np.clip(got[1, prefix:], 0, num_slots - 1) >> shift
    buckets[got[1, prefix:] >= num_slots] = _native.ORDER_BUCKETS - 1
    assert (np.diff(buckets) >= 0).all()
    if with_mask:
        assert np.array_equal(out_mask.cpu().numpy()[np.argsort(got[3])], mask_host)
    assert int(workspace.count_nonzero()) == 0 or n > 2048


@pytest.mark.gpu
@pytest.mark.parametrize("key_row", [0, 1])
@pytest.mark.parametrize("with_mask", [False, True])
@pytest.mark.parametrize("case", CASES, ids=str)
def test_exact_order(gpu_device, case, with_mask, key_row):
    n, prefix, num_slots, distinct, outside = case
    rng = np.random.default_rng([n, num_slots, key_row])
    slots = rng.choice(num_slots, distinct, replace=False) if distinct else np.arange(num_slots)
    host = np.stack([rng.integers(0, 1 << 40, n) for _ in range(3)] + [np.arange(n) * 5 + 1]).astype(np.int64)
    host[key_row] = rng.choice(slots, n)
    if outside:
        pick = rng.choice(n, n // 40, replace=False)
        host[key_row, pick] = rng.choice([-1, -(1 << 40), num_slots, 1 << 50], pick.size)
    mask_host = rng.integers(0, 2, n).astype(np.uint8)
    maps = torch.from_numpy(host).to(gpu_device)
    mask = torch.from_numpy(mask_host).to(gpu_device) if with_mask else None
    workspace = torch.zeros(_native.ORDER_WORKSPACE_BYTES, dtype=torch.uint8, device=gpu_device)
    for _ in range(2):  # the second call reuses the workspace
        out, out_mask = link_maps.order_link_maps(maps, mask, key_row=key_row, prefix=prefix, num_slots=num_slots,
                                                  workspace=workspace, exact=True)
        got = out.cpu().numpy()
        assert np.array_equal(got[:, :prefix], host[:, :prefix])
        assert np.array_equal(got[:, np.argsort(got[3])], host)  # column 3 tells the entries apart
        tail = got[key_row, prefix:]
        if outside:
            tail = tail[(tail >= 0) & (tail < num_slots)]
        assert (np.diff(tail) >= 0).all()
        if with_mask:
            assert np.array_equal(out_mask.cpu().numpy()[np.argsort(got[3])], mask_host)
        assert int(workspace.view(torch.int32)[: _native.ORDER_BUCKETS].count_nonzero()) == 0


@pytest.mark.gpu
@pytest.mark.parametrize("n,prefix,num_slots", [(524288, 0, 1 << 20), (524289, 1025, 1 << 20), (1200003, 600, 16384)])
def test_exact_order_of_runs_of_several_chunks(gpu_device, n, prefix, num_slots):
    """More entries than one chunk of 1,024 for each of the 512 workgroups."""

    generator = torch.Generator(device=gpu_device).manual_seed(n)
    maps = torch.randint(0, 1 << 40, (4, n), device=gpu_device, generator=generator)
    maps[0] = torch.randint(0, num_slots, (n,), device=gpu_device, generator=generator)
    maps[3] = torch.arange(n, device=gpu_device)  # tells the entries apart
    workspace = torch.zeros(_native.ORDER_WORKSPACE_BYTES, dtype=torch.uint8, device=gpu_device)
    out, _ = link_maps.order_link_maps(maps, None, key_row=0, prefix=prefix, num_slots=num_slots,
                                       workspace=workspace, exact=True)
    assert torch.equal(out[:, :prefix], maps[:, :prefix])
    assert bool((out[0, prefix:].diff() >= 0).all())
    assert torch.equal(out[:, torch.argsort(out[3])], maps)


@pytest.mark.gpu
def test_piled_up_slots_order_as_fast_as_spread_ones(gpu_device):
    """24 requests of the same eight blocks, their slots side by side in a large
    pool or scattered over it: within a factor of four (measured 1.1; with an
    atomic per entry on the buckets' counters 20)."""

    pool, blocks, tokens, requests = 1 << 20, 8, 512, 24
    workspace = torch.zeros(_native.ORDER_WORKSPACE_BYTES, dtype=torch.uint8, device=gpu_device)
    times = []
    for slots in (torch.arange(1000, 1000 + blocks * tokens, device=gpu_device),
                  torch.randperm(pool, device=gpu_device)[:blocks * tokens]):
        maps = torch.zeros(4, requests * slots.numel(), dtype=torch.int64, device=gpu_device)
        maps[0] = slots.repeat(requests)
        best = float("inf")
        for _ in range(5):
            begin, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            begin.record()
            for _ in range(20):
                link_maps.order_link_maps(maps, None, key_row=0, prefix=0, num_slots=pool, workspace=workspace,
                                          exact=True)
            end.record()
            torch.cuda.synchronize(gpu_device)
            best = min(best, begin.elapsed_time(end))
        times.append(best)
    assert times[0] < 4 * times[1], times


def test_exact_order_refuses_what_it_cannot_take():
    """Host checks only: no GPU work is enqueued for these."""

    buffers = [np.zeros(4 * 16, dtype=np.int64) for _ in range(3)]
    workspace = np.zeros(_native.ORDER_WORKSPACE_BYTES + 16, dtype=np.uint8)
    args = _native.OrderMapsArgs()
    args.maps, args.out_maps = buffers[0].ctypes.data, buffers[1].ctypes.data
    args.capacity = args.count = 16
    args.workspace = (workspace.ctypes.data + 15) // 16 * 16
    args.workspace_bytes = _native.ORDER_WORKSPACE_BYTES
    scratch = buffers[2].ctypes.data
    for num_slots, scratch_maps, text in (((1 << 20) + 1, scratch, "at most"), (100, None, "scratch maps"),
                                          (100, args.maps, "overlap"), (100, args.out_maps + 8, "overlap"),
                                          (100, scratch + 4, "scratch maps")):
        args.num_slots = num_slots
        with pytest.raises(_native.NativeCallError, match=text):
            _native.order_link_maps_exact(args, scratch_maps, None, 0)


def test_exact_order_refuses_a_scratch_mask_that_overlaps():
    """Host checks only, as above: the scratch mask is read after the output mask is written."""

    maps, out, scratch = (np.zeros(4 * 16, dtype=np.int64) for _ in range(3))
    masks = np.zeros(16 * 3, dtype=np.uint8)
    workspace = np.zeros(_native.ORDER_WORKSPACE_BYTES + 16, dtype=np.uint8)
    args = _native.OrderMapsArgs()
    args.maps, args.out_maps = maps.ctypes.data, out.ctypes.data
    args.mask, args.out_mask = masks.ctypes.data, masks.ctypes.data + 16
    args.capacity = args.count = 16
    args.num_slots = 1 << 20
    args.workspace = (workspace.ctypes.data + 15) // 16 * 16
    args.workspace_bytes = _native.ORDER_WORKSPACE_BYTES
    for mask in (args.mask, args.out_mask, args.mask + 15, args.out_mask - 1, args.out_mask + 15, maps.ctypes.data + 8,
                 out.ctypes.data + 511, scratch.ctypes.data - 15):
        with pytest.raises(_native.NativeCallError, match="scratch mask overlaps"):
            _native.order_link_maps_exact(args, scratch.ctypes.data, mask, 0)
