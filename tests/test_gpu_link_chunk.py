"""The chunk kernel of the link: shapes that are whole 16-byte chunks but not
the vector kernel's (other rotary widths, K and V heads of different dims,
head dims that are no power of two, maps of mixed index types).

Every case runs on the chunk kernel and, asked for, on the generic kernel
(``KERNEL_GENERIC``), each bit-exact against the CPU oracle on the same inputs;
the launch record's kernel name says which one ran.  The limits of the choice
are checked on the CPU, from the arguments alone.
"""

from __future__ import annotations

import ctypes

import numpy as np
import pytest
import torch

from legolink_amd import _native, kv_link
from legolink_amd.rope import build_cos_sin_cache
from tests.gpu_helpers import bits, make_pool
from tests.test_gpu_link_parity import _run_case

B, H, F = torch.bfloat16, torch.float16, torch.float32
I64, I32 = torch.int64, torch.int32
MIXED = (torch.int64, torch.int32, torch.int32, torch.int64)

CHUNK, GENERIC = "kv_link_chunk_kernel", "kv_link_generic_kernel"

# name, kv dtype, table dtype, heads, key dim, value dim, rotary, neox, index, prefix, mask share, layers, tokens
CASES = [
    ("quarter_rotary", B, F, 4, 128, 128, 32, True, I64, 7, 0.1, 5, 130),
    ("narrow_values_full_rotary", B, F, 8, 128, 64, 128, True, I32, 0, 0.1, 4, 65),
    ("wide_values", H, F, 2, 64, 256, 64, True, I64, 3, 0.0, 3, 64),
    ("head_dim_96_five_heads_per_wave", B, F, 3, 96, 96, 96, True, I64, 2, 0.1, 9, 63),
    ("head_dim_80_partial", B, B, 4, 80, 80, 32, True, I64, 0, 0.1, 2, 151),
    ("head_dim_192_two_per_wave", H, B, 5, 192, 128, 64, True, I32, 11, 0.2, 3, 77),
    ("head_dim_248_two_per_wave", B, F, 3, 248, 8, 240, True, I64, 0, 0.1, 2, 33),
    ("head_dim_176_two_per_wave", B, H, 7, 176, 24, 176, True, I64, 1, 0.1, 2, 40),
    ("narrowest_gptj", B, F, 1, 8, 8, 8, False, I32, 0, 0.1, 6, 129),
    ("narrowest_neox", H, F, 5, 16, 8, 16, True, I64, 0, 0.1, 5, 100),
    ("gptj_partial_bf16_table", B, B, 3, 40, 24, 16, False, I64, 4, 0.1, 4, 151),
    ("gptj_24_fp16_table", H, H, 2, 128, 120, 24, False, I32, 0, 0.1, 2, 90),
    ("mixed_maps", B, F, 4, 128, 128, 128, True, MIXED, 6, 0.1, 3, 200),
    ("one_token", B, F, 4, 128, 128, 32, True, I64, 0, 0.0, 28, 1),
    ("all_prefix", B, F, 4, 128, 64, 128, True, I64, 150, 0.0, 2, 150),
    ("all_masked", B, F, 4, 128, 64, 128, True, I64, 0, 1.0, 2, 150),
    ("two_launches", B, F, 2, 128, 128, 32, True, I64, 3, 0.1, 70, 64),
]


def _as_parity_case(case, kernel):
    name, dtype, table, heads, kdim, vdim, rotary, neox, index, prefix, mask, layers, tokens = case
    return (name, dtype, table, heads, kdim, vdim, rotary, neox, kernel, index, prefix, mask, layers, tokens, "generic")


def _run_on(kernel_name, monkeypatch, device, case, kernel, **options):
    """``_run_case``, and the kernel that its launch record names."""

    records = []
    describe = kv_link.describe_link_launch
    monkeypatch.setattr(kv_link, "describe_link_launch",
                        lambda **arguments: records.append(describe(**arguments)) or records[-1])
    _run_case(device, _as_parity_case(case, kernel), **options)
    assert [record["kernel_name"] for record in records] == [kernel_name]


@pytest.mark.gpu
@pytest.mark.parametrize("kernel,kernel_name", [(_native.KERNEL_AUTO, CHUNK), (_native.KERNEL_GENERIC, GENERIC)],
                         ids=["auto", "generic"])
@pytest.mark.parametrize("rounding", ["fused", "eager"])
@pytest.mark.parametrize("case", CASES, ids=[case[0] for case in CASES])
def test_chunk_link_matches_oracle(gpu_device, monkeypatch, case, rounding, kernel, kernel_name):
    _run_on(kernel_name, monkeypatch, gpu_device, case, kernel, rounding=rounding)


@pytest.mark.gpu
@pytest.mark.parametrize("case", [CASES[0], CASES[5], CASES[10]], ids=lambda case: case[0])
def test_chunk_link_skips_and_counts_out_of_range_tokens(gpu_device, monkeypatch, case):
    _run_on(CHUNK, monkeypatch, gpu_device, case, _native.KERNEL_AUTO, corrupt=0.2)


@pytest.mark.gpu
@pytest.mark.parametrize("kdim,rotary", [(96, 96), (128, 32), (176, 176), (40, 32)])
def test_chunk_link_onto_the_tokens_own_slots(gpu_device, kdim, rotary):
    """Source slot == destination slot: each row turned in place, as the generic kernel does."""

    tokens, layers = 501, 6
    rng = np.random.default_rng(kdim)
    slots = torch.from_numpy(rng.permutation(tokens + 9)[:tokens]).to(gpu_device)
    local, position = (torch.from_numpy(rng.integers(0, 4000, tokens)).to(gpu_device) for _ in range(2))
    table = build_cos_sin_cache(4000, rotary).to(gpu_device)
    pools = []
    for kernel in (_native.KERNEL_AUTO, _native.KERNEL_GENERIC):
        keys, values = make_pool(layers, tokens + 9, 3, kdim, 64, torch.bfloat16, gpu_device, 5)
        kv_link.fused_kv_link_layers_inplace(
            key_buffers=keys, value_buffers=values, source_slots=slots, destination_slots=slots,
            local_positions=local, global_positions=position, cos_sin_cache=table, prefix_token_count=0,
            rotary_dim=rotary, is_neox_style=True, kernel=kernel)
        pools.append([bits(buffer) for buffer in (*keys, *values)])
    for got, want in zip(*pools):
        assert np.array_equal(got, want)


@pytest.mark.gpu
def test_unaligned_and_strided_forms_stay_on_the_generic_kernel(gpu_device, monkeypatch):
    """Buffers off 16 bytes and strided tables keep the general path, and its result."""

    _run_on(GENERIC, monkeypatch, gpu_device, CASES[0], _native.KERNEL_AUTO, cache_layout="strided")
    tokens = 33
    keys = [torch.randn(100 * 2 * 48 + 1, device=gpu_device).to(B)[1:].view(100, 2, 48) for _ in range(2)]
    values = [torch.randn(100 * 2 * 48 + 1, device=gpu_device).to(B)[1:].view(100, 2, 48) for _ in range(2)]
    aligned_keys, aligned_values = [k.clone() for k in keys], [v.clone() for v in values]
    assert keys[0].data_ptr() % 16 and not aligned_keys[0].data_ptr() % 16
    perm = torch.randperm(100, device=gpu_device)
    arguments = dict(source_slots=perm[:tokens], destination_slots=perm[tokens:2 * tokens],
                     local_positions=torch.arange(tokens, device=gpu_device),
                     global_positions=torch.arange(70, 70 + tokens, device=gpu_device),
                     cos_sin_cache=build_cos_sin_cache(200, 48).to(gpu_device), prefix_token_count=2,
                     rotary_dim=48, is_neox_style=True)
    for key_buffers, value_buffers, name in ((keys, values, GENERIC), (aligned_keys, aligned_values, CHUNK)):
        link = kv_link.PreparedKVLink(key_buffers=key_buffers, value_buffers=value_buffers, **arguments)
        assert link.launch["kernel_name"] == name
        link()
    for got, want in zip((*keys, *values), (*aligned_keys, *aligned_values)):
        assert np.array_equal(bits(got), bits(want))


def _name(*, kdim=128, vdim=128, rotary=32, neox=True, heads=2, tokens=8, table=torch.float32, table_row=None,
          table_column=1, off_buffer=0, off_table=0, index=torch.int64, kernel=_native.KERNEL_AUTO):
    """The kernel of a link with these arguments (no device, nothing is read)."""

    keys = [torch.zeros(64, heads, kdim, dtype=B) for _ in range(2)]
    values = [torch.zeros(64, heads, vdim, dtype=B) for _ in range(2)]
    maps = [torch.arange(8, dtype=torch.int64) for _ in range(4)]
    maps[1] = maps[1].to(index)
    args, keep = kv_link._link_args(keys, values, *maps, build_cos_sin_cache(32, rotary).to(table), 0, rotary, neox,
                                    None, 4, 0, kernel)
    args.num_tokens = tokens
    if table_row is not None:
        args.cos_sin_stride_row = table_row
    args.cos_sin_stride_col = table_column
    args.cos_sin_cache += off_table
    if off_buffer:
        ctypes.c_void_p.from_address(args.value_layers + 8).value += off_buffer
    name = _native.kv_link_kernel_name(args)
    del keep
    return name


@pytest.mark.parametrize("options,name", [
    (dict(), CHUNK),
    (dict(kernel=_native.KERNEL_GENERIC), GENERIC),
    (dict(kernel=_native.KERNEL_VECTOR), None),
    (dict(rotary=128), "kv_link_vec_kernel"),
    (dict(rotary=128, index=torch.int32), CHUNK),
    # Head dims and rotary halves (neox) or dims (GPT-J) in whole 16-byte chunks.
    (dict(kdim=8, rotary=8, neox=False), CHUNK),
    (dict(kdim=16, rotary=16), CHUNK),
    (dict(kdim=36), GENERIC),
    (dict(vdim=12), GENERIC),
    (dict(vdim=8), CHUNK),
    (dict(rotary=8), GENERIC),
    (dict(rotary=24), GENERIC),
    (dict(rotary=24, neox=False), CHUNK),
    (dict(rotary=20, neox=False), GENERIC),
    # Table rows and buffers on 16 bytes, unit column stride.
    (dict(table_row=36), CHUNK),
    (dict(table_row=34), GENERIC),
    (dict(table=torch.bfloat16, table_row=40), CHUNK),
    (dict(table=torch.bfloat16, table_row=36), GENERIC),
    (dict(table_column=2), GENERIC),
    (dict(off_table=8), GENERIC),
    (dict(off_table=16), CHUNK),
    (dict(off_buffer=2), GENERIC),
    (dict(off_buffer=8), GENERIC),
    (dict(off_buffer=16), CHUNK),
    # Fewer than 2^31 tokens and V chunks.
    (dict(vdim=8, heads=1, tokens=0x7fffffff), CHUNK),
    (dict(vdim=8, heads=1, tokens=0x80000000), GENERIC),
    (dict(vdim=8, heads=2, tokens=0x3fffffff), CHUNK),
    (dict(vdim=8, heads=2, tokens=0x40000000), GENERIC),
    (dict(vdim=64, heads=4, tokens=0x3ffffff), CHUNK),
    (dict(vdim=64, heads=4, tokens=0x4000000), GENERIC),
])
def test_the_chunk_kernel_takes_whole_chunks(options, name):
    assert _name(**options) == name
