"""The chunk kernel of the link: shapes that are whole 16-byte chunks but not
the vector kernel's (other rotary widths, K and V heads of different dims,
head dims that are no power of two, maps of mixed index types).

Every result is bit-exact against the CPU oracle, and equal to the generic
kernel's (``KERNEL_GENERIC``) on the same inputs.
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

from legolink_amd import _native, kv_link
from legolink_amd.rope import build_cos_sin_cache
from tests.gpu_helpers import bits, make_pool
from tests.test_gpu_link_parity import _run_case

pytestmark = pytest.mark.gpu

B, H, F = torch.bfloat16, torch.float16, torch.float32
I64, I32 = torch.int64, torch.int32
MIXED = (torch.int64, torch.int32, torch.int32, torch.int64)

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


@pytest.mark.parametrize("rounding", ["fused", "eager"])
@pytest.mark.parametrize("case", CASES, ids=[case[0] for case in CASES])
def test_chunk_link_matches_oracle(gpu_device, case, rounding):
    _run_case(gpu_device, _as_parity_case(case, _native.KERNEL_AUTO), rounding=rounding)


@pytest.mark.parametrize("case", [CASES[0], CASES[5], CASES[10]], ids=lambda case: case[0])
def test_chunk_link_skips_and_counts_out_of_range_tokens(gpu_device, case):
    _run_case(gpu_device, _as_parity_case(case, _native.KERNEL_AUTO), corrupt=0.2)


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


def test_unaligned_and_strided_forms_stay_on_the_generic_kernel(gpu_device):
    """Buffers or table rows off 16 bytes and strided tables keep the general path's result."""

    case = _as_parity_case(CASES[0], _native.KERNEL_AUTO)
    _run_case(gpu_device, case, cache_layout="strided")
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
    kv_link.fused_kv_link_layers_inplace(key_buffers=keys, value_buffers=values, **arguments)
    kv_link.fused_kv_link_layers_inplace(key_buffers=aligned_keys, value_buffers=aligned_values, **arguments)
    for got, want in zip((*keys, *values), (*aligned_keys, *aligned_values)):
        assert np.array_equal(bits(got), bits(want))
