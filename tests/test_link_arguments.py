"""The native check-and-fill of link and write-back argument blocks: it takes a
call exactly where the Python checks support it (or leaves it to them), and
fills what they fill."""

from __future__ import annotations

import ctypes
import os
import subprocess
import sys
from pathlib import Path

import pytest
import torch

from legolink_amd import _link_arguments, _native, kv_link
from legolink_amd.rope import build_cos_sin_cache


def _inputs(device, *, layers=3, slots=50, heads=2, kdim=64, vdim=64, tokens=20, source=False):
    def buffers(rows, dim):
        return [torch.zeros(rows, heads, dim, dtype=torch.bfloat16, device=device) for _ in range(layers)]

    index = torch.arange(tokens, device=device)
    return {"keys": buffers(slots, kdim), "values": buffers(slots, vdim),
            "source_keys": buffers(33, kdim) if source else [], "source_values": buffers(33, vdim) if source else [],
            "src": index, "dst": index + 20, "local": index.clone(), "global": index + 3,
            "table": build_cos_sin_cache(64, kdim).to(device), "mask": None, "rotary": kdim}


def _fill(inputs):
    args = _native.LinkArgs()
    tables = (ctypes.c_void_p * (4 * max(1, len(inputs["keys"]))))()
    filled = _link_arguments.fill_link(
        ctypes.addressof(args), ctypes.addressof(tables), inputs["keys"], inputs["values"], inputs["source_keys"],
        inputs["source_values"], inputs["src"], inputs["dst"], inputs["local"], inputs["global"], inputs["table"],
        inputs["mask"], inputs["rotary"])
    return filled, args, tables


def _python(inputs):
    return kv_link._eligibility(
        inputs["keys"], inputs["values"], inputs["src"], inputs["dst"], inputs["local"], inputs["global"],
        inputs["table"], inputs["rotary"], inputs["mask"], inputs["source_keys"], inputs["source_values"])


def _changed(**changes):
    def apply(inputs):
        for name, change in changes.items():
            inputs[name] = change(inputs[name])
    return apply


def _layer(index, change):
    return lambda buffers: [change(b) if i == index else b for i, b in enumerate(buffers)]


FORMS = {
    "plain": lambda inputs: None,
    "uint8_mask": _changed(mask=lambda _: "uint8"),
    "bool_mask": _changed(mask=lambda _: "bool"),
    "float_mask": _changed(mask=lambda _: "float32"),
    "short_mask": _changed(mask=lambda _: "short"),
    "strided_mask": _changed(mask=lambda _: "strided"),
    "int32_map": _changed(src=lambda t: t.int()),
    "int16_map": _changed(dst=lambda t: t.short()),
    "strided_map": _changed(local=lambda t: t.repeat_interleave(2)[::2]),
    "short_map": _changed(**{"global": lambda t: t[:-1]}),
    "no_tokens": _changed(src=lambda t: t[:0], dst=lambda t: t[:0], local=lambda t: t[:0], **{"global": lambda t: t[:0]}),
    "host_map": _changed(src=lambda t: t.cpu()),
    "host_layer": _changed(values=_layer(2, lambda b: b.cpu())),
    "flat_layer": _changed(keys=_layer(1, lambda b: b.flatten(1))),
    "other_rows": _changed(keys=_layer(1, lambda b: b[:-1])),
    "other_heads": _changed(values=lambda bs: [b[:, :1].contiguous() for b in bs]),
    "other_dtype": _changed(values=_layer(0, lambda b: b.half())),
    "fp32_pool": _changed(keys=lambda bs: [b.float() for b in bs], values=lambda bs: [b.float() for b in bs]),
    "strided_layer": _changed(keys=_layer(2, lambda b: b.transpose(0, 1).contiguous().transpose(0, 1))),
    "narrow_values": _changed(values=lambda bs: [b[..., :24].contiguous() for b in bs]),
    "wide_heads": _changed(keys=lambda bs: [b.repeat(1, 1, 5) for b in bs]),
    "odd_rotary": _changed(rotary=lambda r: 31),
    "zero_rotary": _changed(rotary=lambda r: 0),
    "wide_rotary": _changed(rotary=lambda r: r + 2),
    "half_rotary": _changed(rotary=lambda r: r // 2),
    "narrow_table": _changed(table=lambda t: t[:, :-2]),
    "flat_table": _changed(table=lambda t: t.flatten()),
    "strided_table": _changed(table=lambda t: t.repeat_interleave(2, 1)[:, ::2]),
    "padded_table": _changed(table=lambda t: torch.cat([t, t], 1)[:, :t.shape[1]]),
    "int_table": _changed(table=lambda t: t.int()),
    "bf16_table": _changed(table=lambda t: t.bfloat16()),
    "parameter_layer": _changed(keys=_layer(0, lambda b: torch.nn.Parameter(b, requires_grad=False))),
    "one_source_side": _changed(source_keys=lambda bs: []),
    "source_rows_differ": _changed(source_values=_layer(1, lambda b: b[:-1])),
    "source_dtype": _changed(source_keys=_layer(0, lambda b: b.half())),
}


@pytest.mark.gpu
@pytest.mark.parametrize("source", [False, True])
@pytest.mark.parametrize("form", FORMS)
def test_native_fill_agrees_with_the_python_checks(gpu_device, form, source):
    if "source" in form and not source:
        pytest.skip("needs a source pool")
    inputs = _inputs(gpu_device, source=source)
    FORMS[form](inputs)
    if isinstance(inputs["mask"], str):
        n = int(inputs["src"].numel())
        kind = inputs["mask"]
        mask = torch.zeros(2 * n, device=gpu_device)
        inputs["mask"] = {"uint8": mask[:n].byte(), "bool": mask[:n].bool(), "float32": mask[:n],
                          "short": mask[: n - 1].byte(), "strided": mask.byte()[::2]}[kind]
    assert form not in ("strided_table", "padded_table") or not inputs["table"].is_contiguous()
    filled, args, tables = _fill(inputs)
    expected = _python(inputs)
    # Taken only where the Python checks support the call; everything of this
    # list that they support is taken.
    assert filled == expected.supported, expected
    if not filled:
        return
    mask = inputs["mask"]
    want, keep = kv_link._link_args(
        inputs["keys"], inputs["values"], inputs["src"], inputs["dst"], inputs["local"], inputs["global"],
        inputs["table"], 3, inputs["rotary"], True, mask.view(torch.uint8) if mask is not None else None, 4, 0, 0, 0,
        inputs["source_keys"], inputs["source_values"])
    kv_link._set_link_options(args, 3, True, 4, 0, 0, 0, "fused", "auto")
    pointers = {"key_layers", "value_layers", "source_key_layers", "source_value_layers"}
    for name, _ in _native.LinkArgs._fields_:
        got, expect = getattr(args, name), getattr(want, name)
        if name not in pointers:
            assert got == expect, name
            continue
        assert (got is None) == (expect is None), name
        if got is not None:
            read = lambda address: list((ctypes.c_void_p * len(inputs["keys"])).from_address(address))
            assert read(got) == read(expect), name
    del keep


def test_native_fill_declines_what_is_no_tensor_list():
    """On the CPU: host tensors, wrong types and short calls are declined, never raised."""

    inputs = _inputs("cpu")
    assert not _fill(inputs)[0]
    for name, value in (("keys", ()), ("keys", []), ("keys", [1, 2, 3]), ("values", None), ("src", "text"),
                        ("table", None), ("rotary", "x")):
        broken = dict(_inputs("cpu"))
        broken[name] = value
        assert not _fill(broken)[0], name
    assert not _link_arguments.fill_link()
    assert not _link_arguments.fill_scatter(0, 0, [], [], None, None, None)


_IMPORT_WITHOUT = """
import sys, types
import torch
name = "legolink_amd._link_arguments"
if {sizes!r} is None:
    sys.modules[name] = None  # as if it were not built
else:
    sys.modules[name] = module = types.ModuleType(name)
    if {sizes!r}:
        module.TORCH_VERSION, module.LINK_ARGS_SIZE, module.SCATTER_ARGS_SIZE = {sizes!r}
    module.fill_link = module.fill_scatter = None  # never called
from legolink_amd import kv_link
assert kv_link._link_arguments is None
buffer, index = torch.zeros(8, 2, 64, dtype=torch.bfloat16), torch.arange(4)
print(kv_link.check_fused_kv_link_eligibility(
    key_buffer=buffer, value_buffer=buffer, source_slots=index, destination_slots=index, local_positions=index,
    global_positions=index, cos_sin_cache=torch.zeros(8, 64), rotary_dim=64).reason)
"""


@pytest.mark.parametrize("sizes", [None, (), ("1.0.0", None, None), (None, 8, None), (None, None, 1 << 20)])
@pytest.mark.parametrize("library,reason", [(None, "cuda_tensors_required"), ("/nowhere/lib.so", "hip_kv_link_not_built")])
def test_operator_imports_without_a_matching_module(sizes, library, reason):
    """An unbuilt tree, another torch or other argument blocks: the operator
    imports, keeps its reasons and takes the Python checks."""

    if sizes:
        own = (_link_arguments.TORCH_VERSION, ctypes.sizeof(_native.LinkArgs), ctypes.sizeof(_native.ScatterArgs))
        sizes = tuple(value if other is None else other for value, other in zip(own, sizes))
    package = Path(kv_link.__file__).resolve().parents[1]
    environment = {**os.environ, "PYTHONPATH": str(package)}
    if library is not None:
        environment["LEGOLINK_KV_LIBRARY"] = library
    done = subprocess.run([sys.executable, "-c", _IMPORT_WITHOUT.format(sizes=sizes)], env=environment,
                          capture_output=True, text=True, timeout=300)
    assert done.returncode == 0, done.stderr
    assert done.stdout.strip() == reason


def test_the_built_module_is_the_one_in_use():
    assert kv_link._link_arguments is _link_arguments
    assert _link_arguments.LINK_ARGS_SIZE == ctypes.sizeof(_native.LinkArgs)
    assert _link_arguments.SCATTER_ARGS_SIZE == ctypes.sizeof(_native.ScatterArgs)
    assert torch.__version__.split("+")[0] == _link_arguments.TORCH_VERSION


@pytest.mark.gpu
def test_python_checks_alone_link_and_write_back_the_same(gpu_device, monkeypatch):
    results = []
    for module in (_link_arguments, None):
        monkeypatch.setattr(kv_link, "_link_arguments", module)
        torch.manual_seed(3)
        inputs = _inputs(gpu_device, vdim=32)
        for buffer in (*inputs["keys"], *inputs["values"]):
            buffer.normal_()
        kv_link.fused_kv_link_layers_inplace(
            key_buffers=inputs["keys"], value_buffers=inputs["values"], source_slots=inputs["src"],
            destination_slots=inputs["dst"], local_positions=inputs["local"], global_positions=inputs["global"],
            cos_sin_cache=inputs["table"], prefix_token_count=2, rotary_dim=64, is_neox_style=True)
        rows = torch.ones(3, 5, 2, 64, dtype=torch.bfloat16, device=gpu_device)
        kv_link.scatter_kv_rows_inplace(
            key_buffers=inputs["keys"], value_buffers=inputs["values"], destination_slots=inputs["src"][:5],
            repaired_keys=rows, repaired_values=rows[..., :32].contiguous())
        results.append(torch.cat([buffer.flatten() for buffer in (*inputs["keys"], *inputs["values"])]))
    assert torch.equal(*results)


class _Subclass(torch.Tensor):
    pass


@pytest.mark.gpu
def test_tensor_subclasses_take_the_python_path(gpu_device):
    inputs = _inputs(gpu_device)
    inputs["keys"][1] = inputs["keys"][1].as_subclass(_Subclass)
    assert not _fill(inputs)[0] and _python(inputs).supported
    before = inputs["values"][0].clone()
    kv_link.fused_kv_link_layers_inplace(
        key_buffers=inputs["keys"], value_buffers=inputs["values"], source_slots=inputs["src"],
        destination_slots=inputs["dst"], local_positions=inputs["local"], global_positions=inputs["global"],
        cos_sin_cache=inputs["table"], prefix_token_count=0, rotary_dim=64, is_neox_style=True)
    assert torch.equal(inputs["values"][0][20:40], before[:20])


@pytest.mark.gpu
@pytest.mark.parametrize("layers,step", [(3, 1), (3, 2), (1, 1)])
@pytest.mark.parametrize("index", [torch.int32, torch.int64])
def test_native_write_back_fill_equals_the_python_one(gpu_device, monkeypatch, layers, step, index):
    """Every field of the block, for dense and layer-strided rows."""

    inputs = _inputs(gpu_device, layers=layers, vdim=32)
    keys = torch.randn(6, 5, 2, 64, device=gpu_device).to(torch.bfloat16)[::step][:layers]
    values = torch.randn(3, 5, 2, 32, device=gpu_device).to(torch.bfloat16)[:layers]
    slots = torch.tensor([3, 49, 0, 7, 20], device=gpu_device, dtype=index)
    args = _native.ScatterArgs()
    tables = (ctypes.c_void_p * (2 * layers))()
    assert _link_arguments.fill_scatter(ctypes.addressof(args), ctypes.addressof(tables), inputs["keys"],
                                        inputs["values"], slots, keys, values)
    prepared = []
    for module in (_link_arguments, None):
        monkeypatch.setattr(kv_link, "_link_arguments", module)
        prepared.append(kv_link.PreparedKVScatter(key_buffers=inputs["keys"], value_buffers=inputs["values"],
                                                  destination_slots=slots, repaired_keys=keys,
                                                  repaired_values=values))
    want = prepared[1]._args
    args.struct_size, args.waves_per_block = want.struct_size, want.waves_per_block
    for got in (args, prepared[0]._args):
        for name, _ in _native.ScatterArgs._fields_:
            field, expect = getattr(got, name), getattr(want, name)
            if name in ("key_layers", "value_layers"):
                field, expect = (list((ctypes.c_void_p * layers).from_address(a)) for a in (field, expect))
            assert field == expect, name


@pytest.mark.gpu
def test_write_back_forms(gpu_device):
    """A write-back with dense, layer-strided and refused repaired rows."""

    inputs = _inputs(gpu_device, vdim=32)
    rows = torch.randn(6, 5, 2, 64, device=gpu_device).to(torch.bfloat16)
    values = torch.randn(3, 5, 2, 32, device=gpu_device).to(torch.bfloat16)
    slots = torch.tensor([3, 49, 0, 7, 20], device=gpu_device, dtype=torch.int32)
    for repaired in (rows[:3], rows[::2]):
        kv_link.scatter_kv_rows_inplace(key_buffers=inputs["keys"], value_buffers=inputs["values"],
                                        destination_slots=slots, repaired_keys=repaired, repaired_values=values)
        for layer in range(3):
            assert torch.equal(inputs["keys"][layer][slots.long()], repaired[layer])
            assert torch.equal(inputs["values"][layer][slots.long()], values[layer])
    for bad, error in ((rows[:2], ValueError), (rows[:3].float(), RuntimeError), (rows[:3].transpose(1, 2), ValueError)):
        with pytest.raises(error):
            kv_link.scatter_kv_rows_inplace(key_buffers=inputs["keys"], value_buffers=inputs["values"],
                                            destination_slots=slots, repaired_keys=bad, repaired_values=values)
