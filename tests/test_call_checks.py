"""Checks that the tensor-level entry points make on the host before anything
is launched, on CPU tensors (with the device check alone taken out)."""
import os
import types

import pytest
import torch

from cloverinfer_amd import _native, build, kernels


@pytest.fixture(autouse=True)
def cpu_tensors(monkeypatch):
    monkeypatch.setattr(kernels, "_require_device", lambda *t: t[0].device)


def tensors(dtype, pool_dtype, n=3, hq=8, hkv=2, d=128, bs=16):
    q = torch.zeros(n, hq, d, dtype=dtype)
    k = torch.zeros(6, bs, hkv, d).to(pool_dtype)
    bt = torch.zeros(n, 2, dtype=torch.int32)
    cl = torch.ones(n, dtype=torch.int32)
    return torch.empty_like(q), q, k, k.clone(), bt, cl


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_fp8_pools_only_where_a_kernel_reads_them(dtype):
    """Calls whose kernels read 16- or 32-bit pools refuse fp8 ones: read as
    16-bit elements they end past the pools."""
    out, q, k, v, bt, cl = tensors(dtype, kernels.FP8)
    qsl = torch.arange(4, dtype=torch.int32)
    with pytest.raises(ValueError):
        kernels.chunked_prefill(out, q, k, v, bt, cl, qsl, 1)
    new = torch.zeros(3, 2, 128).to(kernels.FP8)
    with pytest.raises(NotImplementedError):
        kernels.paged_attention_append(out, q, k, v, bt, cl, 16, 32, new, new)
    with pytest.raises(NotImplementedError):
        kernels.SplitAppendDecode(out, q, k, v, bt, cl, 16, 32)
    # a pool of the queries' dtype passes the same checks
    out, q, k, v, bt, cl = tensors(dtype, dtype)
    kernels._prefill_args(out, q, k, v, bt, cl, qsl, 1, None)
    kernels.AppendDecodeLaunch(out, q, k, v, bt, cl, 16, 32, new.to(dtype), new.to(dtype))
    kernels.SplitAppendDecode(out, q, k, v, bt, cl, 16, 32)


def test_host_module_of_another_layout_fills_nothing():
    """The native fills write whole argument blocks at an address: a module
    compiled for another layout of them must not be called."""
    if not os.path.exists(build.HOST_EXT_PATH):
        build.build_host_ext()
    host = _native.load_host()
    assert host.call_args_layout == _native.call_args_layout()
    assert all(callable(getattr(host, n)) for n in _native._FILLS)
    wrong = list(host.call_args_layout)
    for i in range(len(wrong) + 1):
        layout = tuple(wrong[:i] + [wrong[i] + 8] + wrong[i + 1:]) if i < len(wrong) else None
        mod = types.SimpleNamespace(gather_rows=host.gather_rows, call_args_layout=layout,
                                    **{n: getattr(host, n) for n in _native._FILLS})
        if layout is None:
            del mod.call_args_layout  # built before there was one
        mod = _native._checked_host(mod)
        assert mod.gather_rows is host.gather_rows
        assert all(getattr(mod, n) is None for n in _native._FILLS), layout


@pytest.mark.parametrize("room", [True, False])
def test_prefill_without_room_for_a_workspace(monkeypatch, room):
    """A call that would be split needs no memory of its own to run: on a
    device that is full it takes the form without a workspace."""
    out, q, k, v, bt, cl = tensors(torch.float16, torch.float16)
    calls = []
    lib = types.SimpleNamespace(
        clv_prefill_workspace_bytes=lambda a: 4096,
        clv_chunked_prefill_split=lambda a, ws, n, s: calls.append(("split", n)) or 0,
        clv_chunked_prefill=lambda a, s: calls.append(("whole",)) or 0)

    def empty(*size, **kw):
        if not room:
            raise torch.cuda.OutOfMemoryError("no room")
        return torch.zeros(*size, **kw)

    monkeypatch.setattr(kernels._native, "load", lambda: lib)
    monkeypatch.setattr(kernels, "_stream", lambda dev: 0)
    monkeypatch.setattr(torch, "empty", empty)
    kernels.chunked_prefill(out, q, k, v, bt, cl, torch.arange(4, dtype=torch.int32), 1)
    assert calls == ([("split", 4096)] if room else [("whole",)])
