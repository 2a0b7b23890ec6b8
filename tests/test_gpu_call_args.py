"""Argument blocks filled by the native host code against those the Python
checks fill, byte for byte, and the calls it leaves to them."""
import os

import pytest
import torch

from cloverinfer_amd import _native, build, kernels

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.fixture(scope="module", autouse=True)
def host():
    if not os.path.exists(build.HOST_EXT_PATH):
        build.build_host_ext()
    assert _native.load_host() is not None


def tensors(dtype, fp8=False):
    pool = torch.zeros(12, 16, 4, 128, dtype=kernels.FP8 if fp8 else dtype, device=DEV)
    q = torch.zeros(5, 2, 8, 128, dtype=dtype, device=DEV)[:, 1]  # strided rows
    out = torch.zeros(8, 5, 128, dtype=dtype, device=DEV).transpose(0, 1)
    k, v = pool[:6], pool[6:]
    bt = torch.zeros(5, 3, dtype=torch.int32, device=DEV)
    cl = torch.ones(5, dtype=torch.int32, device=DEV)
    return out, q, k, v, bt, cl


def both(monkeypatch, name, fn):
    """fn() with the native fill (which must have taken the call) and without."""
    used = []
    real = kernels._filled

    def spy(n, *a):
        r = real(n, *a)
        used.append((n, r is not None))
        return r

    monkeypatch.setattr(kernels, "_filled", spy)
    native = fn()
    assert used == [(name, True)], used
    monkeypatch.setattr(kernels, "_filled", lambda *a: None)
    python = fn()
    monkeypatch.setattr(kernels, "_filled", real)
    assert bytes(native) == bytes(python)


@pytest.mark.parametrize("dtype,fp8", [(torch.float32, False), (torch.float16, False),
                                       (torch.bfloat16, False), (torch.bfloat16, True)])
@pytest.mark.parametrize("scale", [None, 0.3])
def test_blocks_equal(monkeypatch, dtype, fp8, scale):
    out, q, k, v, bt, cl = tensors(dtype, fp8)
    both(monkeypatch, "fill_decode_args",
         lambda: kernels._decode_args(out, q, k, v, bt, cl, 16, 40, scale))
    key, value = q[:, :4], torch.zeros(5, 4, 128, dtype=dtype, device=DEV)
    slots = torch.zeros(5, dtype=torch.int64, device=DEV)
    both(monkeypatch, "fill_cache_args", lambda: kernels._cache_args(key, value, k, v, slots))
    if fp8:
        return
    a = _native.PrefillArgs()
    qsl = torch.arange(6, dtype=torch.int32, device=DEV)
    assert kernels._filled("fill_prefill_args", a, out, q, k, v, bt, cl, qsl, 7, scale) is a
    assert bytes(a) == bytes(kernels._prefill_args(out, q, k, v, bt, cl, qsl, 7, scale))


def test_refusals():
    out, q, k, v, bt, cl = tensors(torch.float16)

    class Sub(torch.Tensor):
        pass

    def fill(out=out, q=q, k=k, v=v, bt=bt, cl=cl, bs=16, mcl=40, scale=None):
        return kernels._filled("fill_decode_args", _native.DecodeArgs(), out, q, k, v, bt, cl, bs,
                               mcl, scale)

    assert fill() is not None
    for bad in (dict(q=q.as_subclass(Sub)), dict(out=out.float()), dict(cl=cl.cpu()),
                dict(cl=cl.long()), dict(bt=bt.t()), dict(bt=None), dict(bs=8), dict(mcl=-1),
                dict(mcl=4.0), dict(scale="x"), dict(k=k.transpose(2, 3)), dict(v=v[:5]),
                dict(q=q[:, :7], out=out[:, :7])):
        assert fill(**bad) is None, bad
    with pytest.raises(ValueError):
        kernels.paged_attention(out, q, k, v, bt, cl, 8, 40)
    with pytest.raises((RuntimeError, ValueError)):
        kernels.paged_attention(out, q, k, v, bt, cl.cpu(), 16, 40)
