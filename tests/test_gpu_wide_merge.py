"""Balanced decode of small batches, whose rows have many partials each: the
merge with several waves per row against the oracle, on both sides of the
rule (partials per segment) that picks it, with and without a new token."""
import math

import pytest
import torch

from cloverinfer_amd import kernels
from oracle import attention as oa
from tests.helpers import assert_attention_close, make_paged_kv, padded_tables

pytestmark = pytest.mark.gpu
DEV = "cuda"


# 256 CUs x 4 waves: 1024 / head group segments-per-group; contexts of 1 and 17
# tokens leave most waves of a row's workgroup without a partial.
@pytest.mark.parametrize("ctx", [[1], [4097], [600, 17], [5000, 1, 0, 2300], [900] * 15, [700] * 17])
@pytest.mark.parametrize("hq,hkv,d,dtype", [(28, 4, 128, torch.bfloat16), (12, 12, 64, torch.float16),
                                            (28, 4, 128, torch.float32)])
def test_wide_merge(ctx, hq, hkv, d, dtype):
    bs = 16
    print(f"wide merge ctx={ctx} {hq}/{hkv} d={d} {dtype}", flush=True)
    k, v, tables = make_paged_kv(len(ctx) + d, [c + 1 for c in ctx], hkv, d, bs, dtype, spare_blocks=1)
    scale = 1.0 / math.sqrt(d)
    g = torch.Generator().manual_seed(3)
    q = torch.randn(len(ctx), hq, d, generator=g).to(dtype)
    qd, bt, lens = q.to(DEV), padded_tables(tables).to(DEV), torch.tensor(ctx, dtype=torch.int32).to(DEV)
    kd, vd = k.to(DEV), v.to(DEV)
    out = torch.full_like(qd, float("nan"))
    waves = kernels._native.load().clv_default_num_waves()
    kernels.paged_attention(out, qd, kd, vd, bt, lens, bs, max(ctx), scale=scale, num_waves=waves)
    torch.cuda.synchronize()
    assert_attention_close(out, oa.paged_decode(q, k, v, tables, ctx, scale), what="wide merge")

    kn = torch.randn(len(ctx), hkv, d, generator=g).to(dtype).to(DEV)
    vn = torch.randn(len(ctx), hkv, d, generator=g).to(dtype).to(DEV)
    slots = torch.tensor([t[c // bs] * bs + c % bs for t, c in zip(tables, ctx)],
                         dtype=torch.int64, device=DEV)
    sp = kernels.SplitAppendDecode(out, qd, kd, vd, bt, lens, bs, max(ctx), scale=scale, num_waves=waves)
    sp.partials()
    sp.reduce(kn, vn, slots)
    torch.cuda.synchronize()
    kf, vf = kd.view(-1, hkv, d), vd.view(-1, hkv, d)
    assert torch.equal(kf[slots], kn) and torch.equal(vf[slots], vn)
    ref = oa.paged_decode(q, kd.cpu(), vd.cpu(), tables, [c + 1 for c in ctx], scale)
    assert_attention_close(out, ref, what="wide merge with a new token")
