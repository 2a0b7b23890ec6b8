"""Append + decode on the balanced kernel, which puts the new row into the last
step itself: against reshape_and_cache followed by the decode, at the edges of
a 16-token step and of a block, with the row's slot holding NaN before."""
import math

import pytest
import torch

from cloverinfer_amd import kernels
from tests.helpers import assert_attention_close, make_paged_kv, padded_tables

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("hq,hkv,d,bs", [(28, 4, 128, 16), (6, 6, 64, 16), (32, 2, 64, 32), (8, 1, 128, 64)])
def test_append_in_kernel(dtype, hq, hkv, d, bs):
    ctx = [1, 2, 15, 16, 17, 31, 32, 33, 700, 0, 2049]
    print(f"append in kernel {hq}/{hkv} d={d} bs={bs} {dtype}", flush=True)
    k, v, tables = make_paged_kv(d + bs, ctx, hkv, d, bs, dtype, spare_blocks=1)
    slots = [t[(c - 1) // bs] * bs + (c - 1) % bs if c else -1 for t, c in zip(tables, ctx)]
    for s in slots:
        if s >= 0:
            k.view(-1, hkv, d)[s] = float("nan")
            v.view(-1, hkv, d)[s] = float("nan")
    tables[5][1 if bs == 16 else 0] = -1  # the new token's block is not mapped: nothing written
    slots[5] = -1
    g = torch.Generator().manual_seed(2)
    n = len(ctx)
    q = torch.randn(n, hq, d, generator=g).to(dtype).to(DEV)
    kn = torch.randn(n, hkv, d, generator=g).to(dtype).to(DEV)
    vn = torch.randn(n, hkv, d, generator=g).to(dtype).to(DEV)
    bt, lens = padded_tables(tables).to(DEV), torch.tensor(ctx, dtype=torch.int32, device=DEV)
    waves = kernels._native.load().clv_default_num_waves()
    k1, v1, k2, v2 = k.to(DEV), v.to(DEV), k.to(DEV), v.to(DEV)
    fused, ref = torch.empty_like(q), torch.empty_like(q)
    scale = 1.0 / math.sqrt(d)
    kernels.paged_attention_append(fused, q, k1, v1, bt, lens, bs, max(ctx), kn, vn, scale=scale,
                                   num_waves=waves)
    kernels.reshape_and_cache(kn, vn, k2, v2, torch.tensor(slots, dtype=torch.int64, device=DEV))
    kernels.paged_attention(ref, q, k2, v2, bt, lens, bs, max(ctx), scale=scale, num_waves=waves)
    torch.cuda.synchronize()
    for a, b in ((k1, k2), (v1, v2)):
        assert torch.equal(a.view(torch.uint8), b.view(torch.uint8))
    # the same kernel over the same values in the same order
    assert_attention_close(fused, ref, atol=0.0, rtol=0.0, what="append in kernel")
