"""Append + decode on the balanced kernel (which for 16 bits at head_dim 128 puts
the new row into the last step itself): against reshape_and_cache followed by
the decode, at the edges of a 16-token step and of a block, with the row's slot
holding NaN before."""
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


@pytest.mark.parametrize("dtype,hq,hkv,d", [(torch.float32, 28, 4, 128), (torch.float32, 6, 6, 64),
                                            (torch.float16, 6, 6, 64), (torch.bfloat16, 32, 2, 64)])
def test_rows_of_shared_tables(dtype, hq, hkv, d):
    """Entries of one table at contexts c + 1 .. c + 4 (several new tokens of a
    sequence as rows of one batch): where the append is a launch of its own,
    every entry sees the rows that the entries before it append."""
    bs, base = 16, [700, 1499, 30]
    ctx = [c + i for c in base for i in (1, 2, 3, 4)]
    print(f"shared tables {hq}/{hkv} d={d} {dtype}", flush=True)
    k, v, own = make_paged_kv(d, [c + 4 for c in base], hkv, d, bs, dtype, spare_blocks=1)
    tables = [t for t in own for _ in range(4)]
    slots = [t[(c - 1) // bs] * bs + (c - 1) % bs for t, c in zip(tables, ctx)]
    for s in slots:  # what the slots hold before must not be read
        k.view(-1, hkv, d)[s] = float("nan")
        v.view(-1, hkv, d)[s] = float("nan")
    g = torch.Generator().manual_seed(4)
    n = len(ctx)
    q = torch.randn(n, hq, d, generator=g).to(dtype).to(DEV)
    kn = torch.randn(n, hkv, d, generator=g).to(dtype).to(DEV)
    vn = torch.randn(n, hkv, d, generator=g).to(dtype).to(DEV)
    bt, lens = padded_tables(tables).to(DEV), torch.tensor(ctx, dtype=torch.int32, device=DEV)
    k1, v1, k2, v2 = k.to(DEV), v.to(DEV), k.to(DEV), v.to(DEV)
    fused, ref = torch.empty_like(q), torch.empty_like(q)
    scale = 1.0 / math.sqrt(d)
    kernels.paged_attention_append(fused, q, k1, v1, bt, lens, bs, max(ctx), kn, vn, scale=scale)
    kernels.reshape_and_cache(kn, vn, k2, v2, torch.tensor(slots, dtype=torch.int64, device=DEV))
    kernels.paged_attention(ref, q, k2, v2, bt, lens, bs, max(ctx), scale=scale)
    torch.cuda.synchronize()
    for a, b in ((k1, k2), (v1, v2)):
        assert torch.equal(a.view(torch.uint8), b.view(torch.uint8))
    assert torch.isfinite(fused.float()).all()
    # the same kernel over the same values in the same order
    assert_attention_close(fused, ref, atol=0.0, rtol=0.0, what="rows of shared tables")
