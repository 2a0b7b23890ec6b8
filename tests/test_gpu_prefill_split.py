"""Chunked prefill split over workgroups (clv_chunked_prefill_split) at the
edges of its tiles and of its rules, against the oracle and against the
unsplit call."""
import math

import pytest
import torch

from cloverinfer_amd import _native, kernels
from oracle import attention as oa
from tests.test_gpu_prefill import DEV, build, oracle_prefill, run_prefill
from tests.helpers import assert_attention_close, padded_tables

pytestmark = pytest.mark.gpu

# fp32 sums of n terms are off by about sqrt(n) * 2^-24 of their scale; with
# the scores' own rounding (2^-22 at |score| < 8) that stays under 1e-5 of
# unit-variance values for the lengths used here.
F32_TOL = 1e-5


def check(got, ref, dtype, what):
    if dtype == torch.float32:
        assert_attention_close(got, ref, atol=F32_TOL, rtol=F32_TOL, what=what)
    else:
        assert_attention_close(got, ref, what=what)


# (cached, new): tile edges (32 / 64 tokens, 64 / 256 rows), one-token rows
# beside long chunks, no cached tokens, a single long item.
LENS = [([0], [511]), ([2000], [1]), ([31, 32, 33, 63, 64, 65], [33, 32, 31, 1, 64, 65]),
        ([1500, 0, 700, 3, 0, 999], [1, 300, 1, 257, 1, 37]), ([4100], [70]),
        ([200] * 9, [64] * 9)]


@pytest.mark.parametrize("lens", range(len(LENS)))
@pytest.mark.parametrize("hq,hkv,d,bs,dtype", [
    (12, 12, 64, 16, torch.float32), (28, 4, 128, 16, torch.float32), (64, 1, 128, 4, torch.float32),
    (28, 4, 128, 16, torch.bfloat16), (12, 12, 64, 32, torch.bfloat16), (8, 8, 128, 16, torch.float16),
])
def test_split_prefill_matches_oracle(lens, hq, hkv, d, bs, dtype):
    cached, new = LENS[lens]
    print(f"split prefill {cached}+{new} {hq}/{hkv} d={d} bs={bs} {dtype}", flush=True)
    q, k, v, tables, ctx, qsl = build(17 + lens, cached, new, hq, hkv, d, bs, dtype)
    scale = 1.0 / math.sqrt(d)
    got = run_prefill(q, k, v, tables, ctx, qsl, scale)
    refs = []
    for s in range(len(ctx)):
        kk, vv = oa.gather_context(k, v, tables[s], ctx[s])
        refs.append(oa.chunked_prefill_masked(q[qsl[s]:qsl[s + 1]], kk, vv, scale))
    check(got, torch.cat(refs), dtype, f"split prefill {cached}+{new}")


def native_call(q, k, v, tables, ctx, qsl, max_q, scale, split):
    """One C call, split or not, on the same arguments."""
    bt = padded_tables(tables).to(DEV)
    cl = torch.tensor(ctx, dtype=torch.int32, device=DEV)
    qs = torch.tensor(qsl, dtype=torch.int32, device=DEV)
    out = torch.full_like(q, float("nan"))
    a = _native.PrefillArgs()
    a.out, a.q, a.k_cache, a.v_cache = out.data_ptr(), q.data_ptr(), k.data_ptr(), v.data_ptr()
    a.block_tables, a.context_lens, a.query_start_loc = bt.data_ptr(), cl.data_ptr(), qs.data_ptr()
    a.q_stride_token, a.q_stride_head = q.stride(0), q.stride(1)
    a.out_stride_token, a.out_stride_head = out.stride(0), out.stride(1)
    a.kv_stride_block, a.kv_stride_token, a.kv_stride_head = k.stride()[:3]
    a.num_seqs, a.num_tokens, a.num_heads, a.num_kv_heads = len(ctx), q.shape[0], q.shape[1], k.shape[2]
    a.head_dim, a.block_size, a.max_blocks_per_seq = q.shape[2], k.shape[1], bt.shape[1]
    a.max_query_len, a.num_blocks, a.dtype, a.scale = max_q, k.shape[0], kernels._dtype_code(q), scale
    lib = _native.load()
    stream = torch.cuda.current_stream().cuda_stream
    if split:
        n = lib.clv_prefill_workspace_bytes(a)
        assert n > 0
        ws = torch.full((n,), 0xff, dtype=torch.uint8, device=DEV)  # NaN wherever it is read unset
        assert lib.clv_chunked_prefill_split(a, ws.data_ptr(), n - 1, stream) == _native.CLV_EWORKSPACE
        assert lib.clv_chunked_prefill_split(a, None, n, stream) == _native.CLV_EWORKSPACE
        _native.check(lib.clv_chunked_prefill_split(a, ws.data_ptr(), n, stream), "split")
    else:
        _native.check(lib.clv_chunked_prefill(a, stream), "whole")
    torch.cuda.synchronize()
    return out.cpu()


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("scale", [0.1, -0.1, 0.0])
def test_split_equals_whole(dtype, scale):
    """Same outputs as one workgroup per item: short contexts (fewer cached
    tokens than rows), rows past max_query_len (NaN), an unmapped block, a
    value that is infinite at a position that early rows do not see."""
    hq, hkv, d, bs = 14, 2, 128, 16
    cached, new = [900, 0, 0, 1300, 40], [1, 200, 90, 120, 75]
    q, k, v, tables, ctx, qsl = build(5, cached, new, hq, hkv, d, bs, dtype)
    ctx[2] = 50            # 90 rows, 50 tokens: the first 40 see nothing
    tables[3][20] = -1     # 16 tokens that are not there
    blk, off = tables[1][150 // bs], 150 % bs
    v[blk, off, 0, 3] = float("inf")
    qd, kd, vd = q.to(DEV), k.to(DEV), v.to(DEV)
    args = (qd, kd, vd, tables, ctx, qsl, 150, scale)  # sequence 1: rows 150.. are a caller error
    whole, split = native_call(*args, False), native_call(*args, True)
    assert torch.isnan(split[qsl[1] + 150:qsl[2]]).all()
    assert not split[qsl[2]:qsl[2] + 40].any()
    fin = torch.isfinite(whole)
    assert torch.equal(fin, torch.isfinite(split))
    if dtype == torch.float32:  # rows before the infinity are untouched by it
        assert fin[qsl[1]:qsl[1] + 150].all()
    check(torch.where(fin, split, 0), torch.where(fin, whole, 0), dtype, f"split, scale {scale}")
