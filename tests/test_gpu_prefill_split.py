"""Chunked prefill split over workgroups (clv_chunked_prefill_split) at the
edges of its tiles and of its rules, against the oracle and against the
unsplit call. Every test states which calls are split."""
import math

import pytest
import torch

from cloverinfer_amd import _native, kernels
from oracle import attention as oa
from tests.test_gpu_prefill import DEV, build, run_prefill
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


def oracle(q, k, v, tables, ctx, qsl, scale):
    refs = []
    for s in range(len(ctx)):
        kk, vv = oa.gather_context(k, v, tables[s], ctx[s])
        refs.append(oa.chunked_prefill_masked(q[qsl[s]:qsl[s + 1]], kk, vv, scale))
    return torch.cat(refs)


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
    # Tables of more than 1024 tokens in 16 bits, 192 in fp32, are split, up to
    # 1024 query tiles; the others here run the same tile edges unsplit.
    call = NativeCall(q.to(DEV), k.to(DEV), v.to(DEV), tables, ctx, qsl, max(new), scale)
    line, rows = (192, 64) if dtype == torch.float32 else (1024, 256)
    tiles = len(ctx) * math.ceil(max(new) / (rows // (hq // hkv)))
    assert (call.nbytes > 0) == (max(len(t) for t in tables) * bs > line and tiles <= 1024)
    got = run_prefill(q, k, v, tables, ctx, qsl, scale)
    check(got, oracle(q, k, v, tables, ctx, qsl, scale), dtype, f"split prefill {cached}+{new}")


class NativeCall:
    """One C call on device tensors, split or not."""

    def __init__(self, q, k, v, tables, ctx, qsl, max_q, scale, out=None):
        bt = padded_tables(tables).to(DEV)
        cl = torch.tensor(ctx, dtype=torch.int32, device=DEV)
        qs = torch.tensor(qsl, dtype=torch.int32, device=DEV)
        self.out = torch.full_like(q, float("nan")) if out is None else out
        a = self.a = kernels._prefill_args(self.out, q, k, v, bt, cl, qs, max_q, scale)
        self.held = (q, k, v, bt, cl, qs)
        self.lib = _native.load()
        self.nbytes = self.lib.clv_prefill_workspace_bytes(a)

    def whole(self):
        _native.check(self.lib.clv_chunked_prefill(self.a, torch.cuda.current_stream().cuda_stream),
                      "whole")
        torch.cuda.synchronize()
        return self.out.cpu()

    def split(self):
        lib, a, n = self.lib, self.a, self.nbytes
        stream = torch.cuda.current_stream().cuda_stream
        assert n > 0
        self.ws = torch.full((n,), 0xff, dtype=torch.uint8, device=DEV)  # NaN wherever it is read unset
        assert lib.clv_chunked_prefill_split(a, self.ws.data_ptr(), n - 1, stream) == _native.CLV_EWORKSPACE
        assert lib.clv_chunked_prefill_split(a, None, n, stream) == _native.CLV_EWORKSPACE
        _native.check(lib.clv_chunked_prefill_split(a, self.ws.data_ptr(), n, stream), "split")
        torch.cuda.synchronize()
        return self.out.cpu()

    def most_pieces(self, groups):
        """Pieces of the item cut into most, from the groups' descriptors."""
        cont = self.ws[:32 * groups].cpu().view(torch.int32).view(groups, 8)[:, 4].tolist()
        most = run = 1
        for c in cont:  # 1: the item goes on in the next group, 2: it ends here
            run += 1 if c else 0
            most = max(most, run)
            if c != 1:
                run = 1
        return most


def native_call(q, k, v, tables, ctx, qsl, max_q, scale, split):
    call = NativeCall(q, k, v, tables, ctx, qsl, max_q, scale)
    return call.split() if split else call.whole()


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


# Long items of few rows: the merge finds an item's last piece past the 64
# groups after its first, and weighs more partials than the lanes of a row.
@pytest.mark.parametrize("new", [1, 5])
@pytest.mark.parametrize("dtype,hq,hkv,d,tokens", [
    (torch.float32, 28, 4, 128, 9001), (torch.float32, 8, 4, 64, 9001),
    (torch.bfloat16, 14, 2, 128, 32768), (torch.float16, 8, 2, 64, 32768),
])
def test_split_items_of_many_pieces(dtype, hq, hkv, d, tokens, new):
    cached = tokens - 8 * new
    print(f"many pieces {cached}+{new} {hq}/{hkv} d={d} {dtype}", flush=True)
    q, k, v, tables, ctx, qsl = build(3, [cached], [new], hq, hkv, d, 16, dtype)
    scale = 1.0 / math.sqrt(d)
    call = NativeCall(q.to(DEV), k.to(DEV), v.to(DEV), tables, ctx, qsl, new, scale)
    got = call.split()
    per_cu = 1 if dtype != torch.float32 else 3 if d == 64 else 2
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    assert call.most_pieces(per_cu * (cus // 8 * 8)) > 65
    check(got, oracle(q, k, v, tables, ctx, qsl, scale), dtype, f"many pieces {cached}+{new}")


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("split", [False, True])
def test_prefill_strided_rows_and_head_major_pools(dtype, split):
    """q and out as views into wider rows, pools whose heads lie apart: bit for
    bit what contiguous tensors give, and nothing written beside out."""
    hq, hkv, d, bs = 14, 2, 128, 16
    q, k, v, tables, ctx, qsl = build(9, [1300, 0, 40], [3, 200, 75], hq, hkv, d, bs, dtype)
    qd, kd, vd = q.to(DEV), k.to(DEV), v.to(DEV)
    qkv = torch.full((q.shape[0], hq + 2 * hkv, d), float("nan"), dtype=dtype, device=DEV)
    qkv[:, :hq] = qd
    pools = [x.transpose(1, 2).contiguous().transpose(1, 2) for x in (kd, vd)]
    assert pools[0].stride(2) > pools[0].stride(1)
    wide = torch.full((q.shape[0], 3, hq, d), 7.0, dtype=dtype, device=DEV)
    wide[:, 1] = float("nan")
    plain = NativeCall(qd, kd, vd, tables, ctx, qsl, 200, 0.09)
    call = NativeCall(qkv[:, :hq], *pools, tables, ctx, qsl, 200, 0.09, out=wide[:, 1])
    assert plain.nbytes > 0 and call.nbytes == plain.nbytes
    ref = plain.split() if split else plain.whole()
    got = call.split() if split else call.whole()
    assert torch.equal(got, ref)
    check(got, oracle(q, k, v, tables, ctx, qsl, 0.09), dtype, "strided")
    assert (wide[:, 0] == 7.0).all() and (wide[:, 2] == 7.0).all()


# (sequences, longest chunk, heads, dtype, split): the table of the split holds
# 1024 (sequence, query tile) pairs, counted at the longest chunk's tiles.
@pytest.mark.parametrize("n,longest,hq,hkv,d,dtype,split", [
    (64, 576, 28, 4, 128, torch.bfloat16, True), (64, 577, 28, 4, 128, torch.bfloat16, False),
    (128, 288, 28, 4, 128, torch.bfloat16, True), (128, 289, 28, 4, 128, torch.bfloat16, False),
    (16, 576, 28, 4, 128, torch.float32, True), (16, 577, 28, 4, 128, torch.float32, False),
    (1024, 36, 28, 4, 64, torch.float16, True), (1025, 36, 28, 4, 64, torch.float16, False),
])
def test_split_item_limit(n, longest, hq, hkv, d, dtype, split):
    """One long chunk among sequences of one row, on both sides of the limit."""
    g = torch.Generator().manual_seed(n)
    cached = torch.randint(0, 60, (n,), generator=g).tolist()
    new = [1] * n
    cached[n // 2], new[n // 2] = 1100, longest
    print(f"{n} sequences, longest {longest}, {dtype}", flush=True)
    q, k, v, tables, ctx, qsl = build(n, cached, new, hq, hkv, d, 16, dtype)
    call = NativeCall(q.to(DEV), k.to(DEV), v.to(DEV), tables, ctx, qsl, longest, d ** -0.5)
    assert (call.nbytes > 0) == split
    got = call.split() if split else call.whole()
    check(got, oracle(q, k, v, tables, ctx, qsl, d ** -0.5), dtype, f"{n} sequences")


@pytest.mark.parametrize("n,split", [(8, False), (7, True)])
def test_equal_chunks_that_fill_rounds_are_not_split(n, split):
    """16-bit chunks of one length whose items fill whole rounds of the device
    run unsplit, whatever is cached before them."""
    hq, hkv, d = 16, 4, 64
    if torch.cuda.get_device_properties(0).multi_processor_count != 256:
        pytest.skip("8 x 8 tiles x 4 heads are whole rounds of 256 compute units")
    cached = [0, 2000, 64, 900, 1, 1500, 333, 0][:n]
    q, k, v, tables, ctx, qsl = build(12, cached, [512] * n, hq, hkv, d, 16, torch.bfloat16)
    call = NativeCall(q.to(DEV), k.to(DEV), v.to(DEV), tables, ctx, qsl, 512, d ** -0.5)
    assert (call.nbytes > 0) == split
    got = call.split() if split else call.whole()
    check(got, oracle(q, k, v, tables, ctx, qsl, d ** -0.5), torch.bfloat16, f"{n} equal chunks")


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_split_prefill_in_a_graph(dtype):
    """Captured with its workspace from the graph's pool: every replay equals
    the eager call, also on inputs changed between the replays."""
    hq, hkv, d = 28, 4, 128
    q, k, v, tables, ctx, qsl = build(21, [2500, 0, 700], [1, 90, 33], hq, hkv, d, 16, dtype)
    qd, kd, vd = q.to(DEV), k.to(DEV), v.to(DEV)
    bt, cl = padded_tables(tables).to(DEV), torch.tensor(ctx, dtype=torch.int32, device=DEV)
    qs, out, ref = torch.tensor(qsl, dtype=torch.int32, device=DEV), torch.empty_like(qd), torch.empty_like(qd)
    assert NativeCall(qd, kd, vd, tables, ctx, qsl, 90, d ** -0.5).nbytes > 0

    def call(dst):
        kernels.chunked_prefill(dst, qd, kd, vd, bt, cl, qs, 90)

    call(ref)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        call(out)
    for i in range(4):
        qd.mul_(-0.5 if i & 1 else 1.25)
        out.fill_(float("nan"))
        call(ref)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, ref), f"replay {i}"
