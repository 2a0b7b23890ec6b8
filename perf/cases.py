"""The attention work that a serving program has this package do, as measurable cases.

Every case is one call of a public entry point of ``cloverinfer_amd.kernels``
on pools, block tables and rows that already lie on the GPU:

* ``decode``: one query row per sequence over its paged context
  (``paged_attention``), with fp32/fp16/bf16 pools or fp8 pools with scales;
* ``append_decode``: the append-then-attend step of the AttentionNode
  (``paged_attention_append``): new key/value rows written, then attended;
* ``prefill``: causal attention of each sequence's new rows over its paged
  context (``chunked_prefill``);
* ``append``: new key/value rows into the pools (``reshape_and_cache``).

Head shapes are those of the benchmark's workloads: 12/12 heads of 64
(OPT-125m), 32/32 of 128 (Llama-7B), 28/4 of 128 (Qwen2.5-7B) and 32/8 of 128.
A case holds plain values only; its sequence lengths follow from them, its
tensors' contents from the seed.
"""
import math
import random

import torch

from cloverinfer_amd import kernels

_DTYPES = {"float32": torch.float32, "float16": torch.float16, "bfloat16": torch.bfloat16}
_HEADS = [(12, 12, 64), (32, 32, 128), (28, 4, 128), (32, 8, 128)]
_DEV = "cuda"

# Most work of one drawn case: those of the largest listed ones.
_MAX_BYTES = 2.1e9
_MAX_FLOPS = {"float32": 2.5e10, "float16": 2.9e11, "bfloat16": 2.9e11}


def _case(name, op, heads, dtype, seqs, cached, new=(1, 1), block=16, partition=0, pool="",
          lens=0, ones=0.0):
    """cached / new: the range of each sequence's cached and new tokens
    (uniform, drawn from ``lens``); ones: share of the sequences that bring a
    single new token instead (decode rows of a mixed step). pool "fp8": e4m3 pools under ``dtype``
    queries. partition: split-K tokens, 0 leaves the schedule to the package."""
    c = {"op": op, "hq": heads[0], "hkv": heads[1], "d": heads[2], "dtype": dtype, "pool": pool,
         "seqs": seqs, "cached_lo": cached[0], "cached_hi": cached[1], "new_lo": new[0],
         "new_hi": new[1], "block": block, "partition": partition, "lens": lens, "ones": ones}
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # The smallest step: OPT-125m in fp32 (the reference's default dtype),
        # eight short chats, one layer's append and attention. Launch latency.
        _case("append_decode_opt125m_f32", "append_decode", (12, 12, 64), "float32", 8, (127, 127)),
        # A few interactive chats of a GQA 7B model, one layer of a token step.
        _case("decode_few_bf16", "decode", (28, 4, 128), "bfloat16", 4, (150, 3900), lens=11),
        # The benchmark's headline: a full ragged batch of a GQA 7B model.
        _case("decode_ragged_bf16", "decode", (28, 4, 128), "bfloat16", 128, (256, 8192), lens=3),
        # The same batch over fp8 pools, the option that halves the cache.
        _case("decode_ragged_fp8", "decode", (28, 4, 128), "bfloat16", 128, (256, 8192), lens=3,
              pool="fp8"),
        # An MHA 7B model at a fixed context, fp16: the most bytes per token.
        _case("decode_mha_f16", "decode", (32, 32, 128), "float16", 64, (2048, 2048)),
        # Long documents: 32K contexts, split-K with its merge.
        _case("decode_long_f16", "decode", (32, 8, 128), "float16", 16, (32768, 32768),
              partition=512),
        # The AttentionNode's step with fp32 payloads and pools.
        _case("append_decode_gqa_f32", "append_decode", (28, 4, 128), "float32", 16, (255, 4095),
              lens=5),
        # The benchmark's chunked prefill: 512-token chunks over 4096 cached.
        _case("prefill_chunks_bf16", "prefill", (32, 8, 128), "bfloat16", 8, (4096, 4096),
              (512, 512)),
        # A mixed step of continuous batching: ragged prompt chunks beside
        # sequences that bring one token each, over ragged cached contexts.
        _case("prefill_mixed_bf16", "prefill", (28, 4, 128), "bfloat16", 24, (0, 6000), (1, 300),
              lens=7, ones=0.6),
        # One user's new prompt on an MHA 7B model: time to the first token.
        _case("prefill_prompt_f16", "prefill", (32, 32, 128), "float16", 1, (0, 0), (777, 777)),
        # Prompts of OPT-125m in fp32.
        _case("prefill_opt125m_f32", "prefill", (12, 12, 64), "float32", 8, (0, 0), (17, 512),
              lens=9),
        # The cache write in front of a prefill: eight 512-token chunks,
        # quantised into fp8 pools.
        _case("append_fp8", "append", (32, 8, 128), "bfloat16", 8, (0, 4096), (512, 512), lens=2,
              pool="fp8"),
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.49)))))))


def draw(rng):
    while True:
        op = rng.choice(["decode", "decode", "append_decode", "prefill", "prefill", "append"])
        heads = rng.choice(_HEADS)
        dtype = rng.choice(["float32", "float16", "bfloat16"])
        block = rng.choice([16, 16, 16, 32])
        lens = rng.randrange(1 << 20)
        pool, partition, new, ones = "", 0, (1, 1), 0.0
        if op in ("decode", "append") and dtype != "float32" and heads[2] == 128 \
                and rng.random() < 0.3:
            pool = "fp8"
        if op in ("decode", "append_decode"):
            seqs = _log_int(rng, 1, 128)
            hi = _log_int(rng, 100, 32768 if seqs <= 16 else 8192)
            cached = (max(1, int(hi * rng.uniform(0.03, 1.0))), hi)
            if op == "decode" and not pool and hi > 8192:
                partition = rng.choice([0, 512])
        elif op == "prefill":
            seqs = _log_int(rng, 1, 16)
            hi = _log_int(rng, 17, 1024)
            new = (max(1, int(hi * rng.uniform(0.01, 1.0))), hi)
            hi = rng.choice([0, _log_int(rng, 32, 8192)])
            cached = (int(hi * rng.uniform(0.0, 1.0)), hi)
            ones = rng.choice([0.0, 0.0, round(rng.random(), 2)])
        else:
            seqs = _log_int(rng, 1, 64)
            hi = _log_int(rng, 16, 1024)
            new = (max(1, int(hi * rng.uniform(0.01, 1.0))), hi)
            cached = (0, 512)
        c = _case("", op, heads, dtype, seqs, cached, new, block, partition, pool, lens, ones)
        w = work(c)
        if w["bytes"] <= _MAX_BYTES and w["flops"] <= _MAX_FLOPS[dtype] and _pool_bytes(c) <= 6e9 \
                and (op not in ("append", "append_decode") or _pool_bytes(c) <= 4e8):
            return c


# ------------------------------------------------------------------ lengths
def _lens(case):
    """(cached tokens, new tokens) of every sequence; decode cases attend to
    ``cached`` tokens, append_decode to ``cached`` + 1."""
    r = random.Random(case["lens"] * 1000003 + case["seqs"])
    cached = [r.randint(case["cached_lo"], case["cached_hi"]) for _ in range(case["seqs"])]
    new = [r.randint(case["new_lo"], case["new_hi"]) for _ in range(case["seqs"])]
    new = [1 if r.random() < case["ones"] else n for n in new]
    if case["op"] == "decode":
        new = [0] * case["seqs"]
    return cached, new


def _contexts(case):
    return [c + n for c, n in zip(*_lens(case))]


def _eb(case):
    return 1 if case["pool"] == "fp8" else 4 if case["dtype"] == "float32" else 2


def _num_blocks(case):
    return math.ceil(1.1 * sum(max(1, math.ceil(c / case["block"])) for c in _contexts(case))) + 1


def _pool_bytes(case):
    return 2 * _num_blocks(case) * case["block"] * case["hkv"] * case["d"] * _eb(case)


def work(case):
    """K/V once per kv head, q and out once, new rows read and written once."""
    cached, new = _lens(case)
    ctx = _contexts(case)
    hq, hkv, d, op = case["hq"], case["hkv"], case["d"], case["op"]
    eb, qb = _eb(case), 4 if case["dtype"] == "float32" else 2
    tables = 4 * sum(math.ceil(c / case["block"]) for c in ctx) + 4 * len(ctx)
    if op == "append":
        return {"bytes": sum(new) * (2 * hkv * d * (qb + eb) + 8), "flops": 0}
    if op == "prefill":
        keys = sum(n * c + n * (n + 1) // 2 for c, n in zip(cached, new))
        rows = sum(new)
        return {"bytes": 2 * sum(ctx) * hkv * d * eb + 2 * rows * hq * d * qb + tables,
                "flops": 4 * keys * hq * d}
    b = 2 * sum(ctx) * hkv * d * eb + 2 * len(ctx) * hq * d * qb + tables
    if op == "append_decode":
        b += 2 * len(ctx) * hkv * d * eb
    return {"bytes": b, "flops": 4 * sum(ctx) * hq * d}


def tolerance(case):
    """Two correct implementations differ by the order of fp32 sums and, for
    16-bit outputs, by the rounding of the result (half an ulp: 2^-9 bf16,
    2^-12 fp16) and of the attention weights."""
    if case["op"] == "append":
        return "exact"  # copies, and one defined rounding to e4m3
    return {"float32": {"rel": 1e-5, "max": 1e-4},
            "float16": {"rel": 1e-3, "max": 1e-2},
            "bfloat16": {"rel": 8e-3, "max": 4e-2}}[case["dtype"]]


# ------------------------------------------------------------------ tensors
def _randn(shape, dtype, gen):
    return torch.randn(shape, generator=gen, device=_DEV, dtype=dtype)


def _tables(case, seed):
    """Block tables as a pool in use has them: physical blocks in no order."""
    need = [max(1, math.ceil(c / case["block"])) for c in _contexts(case)]
    g = torch.Generator().manual_seed(seed)
    perm = torch.randperm(_num_blocks(case), generator=g).to(torch.int32)
    table = torch.full((len(need), max(need)), -1, dtype=torch.int32)
    pos = 0
    for i, n in enumerate(need):
        table[i, :n] = perm[pos:pos + n]
        pos += n
    return table


def prepare(case, seed):
    dtype = _DTYPES[case["dtype"]]
    hq, hkv, d, bs, op = case["hq"], case["hkv"], case["d"], case["block"], case["op"]
    cached, new = _lens(case)
    ctx = _contexts(case)
    gen = torch.Generator(device=_DEV).manual_seed(seed)
    table = _tables(case, seed)
    st = {"case": case, "table": table.to(_DEV), "ctx": torch.tensor(ctx, dtype=torch.int32).to(_DEV),
          "max_ctx": max(ctx), "k_scale": None, "v_scale": None}
    shape = (_num_blocks(case), bs, hkv, d)
    if case["pool"] == "fp8":
        st["k_scale"] = torch.rand(hkv, generator=gen, device=_DEV) * 0.01 + 0.01
        st["v_scale"] = torch.rand(hkv, generator=gen, device=_DEV) * 0.01 + 0.01
    pools = []
    for name in ("k_scale", "v_scale"):
        if op == "append":  # the cache before the write: empty slots
            pools.append(torch.zeros(shape, dtype=torch.float8_e4m3fn if st[name] is not None
                                     else dtype, device=_DEV))
        elif st[name] is not None:
            x = _randn(shape, torch.bfloat16, gen) / st[name].to(torch.bfloat16).view(1, 1, -1, 1)
            pools.append(x.clamp(-448, 448).to(torch.float8_e4m3fn))
        else:
            pools.append(_randn(shape, dtype, gen))
    st["k"], st["v"] = pools
    rows = sum(new) if op in ("prefill", "append") else case["seqs"]
    if op != "append":
        st["q"] = _randn((rows, hq, d), dtype, gen)
        st["out"] = torch.empty_like(st["q"])
    if op in ("append", "append_decode"):
        st["key"] = _randn((rows, hkv, d), dtype, gen)
        st["value"] = _randn((rows, hkv, d), dtype, gen)
    if op == "append":
        slots = []
        for i, (c, n) in enumerate(zip(cached, new)):
            p = torch.arange(c, c + n)
            slots.append(table[i, p // bs].to(torch.int64) * bs + p % bs)
        st["slots"] = torch.cat(slots).to(_DEV)
    if op == "prefill":
        qsl = [0]
        for n in new:
            qsl.append(qsl[-1] + n)
        st["qsl"] = torch.tensor(qsl, dtype=torch.int32).to(_DEV)
        st["max_new"] = max(new)
    return st


def run(st):
    case = st["case"]
    op, bs = case["op"], case["block"]
    if op == "decode":
        kernels.paged_attention(st["out"], st["q"], st["k"], st["v"], st["table"], st["ctx"], bs,
                                st["max_ctx"], partition_size=case["partition"] or None,
                                k_scale=st["k_scale"], v_scale=st["v_scale"])
        return st["out"]
    if op == "append_decode":
        kernels.paged_attention_append(st["out"], st["q"], st["k"], st["v"], st["table"],
                                       st["ctx"], bs, st["max_ctx"], st["key"], st["value"])
        return st["out"], st["k"], st["v"]
    if op == "prefill":
        kernels.chunked_prefill(st["out"], st["q"], st["k"], st["v"], st["table"], st["ctx"],
                                st["qsl"], st["max_new"])
        return st["out"]
    kernels.reshape_and_cache(st["key"], st["value"], st["k"], st["v"], st["slots"],
                              k_scale=st["k_scale"], v_scale=st["v_scale"])
    if case["pool"] == "fp8":
        return st["k"].view(torch.uint8), st["v"].view(torch.uint8)
    return st["k"], st["v"]


# ------------------------------------------------------------------ 64 bits
def exact(case, seed):
    if case["op"] == "append":
        return None  # bytes moved or rounded once; nothing summed
    st = prepare(case, seed)
    hq, hkv, d, op = case["hq"], case["hkv"], case["d"], case["op"]
    group = hq // hkv
    cached, new = _lens(case)
    out = torch.zeros(st["q"].shape, dtype=torch.float64, device=_DEV)
    row = 0
    for s, c in enumerate(_contexts(case)):
        blocks = st["table"][s, :max(1, math.ceil(c / case["block"]))].long()
        k = st["k"][blocks].reshape(-1, hkv, d)[:c].double()
        v = st["v"][blocks].reshape(-1, hkv, d)[:c].double()
        if case["pool"] == "fp8":
            k = k * st["k_scale"].double().view(1, -1, 1)
            v = v * st["v_scale"].double().view(1, -1, 1)
        n = new[s] if op == "prefill" else 1
        if op == "append_decode":
            k[c - 1], v[c - 1] = st["key"][s].double(), st["value"][s].double()
        q = st["q"][row:row + n].double()
        hidden = None
        if op == "prefill":
            last = torch.arange(c - n, c, device=_DEV).view(-1, 1).repeat(1, group).reshape(-1, 1)
            hidden = torch.arange(c, device=_DEV).view(1, -1) > last
        for h in range(hkv):
            qh = q[:, h * group:(h + 1) * group].reshape(n * group, d)
            x = (qh @ k[:, h].t().contiguous()) / math.sqrt(d)
            if hidden is not None:
                x.masked_fill_(hidden, -math.inf)
            out[row:row + n, h * group:(h + 1) * group] = \
                (torch.softmax(x, dim=-1) @ v[:, h].contiguous()).view(n, group, d)
        row += n
    return (out, None, None) if op == "append_decode" else out
