"""The attention layer's calls as a serving engine makes them, with what each cannot do without.

A case is one of two kinds:

  step     one engine step through one layer: n_decode sequences that bring one
           token each over ctx_lo..ctx_hi visible keys, and n_prefill sequences
           that bring new_lo..new_hi tokens over a cached prefix of
           prefix_lo..prefix_hi tokens (whole blocks).  PagedAttention.forward,
           or forward_fused (q/k norm, rotary embedding and KV write in front)
           where "fused" is set.
  handoff  KV blocks of every layer packed for another worker and unpacked into
           its pool: export_kv_blocks, then import_kv_blocks.

Lengths come from the case alone ("shape" seeds them), so that work(case) is
exact; block tables and values come from the seed given to prepare().  Pools
are random throughout, as a pool that earlier sequences have used is.
"""
from __future__ import annotations

import math
import random

import torch

from nanovllm_self_amd.kv_cache import (KVCacheConfig, SeqSlice, allocate_kv_cache, bind_kv_cache, build_context,
                                        export_kv_blocks, import_kv_blocks)
from nanovllm_self_amd.layers.attention import PagedAttention

HEAD_DIM = 128
EPS = 1e-6
MAX_POSITION = 40960
ELEM = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp8": torch.bfloat16, "int8": torch.bfloat16}
CODE = {"fp8": (torch.float8_e4m3fn, 448.0), "int8": (torch.int8, 127.0)}
MODE = {"bf16": "none", "fp16": "none", "fp8": "fp8_e4m3", "int8": "int8_mock"}


def _step(name, hq, hkv, kv, block=256, fused=False, n_decode=0, ctx=(1, 1), n_prefill=0, new=(1, 1), prefix=(0, 0),
          shape=0):
    case = {"kind": "step", "hq": hq, "hkv": hkv, "kv": kv, "block": block, "fused": fused, "n_decode": n_decode,
            "ctx_lo": ctx[0], "ctx_hi": ctx[1], "n_prefill": n_prefill, "new_lo": new[0], "new_hi": new[1],
            "prefix_lo": prefix[0], "prefix_hi": prefix[1], "shape": shape}
    return {"name": name, **case} if name else case


def listed():
    return [
        # One user's long conversation: a single row, decoded token by token.
        _step("decode_chat", 32, 8, "bf16", n_decode=1, ctx=(20011, 20011)),
        # A small model serving a few short conversations: the launch-bound end.
        _step("decode_small", 16, 8, "bf16", n_decode=8, ctx=(128, 1024), shape=1),
        # The same step through the fused entry, at a modest load.
        _step("decode_fused", 32, 8, "bf16", fused=True, n_decode=33, ctx=(500, 4100), shape=2),
        # The 8B shape under load with long contexts.
        _step("decode_8b", 32, 8, "bf16", n_decode=64, ctx=(2048, 8192), shape=3),
        # A large batch over an fp8 cache.
        _step("decode_fp8", 32, 8, "fp8", n_decode=256, ctx=(1024, 4096), shape=4),
        # Conversations of very different lengths over an int8 cache, the 32B shape.
        _step("decode_int8_ragged", 64, 8, "int8", n_decode=48, ctx=(256, 32768), shape=5),
        # New prompts of a small fp16 model, nothing cached.
        _step("prompts_fp16", 16, 8, "fp16", n_prefill=4, new=(40, 700), shape=6),
        # Follow-up turns: a few new tokens each over what the prefix cache holds.
        _step("prefix_hits", 32, 8, "bf16", n_prefill=6, new=(20, 300), prefix=(1024, 16384), shape=7),
        # Long prompts, some of them over shared prefixes: the compute-bound end.
        _step("prefill_8b", 32, 8, "bf16", n_prefill=16, new=(512, 4096), prefix=(0, 2048), shape=8),
        # Prompts over shared prefixes through the fused entry, fp8 cache of small blocks.
        _step("prefill_fused_fp8", 32, 8, "fp8", block=64, fused=True, n_prefill=4, new=(300, 2100), prefix=(0, 4096),
              shape=9),
        # A full step of the 32B shape: decode rows beside chunks of long prompts.
        _step("mixed_32b", 64, 8, "bf16", n_decode=128, ctx=(256, 32768), n_prefill=4, new=(2048, 2048),
              prefix=(0, 16384), shape=10),
        # One prompt's blocks handed from a prefill worker to a decode worker.
        {"name": "handoff", "kind": "handoff", "layers": 36, "hkv": 8, "kv": "bf16", "block": 256, "n_blocks": 16,
         "pool": 40},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _cost(case):
    w = work(case)
    return max(w["bytes"], w["flops"] / 50)


def _draw_any(rng):
    kind = rng.choice(("decode", "decode", "prompts", "prefix", "prefix", "mixed", "handoff"))
    hq, hkv = rng.choice(((16, 8), (32, 8), (32, 8), (64, 8), (8, 1)))  # the last: one rank of eight
    kv = rng.choice(("bf16", "bf16", "fp16", "fp8", "int8"))
    block = rng.choice((256, 256, 64))
    fused = kv != "fp16" and rng.random() < 0.3
    shape = rng.randrange(1 << 16)
    if kind == "handoff":
        n = _log_int(rng, 1, 32)
        return {"kind": "handoff", "layers": rng.choice((28, 36)), "hkv": hkv, "kv": kv, "block": block,
                "n_blocks": n, "pool": n + rng.randrange(1, 25)}
    lo = _log_int(rng, 64, 16384)
    ctx = (lo, min(32768, _log_int(rng, lo, 8 * lo)))
    new_lo = _log_int(rng, 2, 2048)
    new = (new_lo, min(4096, _log_int(rng, new_lo, 8 * new_lo)))
    top = _log_int(rng, block, 16384)
    prefix = (rng.choice((0, top // 8)), top)
    if kind == "decode":
        return _step("", hq, hkv, kv, block, fused, n_decode=_log_int(rng, 1, 256), ctx=ctx, shape=shape)
    if kind == "prompts":
        return _step("", hq, hkv, kv, block, fused, n_prefill=_log_int(rng, 1, 16), new=new, shape=shape)
    if kind == "prefix":
        return _step("", hq, hkv, kv, block, fused, n_prefill=_log_int(rng, 1, 16), new=new, prefix=prefix,
                     shape=shape)
    return _step("", hq, hkv, kv, block, fused, n_decode=_log_int(rng, 1, 128), ctx=ctx,
                 n_prefill=rng.randrange(1, 5), new=new, prefix=prefix, shape=shape)


def draw(rng):
    most = next(_cost(c) for c in listed() if c["name"] == "mixed_32b")
    while True:
        case = _draw_any(rng)
        if _cost(case) <= most:
            return case


# ------------------------------------------------------------------ lengths
def _lengths(case):
    """(new tokens, cached tokens) of every sequence, decode rows first."""
    rng = random.Random(case["shape"])
    bs = case["block"]
    out = [(1, _log_int(rng, case["ctx_lo"], case["ctx_hi"]) - 1) if case["ctx_hi"] > 16 * case["ctx_lo"]
           else (1, rng.randint(case["ctx_lo"], case["ctx_hi"]) - 1) for _ in range(case["n_decode"])]
    for _ in range(case["n_prefill"]):
        out.append((rng.randint(case["new_lo"], case["new_hi"]),
                    bs * (rng.randint(case["prefix_lo"], case["prefix_hi"]) // bs)))
    return out


def _elem_bytes(kv):
    """Bytes of one cached head row of one token, K and V together."""
    return 2 * HEAD_DIM * 2 if kv in ("bf16", "fp16") else 2 * (HEAD_DIM + 4)


def work(case):
    if case["kind"] == "handoff":
        moved = case["layers"] * case["n_blocks"] * case["block"] * case["hkv"] * _elem_bytes(case["kv"])
        return {"bytes": 4 * moved, "flops": 0}  # read and written on either side
    lens = _lengths(case)
    tokens = sum(n for n, _ in lens)
    cached = sum(p for _, p in lens)
    pairs = sum(n * p + n * (n + 1) // 2 for n, p in lens)
    row = _elem_bytes(case["kv"])
    nbytes = cached * case["hkv"] * row  # history read
    nbytes += tokens * case["hkv"] * (4 * HEAD_DIM + row)  # new k, v read and written to the cache
    nbytes += tokens * case["hq"] * 4 * HEAD_DIM  # q read, output written
    if case["fused"]:
        nbytes += tokens * 4 * HEAD_DIM  # the rotary table's row
    return {"bytes": nbytes, "flops": 4 * case["hq"] * HEAD_DIM * pairs}


def tolerance(case):
    """About four times what the calls are off by against sums in 64 bits, over
    the listed cases and two dozen drawn ones (rel: 2-norms; max: the largest
    value, over the output's root mean square or the value itself):
    bf16 2.4e-3 and 0.05; fp16 2.5e-4 and 2.8e-3; decode over codes 2.4e-3 and
    0.09.  Prefill over codes attends over their bf16 values, which moves the
    sharp scores of large keys: 5.3e-3 and 0.96."""
    if case["kind"] == "handoff":
        return "exact"
    if case["kv"] == "fp16":
        return {"rel": 1e-3, "max": 0.02}
    if case["kv"] in CODE:
        return {"rel": 2e-2, "max": 0.95} if case["n_prefill"] else {"rel": 1e-2, "max": 0.35}
    return {"rel": 1e-2, "max": 0.2}


# ------------------------------------------------------------------- inputs
def _quantise(x, kv):
    """Codes and fp32 scales [..., 1] of the last dimension's rows."""
    dtype, top = CODE[kv]
    x = x.float()
    scale = torch.clamp(x.abs().amax(dim=-1, keepdim=True) / top, min=1e-6)
    q = x / scale
    q = torch.clamp(torch.round(q), -top, top) if kv == "int8" else torch.clamp(q, -top, top)
    return q.to(dtype), scale


def _normal(shape, gen, kv):
    """N(0, 1) in the step's type; with a code cache 1 % of the values are eight times as large."""
    x = torch.randn(shape, generator=gen, device="cuda", dtype=ELEM[kv])
    if kv in CODE:
        x = torch.where(torch.rand(shape, generator=gen, device="cuda") < 0.01, x * 8, x)
    return x


def _fill_pool(cache, scales, gen, kv):
    """Random K and V in every block of a [2, L, NB, bs, Hkv, D] pool."""
    planes = cache.view(-1, *cache.shape[2:])
    for i in range(planes.shape[0]):
        step = max(1, (1 << 27) // planes[i][0].numel())
        for a in range(0, planes.shape[1], step):
            part = planes[i, a:a + step]
            x = _normal(part.shape, gen, kv)
            if kv in CODE:
                codes, sc = _quantise(x, kv)
                part.copy_(codes)
                scales.view(-1, *scales.shape[2:])[i, a:a + step].copy_(sc)
            else:
                part.copy_(x)


def _pool(layers, hkv, kv, block, num_blocks, gen):
    cfg = KVCacheConfig(dtype=ELEM[kv], kv_cache_dtype=ELEM[kv], attention_compute_dtype=ELEM[kv],
                        kv_cache_quant_mode=MODE[kv], block_size=block, num_blocks=num_blocks)
    cache, scales = allocate_kv_cache(layers, hkv, HEAD_DIM, cfg, "cuda")
    _fill_pool(cache, scales, gen, kv)
    return cfg, cache, scales


def _rope_table():
    inv = 1.0 / (1e6 ** (torch.arange(0, HEAD_DIM, 2, dtype=torch.float64, device="cuda") / HEAD_DIM))
    freqs = torch.arange(MAX_POSITION, dtype=torch.float64, device="cuda")[:, None] * inv
    return torch.cat((freqs.cos(), freqs.sin()), dim=-1).float().unsqueeze(1)


def prepare(case, seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    rng = random.Random(seed)
    kv, bs = case["kv"], case["block"]
    if case["kind"] == "handoff":
        _, src, src_sc = _pool(case["layers"], case["hkv"], kv, bs, case["pool"], gen)
        dst = torch.zeros_like(src)
        dst_sc = None if src_sc is None else torch.ones_like(src_sc)
        ids = [rng.sample(range(case["pool"]), case["n_blocks"]) for _ in range(2)]
        return {"case": case, "src": src, "src_sc": src_sc, "dst": dst, "dst_sc": dst_sc, "from": ids[0], "to": ids[1]}
    lens = _lengths(case)
    need = [-(-(n + p) // bs) for n, p in lens]
    num_blocks = sum(need) + max(1, sum(need) // 16)
    cfg, cache, scales = _pool(1, case["hkv"], kv, bs, num_blocks, gen)
    free = list(range(num_blocks))
    rng.shuffle(free)
    seqs = []
    for (n, p), m in zip(lens, need):
        seqs.append(SeqSlice(free[:m], p, n))
        del free[:m]
    attn = PagedAttention(case["hq"], case["hkv"], HEAD_DIM, dtype=ELEM[kv])
    bind_kv_cache([attn], cache, scales, cfg)
    tokens = sum(n for n, _ in lens)
    state = {"case": case, "attn": attn, "cache": cache, "scales": scales, "seqs": seqs,
             "ctx": build_context(seqs, bs, "cuda"),
             "q": _normal((tokens, case["hq"], HEAD_DIM), gen, "bf16").to(ELEM[kv]),
             "k": _normal((tokens, case["hkv"], HEAD_DIM), gen, kv),
             "v": _normal((tokens, case["hkv"], HEAD_DIM), gen, kv)}
    if case["fused"]:
        state["positions"] = torch.cat([torch.arange(p, p + n, device="cuda") for n, p in lens])
        state["qw"], state["kw"] = (1 + 0.1 * torch.randn(HEAD_DIM, generator=gen, device="cuda",
                                                          dtype=torch.bfloat16) for _ in range(2))
        state["table"] = _rope_table()
    return state


def run(state):
    if "src" in state:
        blocks, scales = export_kv_blocks(state["src"], state["src_sc"], state["from"])
        import_kv_blocks(state["dst"], state["dst_sc"], blocks, scales, state["to"])
        codes = state["case"]["kv"] == "fp8"
        return [blocks.view(torch.uint8) if codes else blocks, scales,
                state["dst"].view(torch.uint8) if codes else state["dst"], state["dst_sc"]]
    attn = state["attn"]
    if state["case"]["fused"]:
        out = attn.forward_fused(state["q"], state["k"], state["v"], state["positions"], state["qw"], state["kw"],
                                 EPS, state["table"], state["ctx"])
    else:
        out = attn.forward(state["q"], state["k"], state["v"], state["ctx"])
    cache = state["cache"]
    return [out, cache.view(torch.uint8) if cache.dtype == torch.float8_e4m3fn else cache, state["scales"]]


# -------------------------------------------------------------------- exact
def _norm_rope(x, w, table, positions):
    """RMSNorm and rotary embedding in 64 bits; the cached element type's rounding is left to the caller."""
    x = x.double()
    n = w.double() * x / torch.sqrt(x.square().mean(-1, keepdim=True) + EPS)
    cos, sin = table[positions, 0].double().unsqueeze(1).chunk(2, dim=-1)
    a, b = n.chunk(2, dim=-1)
    return torch.cat((a * cos - b * sin, b * cos + a * sin), dim=-1)


def exact(case, seed):
    """The attention output in 64 bits over the cache as stored (its element
    type's rounding, or its codes and scales); None for the caches."""
    if case["kind"] == "handoff":
        return None
    s = prepare(case, seed)
    kv, bs, hkv, g = case["kv"], case["block"], case["hkv"], case["hq"] // case["hkv"]
    q, k, v = s["q"].double(), s["k"], s["v"]
    if case["fused"]:
        q = _norm_rope(s["q"], s["qw"], s["table"], s["positions"])
        k = _norm_rope(s["k"], s["kw"], s["table"], s["positions"]).to(torch.bfloat16)
    slots = s["ctx"].slot_mapping.long()
    local = s["ctx"].block_tables is None
    planes = []
    for i, x in enumerate((k, v)):
        plane = s["cache"][i, 0].view(-1, hkv, HEAD_DIM)
        sc = None if s["scales"] is None else s["scales"][i, 0].view(-1, hkv, 1)
        if kv in CODE:
            codes, scale = _quantise(x, kv)
            plane.view(torch.uint8)[slots] = codes.view(torch.uint8)
            sc[slots] = scale
        else:
            plane[slots] = x
        planes.append((plane, sc))
    out = torch.empty_like(q)
    at = 0
    for seq in s["seqs"]:
        n, p = seq.num_new_tokens, seq.num_cached_tokens
        pos = torch.arange(n + p, device="cuda")
        rows = torch.tensor(seq.block_table, device="cuda")[pos // bs] * bs + pos % bs
        both = []
        for (plane, sc), x in zip(planes, (k, v)):
            if local:  # nothing cached: the call attends over the step's own k and v
                both.append(x[at:at + n].double())
            elif sc is None:
                both.append(plane[rows].double())
            else:
                codes = plane.view(torch.uint8)[rows].view(plane.dtype)
                both.append(codes.double() * sc[rows].double())
        hidden = torch.arange(n + p, device="cuda")[None, :] > torch.arange(p, p + n, device="cuda")[:, None]
        for h in range(hkv):
            kh, vh = (x[:, h].contiguous() for x in both)
            for j in range(h * g, (h + 1) * g):
                a = (q[at:at + n, j] @ kh.t().contiguous()) * HEAD_DIM ** -0.5
                a = torch.softmax(a.masked_fill_(hidden, -math.inf), dim=-1)
                out[at:at + n, j] = a @ vh
        at += n
    return [out, None, None]
