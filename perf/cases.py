"""Performance cases of the attention library, one pass of each through a public entry point.

Two surfaces are used, as programs use them: the launcher level (``sca_amd.hip``: an engine that
owns its output and scratch buffers and passes plain pointers) for the headline and the smallest
calls, and the host API (``sca_amd.host``: the sca:: calls that pick a backend and return a new
output) for everything else. Sizes are those of the repository's benchmark, tests and design
notes, or generic.

Kinds of case:
  prefill   one attention over [B, H, S, D] tensors (S_q <= S_kv when causal); ``api`` "launcher"
            or "host", ``layout`` "bhsd" or "bshd", ``lse`` asks for the log-sum-exp too
  varlen    packed sequences of mixed lengths in one call
  decode    one query token per sequence over contiguous K/V
  paged     one layer of a serving step: write this step's K/V rows into the paged cache and
            attend over it
"""

import math
import os
import random
import sys

import torch

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
_PY = os.path.join(_ROOT, "scicompute-attention_amd", "python")
if _PY not in sys.path:
    sys.path.insert(0, _PY)

from sca_amd import hip, host  # noqa: E402

_TORCH = {"f16": torch.float16, "bf16": torch.bfloat16, "f32": torch.float32}
_BYTES = {"f16": 2, "bf16": 2, "f32": 4}
_HIP_DTYPE = {"f16": hip.DTYPE_F16, "bf16": hip.DTYPE_BF16, "f32": hip.DTYPE_F32}


# ---- the cases ------------------------------------------------------------------------------------

def _prefill(name, dtype, batch, heads, kv_heads, seq_q, seq_kv, head_dim, causal, api="host",
             layout="bhsd", lse=False, std=1.0):
    c = {"kind": "prefill", "dtype": dtype, "batch": batch, "heads": heads, "kv_heads": kv_heads,
         "seq_q": seq_q, "seq_kv": seq_kv, "head_dim": head_dim, "causal": causal, "api": api,
         "layout": layout, "lse": lse, "std": std}
    return {"name": name, **c} if name else c


def _decode(name, dtype, batch, heads, kv_heads, seq_kv, head_dim, api="host"):
    c = {"kind": "decode", "dtype": dtype, "batch": batch, "heads": heads, "kv_heads": kv_heads,
         "seq_kv": seq_kv, "head_dim": head_dim, "api": api}
    return {"name": name, **c} if name else c


def _varlen(name, dtype, seqs, low, high, mix, heads, kv_heads, head_dim, causal):
    c = {"kind": "varlen", "dtype": dtype, "seqs": seqs, "low": low, "high": high, "mix": mix,
         "heads": heads, "kv_heads": kv_heads, "head_dim": head_dim, "causal": causal}
    return {"name": name, **c} if name else c


def _paged(name, dtype, seqs, low, high, mix, block, heads, kv_heads, head_dim):
    c = {"kind": "paged", "dtype": dtype, "seqs": seqs, "low": low, "high": high, "mix": mix,
         "block": block, "heads": heads, "kv_heads": kv_heads, "head_dim": head_dim}
    return {"name": name, **c} if name else c


def listed():
    return [
        # The headline: one long causal prompt of an 8-head shard, fp16, on an engine's own buffers.
        _prefill("prompt_4k", "f16", 1, 8, 8, 4096, 4096, 128, True, api="launcher"),
        # A batch of long prompts with grouped KV heads: the largest prefill of the benchmark.
        _prefill("prompt_batch_8k", "bf16", 4, 32, 8, 8192, 8192, 128, True, std=0.5),
        # A short ragged prompt (the benchmark's 1000-token tail): one small launch.
        _prefill("prompt_1000", "bf16", 1, 32, 8, 1000, 1000, 128, True, api="launcher", std=0.5),
        # An encoder layer: a batch of odd-length bidirectional sequences, token-major, head_dim 64.
        _prefill("encoder_197", "f16", 16, 16, 16, 197, 197, 64, False, api="launcher",
                 layout="bshd"),
        # Chunked prefill: the last 512 tokens of a long context, the diagonal far to the right.
        _prefill("chunk_512", "bf16", 1, 32, 8, 512, 12801, 128, True),
        # A few new tokens per conversation over its context (a short turn, or drafted tokens to
        # be checked).
        _prefill("few_tokens", "bf16", 8, 32, 8, 6, 4102, 128, True),
        # The widest supported head, grouped, with the log-sum-exp a later merge needs.
        _prefill("prompt_d256_lse", "bf16", 1, 16, 8, 4096, 4096, 256, True, lse=True),
        # Mixed prompts packed into one call.
        _varlen("packed_prompts", "bf16", 16, 256, 4096, 5, 32, 8, 128, True),
        # Split-K decode of the benchmark: 16 sequences of 4096 keys.
        _decode("decode_16x4096", "f16", 16, 32, 8, 4096, 128),
        # The smallest decode: one sequence, latency and launches.
        _decode("decode_1x1500", "f16", 1, 32, 8, 1500, 128, api="launcher"),
        # Decode at a head_dim between the powers of two.
        _decode("decode_d96", "bf16", 16, 32, 8, 4096, 96),
        # One layer of the benchmark's paged serving step: 64 ragged sequences, 16-token pages.
        _paged("paged_64_ragged", "bf16", 64, 512, 16384, 1, 16, 32, 8, 128),
    ]


def _log_int(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def _odd_mostly(rng, n):
    """Lengths in use are rarely round; every third one is rounded to a multiple of 64."""
    return max(64, (n + 32) // 64 * 64) if rng.random() < 1 / 3 else n


_HEADS = [(8, 8), (16, 16), (32, 32), (16, 8), (32, 8), (24, 8), (64, 8), (28, 4), (16, 2)]
_MOST_FLOPS = 1.0e12
_MOST_BYTES = 2.0e9


def _fits(c):
    w = work(c)
    return w["flops"] <= _MOST_FLOPS and w["bytes"] <= _MOST_BYTES


def draw(rng):
    while True:
        heads, kv_heads = rng.choice(_HEADS)
        dtype = rng.choice(["bf16", "f16"])
        # 128 and 64 are the common head dims; the others are supported and in use too.
        head_dim = rng.choice([128, 128, 128, 64, 64, 32, 96, 160, 192, 256])
        kind = rng.choice(["prompt", "prompt", "encoder", "chunk", "few", "varlen", "decode",
                           "decode", "paged"])
        if kind == "prompt":
            s = _odd_mostly(rng, _log_int(rng, 30, 12000))
            c = _prefill("", dtype, _log_int(rng, 1, 16), heads, kv_heads, s, s, head_dim, True,
                         layout=rng.choice(["bhsd", "bshd"]), lse=rng.random() < 0.25,
                         api=rng.choice(["host", "launcher"]))
        elif kind == "encoder":
            s = _odd_mostly(rng, _log_int(rng, 30, 6000))
            cross = _odd_mostly(rng, _log_int(rng, 30, 6000)) if rng.random() < 0.3 else s
            c = _prefill("", dtype, _log_int(rng, 1, 32), heads, heads, s, cross, head_dim, False,
                         layout=rng.choice(["bhsd", "bshd"]), api="launcher")
        elif kind == "chunk":
            s = rng.choice([128, 256, 512, 1024, 2048])
            c = _prefill("", dtype, _log_int(rng, 1, 4), heads, kv_heads, s,
                         s + _log_int(rng, 500, 30000), head_dim, True)
        elif kind == "few":
            s = rng.randint(2, 40)
            c = _prefill("", dtype, _log_int(rng, 1, 32), heads, kv_heads, s,
                         s + _log_int(rng, 250, 20000), head_dim, True)
        elif kind == "varlen":
            low = _log_int(rng, 16, 500)
            c = _varlen("", dtype, _log_int(rng, 2, 48), low, low * rng.randint(2, 12),
                        rng.randrange(1 << 20), heads, kv_heads, head_dim, rng.random() < 0.75)
        elif kind == "decode":
            # fp32 caches are served by decode only.
            c = _decode("", rng.choice([dtype, dtype, dtype, "f32"]), _log_int(rng, 1, 128), heads,
                        kv_heads, _odd_mostly(rng, _log_int(rng, 260, 40000)), head_dim,
                        api=rng.choice(["host", "host", "launcher"]))
        else:
            low = _log_int(rng, 64, 4000)
            c = _paged("", dtype, _log_int(rng, 1, 160), low, low * rng.randint(1, 16),
                       rng.randrange(1 << 20), rng.choice([16, 16, 32, 64]), heads, kv_heads,
                       head_dim)
        if _fits(c):
            return c


# ---- shapes -----------------------------------------------------------------------------------------

def _lengths(c):
    rng = random.Random(1000003 * c["mix"] + c["seqs"])
    return [rng.randint(c["low"], c["high"]) for _ in range(c["seqs"])]


def _pairs(seq_q, seq_kv, causal):
    """Visible (query, key) pairs; causal is aligned at the bottom right."""
    if not causal:
        return seq_q * seq_kv
    return seq_q * (seq_kv - seq_q) + seq_q * (seq_q + 1) // 2


def work(case):
    c = case
    d, hq, hkv, eb = c["head_dim"], c["heads"], c["kv_heads"], _BYTES[c["dtype"]]
    if c["kind"] == "prefill":
        b, sq, skv = c["batch"], c["seq_q"], c["seq_kv"]
        bytes_ = 2 * b * hq * sq * d * eb + 2 * b * hkv * skv * d * eb
        if c["lse"]:
            bytes_ += b * hq * sq * 4
        return {"bytes": bytes_, "flops": 4 * b * hq * d * _pairs(sq, skv, c["causal"])}
    if c["kind"] == "varlen":
        lens = _lengths(c)
        pairs = sum(_pairs(n, n, c["causal"]) for n in lens)
        return {"bytes": sum(lens) * 2 * (hq + hkv) * d * eb, "flops": 4 * hq * d * pairs}
    if c["kind"] == "decode":
        b, skv = c["batch"], c["seq_kv"]
        return {"bytes": 2 * b * d * eb * (hkv * skv + hq), "flops": 4 * b * hq * skv * d}
    lens = [n + 1 for n in _lengths(c)]
    pages = sum(-(-n // c["block"]) for n in lens)
    row = hkv * d * eb
    # K and V of every key, the page table, q and out, and the step's new rows in and out.
    return {"bytes": 2 * sum(lens) * row + 4 * pages + 2 * len(lens) * hq * d * eb
            + 4 * len(lens) * row, "flops": 4 * hq * d * sum(lens)}


# Measured on MI355X against the 64-bit result (2-norm; the weights and the output are rounded to
# the type): bf16 1.7e-3 .. 2.3e-3 off, fp16 2.0e-4 .. 3.0e-4, fp32 2e-7 .. 3e-7, single values up to
# 2.5e-2, 3e-3 and 2e-6. Two correct implementations round differently, so they are up to about
# 1.5 times that apart; the limits are about four times what is seen (fp32: 32-bit sums over tens of
# thousands of keys in another order).
def tolerance(case):
    return {"bf16": {"rel": 9e-3, "max": 0.1}, "f16": {"rel": 1.2e-3, "max": 0.015},
            "f32": {"rel": 5e-6, "max": 5e-5}}[case["dtype"]]


# ---- inputs -----------------------------------------------------------------------------------------

def _normal(gen, shape, dtype, std=1.0):
    return (torch.randn(shape, generator=gen, device="cuda") * std).to(_TORCH[dtype])


def _generator(seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    return gen


def _prefill_inputs(c, seed):
    gen = _generator(seed)

    def make(heads, seq):
        dims = (c["batch"], heads, seq) if c["layout"] == "bhsd" else (c["batch"], seq, heads)
        return _normal(gen, (*dims, c["head_dim"]), c["dtype"], c["std"])

    return (make(c["heads"], c["seq_q"]), make(c["kv_heads"], c["seq_kv"]),
            make(c["kv_heads"], c["seq_kv"]))


def _varlen_inputs(c, seed):
    gen = _generator(seed)
    total = sum(_lengths(c))
    return tuple(_normal(gen, (total, h, c["head_dim"]), c["dtype"])
                 for h in (c["heads"], c["kv_heads"], c["kv_heads"]))


def _decode_inputs(c, seed):
    gen = _generator(seed)
    kv = (c["batch"], c["kv_heads"], c["seq_kv"], c["head_dim"])
    return (_normal(gen, (c["batch"], c["heads"], 1, c["head_dim"]), c["dtype"]),
            _normal(gen, kv, c["dtype"]), _normal(gen, kv, c["dtype"]))


def _paged_inputs(c, seed):
    """Queries, the context's K and V rows of all sequences one after the other, and the step's."""
    gen = _generator(seed)
    n, row = c["seqs"], (c["kv_heads"], c["head_dim"])
    total = sum(_lengths(c))
    return (_normal(gen, (n, c["heads"], 1, c["head_dim"]), c["dtype"]),
            _normal(gen, (total, *row), c["dtype"]), _normal(gen, (total, *row), c["dtype"]),
            _normal(gen, (n, *row), c["dtype"]), _normal(gen, (n, *row), c["dtype"]))


def _wrap(t, dtype):
    """A borrowed sci::Tensor handle over a torch tensor."""
    dims = (host.c_i64 * t.dim())(*t.shape)
    return host.Tensor(host.host_lib().sca_tensor_wrap(t.data_ptr(), dims, t.dim(),
                                                       host.DTYPES[dtype], host.GPU), dtype)


class _Memory:
    """Device memory as torch sees it; `owner` keeps it alive."""

    def __init__(self, ptr, shape, dtype, owner):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": tuple(shape), "data": (ptr, False), "version": 3,
                                         "typestr": "<f4" if dtype == "f32" else "<i2"}


def _as_torch(ptr, shape, dtype, owner):
    t = torch.as_tensor(_Memory(ptr, shape, dtype, owner), device="cuda")
    return t if dtype == "f32" else t.view(_TORCH[dtype])


def _result(t):
    """A tensor that the host API returned."""
    return _as_torch(t.data_ptr, t.shape, t.dtype, t)


def _scale(c):
    return 1.0 / math.sqrt(c["head_dim"])


def _strides(layout, seq, heads, d):
    return (heads * seq * d, seq * d, d) if layout == "bhsd" else (seq * heads * d, d, heads * d)


def _prepare_prefill(c, seed):
    q, k, v = _prefill_inputs(c, seed)
    if c["api"] == "host":
        cfg = host.AttentionConfig(causal=c["causal"], layout=c["layout"], return_lse=c["lse"])
        return {"case": c, "keep": (q, k, v), "cfg": cfg,
                "qkv": tuple(_wrap(t, c["dtype"]) for t in (q, k, v))}
    b, hq, hkv, sq, skv, d = (c[n] for n in ("batch", "heads", "kv_heads", "seq_q", "seq_kv",
                                             "head_dim"))
    out = torch.empty((b, hq, sq, d), dtype=_TORCH[c["dtype"]], device="cuda")
    lse = torch.empty((b, hq, sq), dtype=torch.float32, device="cuda") if c["lse"] else None
    p = hip.FlashParams()
    p.q, p.k, p.v, p.out = (t.data_ptr() for t in (q, k, v, out))
    p.lse = lse.data_ptr() if c["lse"] else None
    p.batch, p.num_heads, p.num_kv_heads, p.seq_q, p.seq_kv, p.head_dim = b, hq, hkv, sq, skv, d
    p.q_sb, p.q_sh, p.q_ss = _strides(c["layout"], sq, hq, d)
    p.k_sb, p.k_sh, p.k_ss = _strides(c["layout"], skv, hkv, d)
    p.v_sb, p.v_sh, p.v_ss = _strides(c["layout"], skv, hkv, d)
    p.o_sb, p.o_sh, p.o_ss = _strides("bhsd", sq, hq, d)
    p.scale, p.causal, p.dtype = _scale(c), int(c["causal"]), _HIP_DTYPE[c["dtype"]]
    p.diagonal = skv - sq if c["causal"] else 0
    return {"case": c, "keep": (q, k, v), "params": p, "out": out, "lse": lse}


def _prepare_varlen(c, seed):
    q, k, v = _varlen_inputs(c, seed)
    lens = _lengths(c)
    cu = [0]
    for n in lens:
        cu.append(cu[-1] + n)
    return {"case": c, "keep": (q, k, v), "qkv": tuple(_wrap(t, c["dtype"]) for t in (q, k, v)),
            "cu": cu, "longest": max(lens), "cfg": host.AttentionConfig(causal=c["causal"])}


def _prepare_decode(c, seed):
    q, k, v = _decode_inputs(c, seed)
    if c["api"] == "host":
        return {"case": c, "keep": (q, k, v), "cfg": host.AttentionConfig(),
                "qkv": tuple(_wrap(t, c["dtype"]) for t in (q, k, v))}
    b, hq, hkv, skv, d = (c[n] for n in ("batch", "heads", "kv_heads", "seq_kv", "head_dim"))
    cus = host.host_lib().sca_device_cu_count()
    splits = host.decode_splits(host.AttentionShape(b, 1, skv, hq, hkv, d), cus)
    out = torch.empty_like(q)
    parts = torch.empty(hip.hip_lib().sca_hip_decode_partial_elements(b, hq, splits, d),
                        dtype=torch.float32, device="cuda")
    p = hip.DecodeParams()
    p.q, p.k, p.v, p.out = (t.data_ptr() for t in (q, k, v, out))
    rows = b * hq * splits
    p.partial_m = parts.data_ptr()
    p.partial_l = p.partial_m + 4 * rows
    p.partial_o = p.partial_l + 4 * rows
    p.batch, p.num_heads, p.num_kv_heads, p.seq_kv, p.head_dim = b, hq, hkv, skv, d
    p.num_splits = splits
    p.q_sb, p.q_sh = hq * d, d
    p.k_sb, p.k_sh, p.k_ss = hkv * skv * d, skv * d, d
    p.v_sb, p.v_sh, p.v_ss = p.k_sb, p.k_sh, p.k_ss
    p.o_sb, p.o_sh = hq * d, d
    p.scale, p.dtype = _scale(c), _HIP_DTYPE[c["dtype"]]
    return {"case": c, "keep": (q, k, v, parts), "params": p, "out": out}


_PIECE = 1024  # tokens a sequence's context grows by at a time while the others grow too


def _prepare_paged(c, seed):
    q, k, v, k_new, v_new = _paged_inputs(c, seed)
    lens = _lengths(c)
    n, bs = c["seqs"], c["block"]
    cache = host.PagedKVCache(host.KVCacheConfig(
        num_layers=1, num_kv_heads=c["kv_heads"], head_dim=c["head_dim"], block_size=bs,
        num_blocks=sum(-(-(m + 1) // bs) for m in lens), max_num_seqs=n, dtype=c["dtype"]))
    # The contexts grow side by side in a shuffled order, so a sequence's pages are scattered
    # over the pool.
    start, at = [0] * n, 0
    for s, m in enumerate(lens):
        start[s], at = at, at + m
    pieces = [(s, a) for s, m in enumerate(lens) for a in range(0, m, _PIECE)]
    random.Random(c["mix"]).shuffle(pieces)
    done = [0] * n
    for s, _ in pieces:
        m = min(_PIECE, lens[s] - done[s])
        lo = start[s] + done[s]
        cache.reserve(s, m)
        cache.write_layer(0, _wrap(k[lo:lo + m], c["dtype"]), _wrap(v[lo:lo + m], c["dtype"]))
        done[s] += m
    # This step's token of every sequence: reserved once, for all layers.
    cache.reserve_batch(range(n))
    cache.sync_page_table()
    seq_lens = torch.tensor([m + 1 for m in lens], dtype=torch.int32, device="cuda")
    pool_shape = (cache.cfg.num_blocks, bs, c["kv_heads"], c["head_dim"])
    pool = tuple(_as_torch(p, pool_shape, c["dtype"], cache) for p in cache.layer_ptrs(0))
    torch.cuda.synchronize()
    return {"case": c, "keep": (q, k_new, v_new, seq_lens), "cache": cache, "pool": pool,
            "q": _wrap(q, c["dtype"]), "k_new": _wrap(k_new, c["dtype"]),
            "v_new": _wrap(v_new, c["dtype"]), "cfg": host.AttentionConfig(),
            "params": {"seq_lens": seq_lens.data_ptr(), "num_seqs": n, "block_size": bs}}


_PREPARE = {"prefill": _prepare_prefill, "varlen": _prepare_varlen, "decode": _prepare_decode,
            "paged": _prepare_paged}


def prepare(case, seed):
    return _PREPARE[case["kind"]](dict(case), seed)


# ---- one pass ---------------------------------------------------------------------------------------

def run(state):
    c = state["case"]
    if c["kind"] == "prefill":
        if c["api"] == "launcher":
            hip.flash_fwd(state["params"])
            return {"out": state["out"], "lse": state["lse"]}
        r = host.attention(*state["qkv"], state["cfg"])
        return {"out": _result(r.out), "lse": _result(r.lse) if r.lse is not None else None}
    if c["kind"] == "varlen":
        r = host.flash_attention_varlen(*state["qkv"], c["seqs"], state["cu"], state["cu"],
                                        state["longest"], state["longest"], state["cfg"])
        return {"out": _result(r.out)}
    if c["kind"] == "decode":
        if c["api"] == "launcher":
            hip.decode_splitk(state["params"])
            return {"out": state["out"]}
        return {"out": _result(host.decode_attention(*state["qkv"], state["cfg"]).out)}
    cache = state["cache"]
    cache.write_layer(0, state["k_new"], state["v_new"])
    r = host.paged_attention(state["q"], cache, state["params"], state["cfg"])
    return {"out": _result(r.out), "k_pool": state["pool"][0], "v_pool": state["pool"][1]}


# ---- the same in 64 bits ----------------------------------------------------------------------------

def _attend64(q, k, v, causal, scale):
    """(out, lse) of q [H_q, S_q, D] over k, v [H_kv, S_kv, D], in blocks of rows."""
    hq, sq, d = q.shape
    hkv, skv, _ = k.shape
    group = hq // hkv
    out = torch.empty((hq, sq, d), dtype=torch.float64, device=q.device)
    lse = torch.empty((hq, sq), dtype=torch.float64, device=q.device)
    rows = max(1, min(sq, (1 << 27) // (group * skv)))
    keys = torch.arange(skv, device=q.device)
    for h in range(hkv):
        kt, vh = k[h].double().t().contiguous(), v[h].double()
        qh = q[h * group:(h + 1) * group].double()
        for a in range(0, sq, rows):
            e = min(sq, a + rows)
            s = torch.matmul(qh[:, a:e].reshape(-1, d), kt).mul_(scale).view(group, e - a, skv)
            if causal:
                last = torch.arange(a, e, device=q.device) + (skv - sq)
                s.masked_fill_(keys[None, :] > last[:, None], float("-inf"))
            m = s.amax(-1, keepdim=True)
            s.sub_(m).exp_()
            l = s.sum(-1, keepdim=True)
            o = torch.matmul(s.view(-1, skv), vh).view(group, e - a, d) / l
            out[h * group:(h + 1) * group, a:e] = o
            lse[h * group:(h + 1) * group, a:e] = (m + l.log()).squeeze(-1)
    return out, lse


def exact(case, seed):
    c, scale = case, _scale(case)
    if c["kind"] == "prefill":
        q, k, v = _prefill_inputs(c, seed)
        if c["layout"] == "bshd":
            q, k, v = (t.transpose(1, 2) for t in (q, k, v))
        both = [_attend64(q[b], k[b], v[b], c["causal"], scale) for b in range(c["batch"])]
        return {"out": torch.stack([o for o, _ in both]),
                "lse": torch.stack([l for _, l in both]) if c["lse"] else None}
    if c["kind"] == "varlen":
        q, k, v = _varlen_inputs(c, seed)
        outs, at = [], 0
        for n in _lengths(c):
            part = [t[at:at + n].transpose(0, 1) for t in (q, k, v)]
            outs.append(_attend64(*part, c["causal"], scale)[0].transpose(0, 1))
            at += n
        return {"out": torch.cat(outs)}
    if c["kind"] == "decode":
        q, k, v = _decode_inputs(c, seed)
        return {"out": torch.stack([_attend64(q[b], k[b], v[b], False, scale)[0]
                                    for b in range(c["batch"])])}
    q, k, v, k_new, v_new = _paged_inputs(c, seed)
    outs, at = [], 0
    for s, n in enumerate(_lengths(c)):
        ks = torch.cat([k[at:at + n], k_new[s:s + 1]]).transpose(0, 1)
        vs = torch.cat([v[at:at + n], v_new[s:s + 1]]).transpose(0, 1)
        outs.append(_attend64(q[s], ks, vs, False, scale)[0])
        at += n
    return {"out": torch.stack(outs), "k_pool": None, "v_pool": None}
