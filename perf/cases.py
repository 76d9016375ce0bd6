"""Performance cases of the paged-attention path and the layer ops beside it.

Each case is one call (or one layer's short run of calls) that a serving
program makes through the public entry points: the vLLM attention backend
(HipAttentionImpl.forward), the functional wrappers (kernels.*) and the engine
ops (EngineMLP, EngineRMSNorm).  listed() names the fixed ones, draw() gives
more of the same ranges.  All inputs come from the seed.

Kinds of case
  decode   one decode step of a batch: the new tokens' K/V go to the paged cache
           and every sequence attends over its context.  entry "forward": the
           backend on vLLM's cache layout; "fused": kernels.paged_decode with
           the write in the same launch, on the engine's cache layout.
  prefill  chunked prefill through the backend: `prefix` cached tokens and a
           chunk of lo..hi new ones per sequence.
  mixed    a step of decodes and prefill chunks together, through the backend.
  encoder  bidirectional attention inside each sequence, no cache (backend).
  mlp      the gated SiLU MLP of a layer (EngineMLP).
  layer    a layer's bandwidth-bound ops: residual add + RMSNorm, then bias,
           rotary embedding and KV write of the QKV projection's output.
  topk     the k largest logits of each row.
"""
import math
import sys
from pathlib import Path
from types import SimpleNamespace

import torch

_PKG = str(Path.cwd() / "vllm-apple_amd")
if _PKG not in sys.path:
    sys.path.insert(1, _PKG)

from vllm_apple_amd import kernels  # noqa: E402
from vllm_apple_amd.backend import (AttentionType, HipAttentionImpl,  # noqa: E402
                                    HipAttentionMetadataBuilder)
from vllm_apple_amd.engine.mlp import EngineMLP  # noqa: E402
from vllm_apple_amd.engine.rmsnorm import EngineRMSNorm  # noqa: E402

DEV = "cuda"
BS = 16  # cache block size, the reference's default
EPS = 1e-5
MAX_POS = 32768
ROPE_BASE = 1e6


def listed():
    """The fixed cases, smallest first inside a kind."""
    return [
        # The smallest call: a small model answering four short conversations.
        # Latency and launches count.
        dict(name="decode-tiny", kind="decode", entry="forward", seqs=4, lo=16, hi=512, heads=14,
             kv=2, dim=64, dtype="fp16"),
        # An ordinary batch: ragged conversations on a bf16 model.
        dict(name="decode-ragged", kind="decode", entry="forward", seqs=27, lo=100, hi=6000,
             heads=32, kv=8, dim=128, dtype="bf16"),
        # The benchmark's headline: 32 contexts of 8192 tokens, write and
        # attention in one launch.
        dict(name="decode-32x8k", kind="decode", entry="fused", seqs=32, lo=8192, hi=8192,
             heads=32, kv=8, dim=128, dtype="fp16"),
        # New prompts of odd lengths with nothing cached, bf16.
        dict(name="prefill-prompts", kind="prefill", seqs=7, prefix=0, lo=20, hi=1500, heads=32,
             kv=8, dim=128, dtype="bf16"),
        # The benchmark's chunked prefill: four chunks of 512 over 2048 cached.
        dict(name="prefill-chunks", kind="prefill", seqs=4, prefix=2048, lo=512, hi=512, heads=32,
             kv=8, dim=128, dtype="fp16"),
        # The benchmark's mixed step: 56 decodes beside 8 chunks of 256.
        dict(name="mixed-step", kind="mixed", seqs=56, chunks=8, chunk=256, lo=256, hi=16384,
             heads=32, kv=8, dim=128, dtype="fp16"),
        # An embedding model's batch: bidirectional, multi-head, ragged.
        dict(name="encoder", kind="encoder", seqs=25, lo=12, hi=512, heads=12, kv=12, dim=64,
             dtype="fp16"),
        # A layer's MLP: a decode batch, a small prompt, a mixed step's tokens.
        dict(name="mlp-24", kind="mlp", tokens=24, hidden=5120, inter=32768, dtype="fp16"),
        dict(name="mlp-300", kind="mlp", tokens=300, hidden=4096, inter=14336, dtype="bf16"),
        dict(name="mlp-2104", kind="mlp", tokens=2104, hidden=5120, inter=32768, dtype="fp16"),
        # The mixed step's tokens through a layer's norm and QKV epilogue.
        dict(name="layer-2104", kind="layer", tokens=2104, hidden=5120, heads=32, kv=8, dim=128,
             dtype="fp16"),
        # Sampling's selection for a batch of 32.
        dict(name="topk-32", kind="topk", tokens=32, vocab=128256, k=50, dtype="fp16"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


# (heads, kv heads, head size) of the repository's configurations and tests.
_HEADS = [(14, 2, 64), (32, 8, 128), (32, 8, 128), (32, 32, 128), (28, 4, 128), (16, 2, 96)]


def draw(rng):
    """One more case of the listed ones' ranges."""
    kind = rng.choice(["decode", "decode", "prefill", "mixed", "encoder", "mlp", "mlp", "layer",
                       "topk"])
    dtype = rng.choice(["fp16", "bf16"])
    heads, kv, dim = rng.choice(_HEADS)
    if kind == "decode":
        seqs = _log_int(rng, 1, 128)
        # At most about 200k cached tokens of 8 kv heads at dim 128.
        cap = max(64, min(MAX_POS, int(200_000 * 1024 / (kv * dim) / seqs)))
        hi = _log_int(rng, 64, cap)
        lo = rng.choice([hi, max(1, hi // 2), max(1, hi // 16)])
        return dict(kind=kind, entry=rng.choice(["forward", "fused"]), seqs=seqs, lo=lo, hi=hi,
                    heads=heads, kv=kv, dim=dim, dtype=dtype)
    if kind == "prefill":
        seqs = _log_int(rng, 1, 8)
        hi = _log_int(rng, 32, max(64, 4096 // seqs))
        return dict(kind=kind, seqs=seqs, prefix=rng.choice([0, 0, _log_int(rng, 16, 4096)]),
                    lo=rng.choice([hi, max(2, hi // 8)]), hi=hi, heads=heads, kv=kv, dim=dim,
                    dtype=dtype)
    if kind == "mixed":
        return dict(kind=kind, seqs=rng.randint(2, 56), chunks=rng.randint(1, 8),
                    chunk=_log_int(rng, 32, 256), lo=256, hi=_log_int(rng, 512, 16384), heads=32,
                    kv=8, dim=128, dtype=dtype)
    if kind == "encoder":
        h, d = rng.choice([(12, 64), (16, 64), (12, 32), (8, 96)])
        return dict(kind=kind, seqs=_log_int(rng, 1, 64), lo=4, hi=_log_int(rng, 16, 512),
                    heads=h, kv=h, dim=d, dtype=dtype)
    if kind == "mlp":
        hidden, inter = rng.choice([(896, 4864), (4096, 14336), (4096, 14336), (5120, 32768),
                                    (2048, 8192)])
        return dict(kind=kind, tokens=_log_int(rng, 1, 2104), hidden=hidden, inter=inter,
                    dtype=dtype)
    if kind == "layer":
        return dict(kind=kind, tokens=_log_int(rng, 1, 4096), hidden=rng.choice([896, 4096, 5120]),
                    heads=heads, kv=kv, dim=dim, dtype=dtype)
    return dict(kind=kind, tokens=_log_int(rng, 1, 320),
                vocab=rng.choice([32000, 32768, 128256, 151936]), k=rng.choice([1, 8, 20, 50, 50, 64]),
                dtype=dtype)


# ------------------------------------------------------------------ inputs


def _dt(case):
    return {"fp16": torch.float16, "bf16": torch.bfloat16}[case["dtype"]]


def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    return g


def _randn(shape, g, dtype, std=1.0):
    t = torch.randn(shape, generator=g, device=DEV, dtype=torch.float32)
    return (t * std if std != 1.0 else t).to(dtype)


def _lengths(case, n):
    """n lengths, log-uniform over [lo, hi], the same for every seed so that
    one case is one amount of work."""
    lo, hi = case["lo"], case["hi"]
    if lo >= hi:
        return [hi] * n
    r = torch.Generator()
    r.manual_seed(1000 * lo + 10 * hi + n)
    u = torch.rand(n, generator=r, dtype=torch.float64)
    return [int(round(math.exp(math.log(lo) + float(x) * (math.log(hi) - math.log(lo)))))
            for x in u]


def _batch(case):
    """(total lengths, new tokens) per sequence, decodes first."""
    kind = case["kind"]
    if kind == "decode":
        lens = _lengths(case, case["seqs"])
        return lens, [1] * len(lens)
    if kind == "prefill":
        new = _lengths(case, case["seqs"])
        return [case["prefix"] + n for n in new], new
    if kind == "mixed":
        lens = _lengths(case, case["seqs"] + case["chunks"])
        new = [1] * case["seqs"] + [case["chunk"]] * case["chunks"]
        return [max(l, n) for l, n in zip(lens, new)], new
    new = _lengths(case, case["seqs"])  # encoder
    return new, new


def _attention(case, seed):
    g, dt = _gen(seed), _dt(case)
    H, KV, D = case["heads"], case["kv"], case["dim"]
    lens, new = _batch(case)
    S, T = len(lens), sum(new)
    s = SimpleNamespace(case=case, lens=lens, new=new)
    s.q, s.k, s.v = (_randn((T, h, D), g, dt) for h in (H, KV, KV))
    s.out = torch.zeros(T, H, D, dtype=dt, device=DEV)
    s.scale = 1.0 / math.sqrt(D)
    qsl = [0]
    for n in new:
        qsl.append(qsl[-1] + n)
    s.qsl = qsl
    s.cache = None
    if case["kind"] != "encoder":
        # A pool of randomly placed blocks, a little larger than the batch.
        nblk = [-(-L // BS) for L in lens]
        pool = sum(nblk) + 8
        perm = torch.randperm(pool, generator=g, device=DEV).to(torch.int32)
        bt = torch.full((S, max(nblk)), -1, dtype=torch.int32, device=DEV)
        off = 0
        for i, n in enumerate(nblk):
            bt[i, :n] = perm[off:off + n]
            off += n
        shape = (pool, KV, BS, D) if case.get("entry") == "fused" else (pool, BS, KV, D)
        s.cache = _randn((2,) + shape, g, dt)
        s.bt = bt
    else:
        s.bt = torch.zeros(S, 1, dtype=torch.int32, device=DEV)
    s.seq_lens = torch.tensor(lens, dtype=torch.int32, device=DEV)
    if case.get("entry") == "fused":
        return s
    qsl_t = torch.tensor(qsl, dtype=torch.int32)
    qsl_d = qsl_t.to(DEV)
    slots = torch.zeros(T, dtype=torch.int64, device=DEV)
    if s.cache is not None:
        tok = torch.repeat_interleave(torch.arange(S), torch.tensor(new)).to(DEV)
        pos = torch.tensor([p for L, n in zip(lens, new) for p in range(L - n, L)], device=DEV)
        slots = s.bt[tok, pos // BS].long() * BS + pos % BS
    causal = case["kind"] != "encoder"
    cm = SimpleNamespace(num_actual_tokens=T, max_query_len=max(new), query_start_loc=qsl_d,
                         query_start_loc_cpu=qsl_t, max_seq_len=max(lens), seq_lens=s.seq_lens,
                         seq_lens_cpu=torch.tensor(lens, dtype=torch.int32),
                         block_table_tensor=s.bt, slot_mapping=slots, causal=causal)
    s.meta = HipAttentionMetadataBuilder(SimpleNamespace(block_size=BS)).build(0, cm)
    s.impl = HipAttentionImpl(H, D, s.scale, KV, None, None, "auto",
                              attn_type=AttentionType.DECODER if causal
                              else AttentionType.ENCODER_ONLY)
    return s


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("decode", "prefill", "mixed", "encoder"):
        return _attention(case, seed)
    g, dt = _gen(seed), _dt(case)
    s = SimpleNamespace(case=case)
    if kind == "mlp":
        T, H, I = case["tokens"], case["hidden"], case["inter"]
        s.x = _randn((T, H), g, dt)
        s.w1 = _randn((2 * I, H), g, dt, std=1.0 / math.sqrt(H))
        s.w2 = _randn((H, I), g, dt, std=1.0 / math.sqrt(I))
        s.out = torch.empty(T, H, dtype=dt, device=DEV)
        s.mlp = EngineMLP(None, H, I)
        s.mlp.set_weights(gate_up_proj=s.w1, down_proj=s.w2)
    elif kind == "layer":
        T, hid, H, KV, D = (case[n] for n in ("tokens", "hidden", "heads", "kv", "dim"))
        # A layer's output is small beside the residual stream that it is
        # added to, and so are the projection's biases.
        s.x = _randn((T, hid), g, dt, std=0.02)
        s.res = _randn((T, hid), g, dt)
        s.w = (1.0 + 0.1 * torch.randn(hid, generator=g, device=DEV)).to(dt)
        s.normed = torch.empty(T, hid, dtype=dt, device=DEV)
        s.norm = EngineRMSNorm(None, hid, eps=EPS)
        s.norm.set_weights(s.w)
        s.qkv = _randn((T, (H + 2 * KV) * D), g, dt)
        s.q, s.k, s.v = (t.view(T, -1, D) for t in s.qkv.split([H * D, KV * D, KV * D], dim=1))
        s.bias = _randn(((H + 2 * KV) * D,), g, dt, std=0.02)
        s.pos = torch.randint(0, MAX_POS, (T,), generator=g, device=DEV).to(torch.int32)
        s.cos, s.sin = kernels.rope_cos_sin_cache(D, MAX_POS, ROPE_BASE, device=DEV)
        pool = -(-T // BS) + 4
        s.slots = torch.randperm(pool * BS, generator=g, device=DEV)[:T].contiguous()
        s.cache = torch.zeros(2, pool, BS, KV, D, dtype=dt, device=DEV)
    else:
        T, V, k = case["tokens"], case["vocab"], case["k"]
        s.logits = _randn((T, V), g, dt, std=2.5)
        s.idx = torch.empty(T, k, dtype=torch.int32, device=DEV)
        s.val = torch.empty(T, k, dtype=dt, device=DEV)
    return s


# --------------------------------------------------------------------- run


def run(state):
    s, kind = state, state.case["kind"]
    if kind == "mlp":
        s.mlp.encode(None, s.x, s.out, s.case["tokens"])
        return s.out
    if kind == "layer":
        s.norm.encode_residual_add_norm(None, s.x, s.res, s.normed, s.case["tokens"])
        kernels.qkv_epilogue(s.q, s.k, s.v, s.pos, s.cos, s.sin, s.slots, s.cache[0], s.cache[1],
                             bias=s.bias, layout="vllm")
        return {"normed": s.normed, "residual": s.res, "qkv": s.qkv, "cache": s.cache}
    if kind == "topk":
        kernels.topk_logits(s.logits, s.case["k"], indices=s.idx, values=s.val)
        return {"indices": s.idx, "values": s.val}
    if s.case.get("entry") == "fused":
        kernels.paged_decode(s.q, s.cache[0], s.cache[1], s.bt, s.seq_lens, scale=s.scale,
                             max_seq_len=max(s.lens), layout="kernel", output=s.out, new_keys=s.k,
                             new_values=s.v, seq_lens_host=s.lens)
    else:
        s.impl.forward(None, s.q, s.k, s.v, s.cache, s.meta, output=s.out)
    return {"out": s.out, "cache": s.cache} if s.cache is not None else {"out": s.out}


# ---------------------------------------------------------------- work done


def work(case):
    """Bytes and floating-point operations one pass cannot do without."""
    kind = case["kind"]
    if kind == "mlp":
        T, H, I = case["tokens"], case["hidden"], case["inter"]
        return {"bytes": 2 * (3 * H * I + 2 * T * H), "flops": 6 * T * H * I}
    if kind == "layer":
        T, hid = case["tokens"], case["hidden"]
        row = (case["heads"] + 2 * case["kv"]) * case["dim"]
        # x and residual read, residual and norm written; QKV read and written,
        # K and V to the cache, the token's cos/sin rows, position and slot.
        per = 2 * (4 * hid + 2 * row + 2 * case["kv"] * case["dim"]) + 4 * case["dim"] + 12
        return {"bytes": T * per + 2 * (hid + row), "flops": T * (6 * hid + 4 * row)}
    if kind == "topk":
        T = case["tokens"]
        return {"bytes": T * (2 * case["vocab"] + 6 * case["k"]), "flops": T * case["vocab"]}
    H, KV, D = case["heads"], case["kv"], case["dim"]
    lens, new = _batch(case)
    T = sum(new)
    nbytes = 2 * T * (2 * H + 2 * KV) * D  # q, out, new K/V read
    if kind == "encoder":
        return {"bytes": nbytes, "flops": sum(4 * D * H * n * n for n in new)}
    # Cached K/V read, new K/V written, block table.
    nbytes += 2 * 2 * KV * D * (sum(lens) - T) + 2 * 2 * T * KV * D + sum(-(-L // BS) * 4
                                                                        for L in lens)
    pairs = sum(n * (L - n) + n * (n + 1) // 2 for L, n in zip(lens, new))
    return {"bytes": nbytes, "flops": 4 * D * H * pairs}


def tolerance(case):
    """About four times the error against 64 bits measured on MI355X: the
    16-bit rounding of the outputs and, in fp16 attention, of the
    probabilities."""
    if case["kind"] == "topk":
        return "exact"
    bf = case["dtype"] == "bf16"
    if case["kind"] == "mlp":
        return {"rel": 9e-3 if bf else 1.8e-3}
    if case["kind"] == "layer":
        return {"rel": 7e-3 if bf else 1e-3}
    return {"rel": 7e-3 if bf else 1.5e-3}


# --------------------------------------------------------------- in 64 bits


def _rows64(cache, bt, L, fused):
    """The first L tokens of one sequence, [L, KV, D] in 64 bits."""
    n = -(-L // BS)
    x = cache[bt[:n].long()]
    if fused:
        x = x.transpose(1, 2)
    return x.reshape(n * BS, x.shape[2], x.shape[3])[:L].double()


def exact(case, seed):
    s, kind = prepare(case, seed), case["kind"]
    if kind == "mlp":
        I = case["inter"]
        x = s.x.double()
        g = x @ s.w1[:I].double().t()
        a = g * torch.sigmoid(g) * (x @ s.w1[I:].double().t())
        return a @ s.w2.double().t()
    if kind == "layer":
        H, KV, D = case["heads"], case["kv"], case["dim"]
        # The residual sum and the biased projection are stored in 16 bits
        # before the norm and the rotation read them.
        res = (s.x.double() + s.res.double()).to(_dt(case)).double()
        normed = res * torch.rsqrt(res.square().mean(1, keepdim=True) + EPS) * s.w.double()
        y = (s.qkv.double() + s.bias.double()).to(_dt(case)).double()
        y = y.view(-1, H + 2 * KV, D)
        c, n = (t[s.pos.long()].double()[:, None] for t in (s.cos, s.sin))
        a, b = y[:, :H + KV, :D // 2].clone(), y[:, :H + KV, D // 2:].clone()
        y[:, :H + KV, :D // 2] = a * c - b * n
        y[:, :H + KV, D // 2:] = a * n + b * c
        cache = s.cache.double().view(2, -1, KV, D)
        cache[0, s.slots] = y[:, H:H + KV]
        cache[1, s.slots] = y[:, H + KV:]
        return {"normed": normed, "residual": res, "qkv": y.view(s.qkv.shape),
                "cache": cache.view(s.cache.shape)}
    if kind == "topk":
        val, idx = torch.sort(s.logits.double(), dim=1, descending=True, stable=True)
        return {"indices": idx[:, :case["k"]].int(), "values": val[:, :case["k"]]}
    H, KV, D = case["heads"], case["kv"], case["dim"]
    out = torch.zeros(s.out.shape, dtype=torch.float64, device=DEV)
    fused = case.get("entry") == "fused"
    for i, (L, n) in enumerate(zip(s.lens, s.new)):
        t0, t1 = s.qsl[i], s.qsl[i + 1]
        kn, vn = s.k[t0:t1].double(), s.v[t0:t1].double()
        if s.cache is None:
            kk, vv = kn, vn
        else:
            kk, vv = (_rows64(c, s.bt[i], L, fused) for c in s.cache)
            kk[L - n:], vv[L - n:] = kn, vn
        q = s.q[t0:t1].double().view(n, KV, H // KV, D).permute(1, 2, 0, 3).contiguous()
        kk, vv = kk.permute(1, 0, 2).contiguous(), vv.permute(1, 0, 2).contiguous()
        see = None
        if s.cache is not None and n > 1:
            see = (torch.arange(L, device=DEV)[None, :]
                   <= torch.arange(L - n, L, device=DEV)[:, None])
        for h in range(KV):
            kt = kk[h].t().contiguous()
            for j in range(H // KV):
                w = (q[h, j] @ kt) * s.scale
                if see is not None:
                    w = w.masked_fill(~see, -math.inf)
                out[t0:t1, h * (H // KV) + j] = torch.softmax(w, dim=1) @ vv[h]
    # The cache is written with copies of the new rows: whole values, which
    # the outputs' comparison covers.
    return {"out": out, "cache": None} if s.cache is not None else {"out": out}
