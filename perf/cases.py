"""The workloads this engine's speed is judged by.

Each case is one call of a public entry point with what a user's program has
in hand at that moment: weights uploaded, caches filled, logits computed. The
model shapes are the repository's own (d12: 768 wide, 6 heads; d24 and its
4-layer draft: 1536 wide, 12 heads with 12 or 4 KV heads; the 256-wide model
of the parity tests; vocabularies up to 65536), the kinds:

  step       one chunk of a few tokens per row through a model on its KV cache:
             a decode or draft step (q = 1), or the verify chunk (q = k + 1)
  prefill    a prompt chunk of up to 256 tokens per row, rows of unequal length
  full       GPT.__call__: logits of every position of a batch of sequences
  attention  the attention operator over one cache layer
  linear     the linear operator (weights in row-major order, as torch has them)
  loss       the cross-entropy operator over logits rows
  stats      top-k / softmax statistics of logits rows
  sample     the token choice of one generate_fast / Engine.generate step
"""

import ctypes
import math

import numpy as np
import torch

import flaxchat_amd.torch_ops  # noqa: F401  (registers torch.ops.flaxchat_mi355x)
from flaxchat_amd import _lib
from flaxchat_amd.config import GPTConfig, compute_window_sizes, has_ve, padded_vocab
from flaxchat_amd.engine import gpt_forward
from flaxchat_amd.runtime import DeviceCache, DeviceModel, pack_operand

HD = 128  # head_dim of every configuration
OPS = torch.ops.flaxchat_mi355x


def listed():
    return [
        # one conversation: the single-token step of generate_fast on the d12
        # model (the smallest call: latency and launches count)
        dict(name="decode_one_row", kind="step", layers=12, width=768, kv=6, vocab=65536, short=1024, batch=1, q=1,
             ctx=640),
        # a draft step of the batched speculative decoder (4-layer draft, 32 rows)
        dict(name="draft_step_32", kind="step", layers=4, width=1536, kv=12, vocab=65536, short=1024, batch=32, q=1,
             ctx=1300),
        # the verify chunk of the same decoder: 6 drafts + 1 pending token per
        # row, logits of all 7 positions (4 of the target's layers)
        dict(name="verify_chunk_32x7", kind="step", layers=4, width=1536, kv=12, vocab=65536, short=1024, batch=32,
             q=7, ctx=1300),
        # a prompt chunk of a batch of unequal prompts, some of it behind them
        dict(name="prefill_16_rows", kind="prefill", layers=4, width=1536, kv=12, vocab=65536, short=1024, batch=16,
             q=256, ctx=512),
        # scoring whole sequences: GPT.__call__ on the d12 model
        dict(name="full_bf16", kind="full", layers=12, width=768, kv=6, vocab=65536, short=1024, batch=4, seq=1500,
             dtype="bf16"),
        # the same in fp32 on the small parity model (what a port is checked with)
        dict(name="full_fp32", kind="full", layers=4, width=256, kv=2, vocab=8192, short=256, batch=2, seq=500,
             dtype="fp32"),
        # the large-batch, long-context verify attention: 128 rows, 12 query
        # heads on 4 KV heads, 9 tokens per row
        dict(name="attention_verify_gqa", kind="attention", heads=12, kv=4, batch=128, q=9, ctx=6400, window=0,
             dtype="bf16"),
        # causal attention of prompt chunks
        dict(name="attention_prompt", kind="attention", heads=12, kv=12, batch=8, q=1000, ctx=500, window=1024,
             dtype="bf16"),
        # the MLP's first matrix over a ragged number of tokens
        dict(name="linear_mlp", kind="linear", m=1000, n=6144, k=1536, softcap=False, dtype="bf16"),
        # per-token loss of evaluation batches
        dict(name="loss_rows", kind="loss", rows=2000, vocab=65536),
        # keep sets of the verify rows at the default top_k
        dict(name="stats_verify_rows", kind="stats", rows=224, vocab=65536, temperature=0.8, top_k=40),
        # the token choice of a 16-row decode step at the default top_k
        dict(name="sample_16_rows", kind="sample", rows=16, vocab=65536, temperature=0.8, top_k=40),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _vocab(rng):
    return rng.choice([65536, 32768, 8192, rng.randrange(8000, 65500)])


def draw(rng):
    kind = rng.choice(["step", "step", "step", "prefill", "full", "full", "attention", "attention", "linear",
                       "loss", "stats", "sample"])
    if kind == "step":
        width, kv = rng.choice([(768, 6), (1536, 12), (1536, 4)])
        layers = rng.choice([2, 4, 12]) if width == 768 else rng.choice([2, 4])
        batch = _log(rng, 1, 128)
        return dict(kind=kind, layers=layers, width=width, kv=kv, vocab=_vocab(rng), short=1024, batch=batch,
                    q=rng.choice([1, 1, 1, 3, 5, 7, 9]), ctx=_log(rng, 32, 1900))
    if kind == "prefill":
        width, kv = rng.choice([(768, 6), (1536, 12), (1536, 4)])
        return dict(kind=kind, layers=rng.choice([2, 4]), width=width, kv=kv, vocab=_vocab(rng), short=1024,
                    batch=_log(rng, 1, 32), q=rng.choice([256, 256, rng.randrange(17, 256)]),
                    ctx=rng.choice([0, 256, rng.randrange(0, 1200)]))
    if kind == "full":
        if rng.random() < 0.4:
            return dict(kind=kind, layers=rng.choice([2, 4]), width=256, kv=2, vocab=8192, short=256,
                        batch=rng.randrange(1, 5), seq=_log(rng, 20, 600), dtype="fp32")
        return dict(kind=kind, layers=rng.choice([4, 12]), width=768, kv=6, vocab=_vocab(rng), short=1024,
                    batch=rng.randrange(1, 5), seq=_log(rng, 64, 1500), dtype="bf16")
    if kind == "attention":
        heads, kv = rng.choice([(6, 6), (12, 12), (12, 4)])
        dtype = rng.choice(["bf16", "bf16", "bf16", "fp32"])
        q = rng.choice([1, 1, 5, 7, 9, rng.randrange(64, 1000)])
        if q >= 64:
            return dict(kind=kind, heads=heads, kv=kv, batch=_log(rng, 1, 8 if dtype == "bf16" else 2),
                        q=q if dtype == "bf16" else min(q, 256), ctx=rng.randrange(0, 1500),
                        window=rng.choice([0, 1024]), dtype=dtype)
        return dict(kind=kind, heads=heads, kv=kv, batch=_log(rng, 1, 64 if dtype == "bf16" else 8), q=q,
                    ctx=_log(rng, 100, 6400 if dtype == "bf16" else 2000), window=rng.choice([0, 1024]), dtype=dtype)
    if kind == "linear":
        n, k = rng.choice([(2304, 768), (768, 768), (3072, 768), (768, 3072), (4608, 1536), (1536, 1536),
                           (6144, 1536), (1536, 6144)])
        if rng.random() < 0.25:
            return dict(kind=kind, m=_log(rng, 1, 256), n=n, k=k, softcap=False, dtype="fp32")
        if rng.random() < 0.25:
            return dict(kind=kind, m=_log(rng, 1, 512), n=65536, k=rng.choice([768, 1536]), softcap=True,
                        dtype="bf16")
        return dict(kind=kind, m=_log(rng, 1, 8192), n=n, k=k, softcap=False, dtype="bf16")
    if kind == "loss":
        return dict(kind=kind, rows=_log(rng, 1, 2000), vocab=_vocab(rng))
    if kind == "stats":
        return dict(kind=kind, rows=_log(rng, 1, 256), vocab=_vocab(rng),
                    temperature=rng.choice([0.8, 1.0, 0.6, 0.0]), top_k=rng.choice([40, 40, 0, 1, 50, 200]))
    return dict(kind=kind, rows=_log(rng, 1, 128), vocab=_vocab(rng), temperature=rng.choice([0.8, 1.0, 0.0]),
                top_k=rng.choice([40, 40, 0, 50, 200]))


# ---------------------------------------------------------------- inputs
def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _rows_of(case):
    """(tokens per row, position of each row's first token): unequal rows."""
    B, q, ctx = case["batch"], case["q"], case["ctx"]
    r = np.random.default_rng([B, q, ctx])
    n = np.full(B, q)
    if q > 16:  # prompt chunks: the last piece of a prompt may be shorter
        n = r.integers(max(1, q // 2), q + 1, B)
        n[r.integers(0, B)] = q
    start = r.integers(ctx * 3 // 4, ctx + 1, B)
    return n, start


def _config(case):
    return GPTConfig(sequence_len=2048, vocab_size=case["vocab"], n_layer=case["layers"],
                     n_head=case["width"] // HD, n_kv_head=case["kv"], n_embd=case["width"], window_pattern="SSSL",
                     short_window=case["short"])


def _weights(case, seed, dtype):
    """Row-major weights of a randomly initialised model, N(0, 0.02)."""
    g, c = _gen(seed), _config(case)
    D, H, G, L, Vp = c.n_embd, c.n_head, c.n_kv_head, c.n_layer, padded_vocab(c)

    def nrm(*shape, dt=dtype):
        out = torch.empty(*shape, device="cuda", dtype=dt)
        flat = out.view(-1)
        for s in range(0, flat.numel(), 1 << 26):
            e = min(flat.numel(), s + (1 << 26))
            flat[s:e] = torch.randn(e - s, device="cuda", generator=g) * 0.02
        return out

    w = dict(wte=nrm(Vp, D), lm_head=nrm(Vp, D), smear_gate=nrm(24, dt=torch.float32), layers=[])
    for i in range(L):
        lt = dict(wqkv=nrm((H + 2 * G) * HD, D), wo=nrm(D, D), wfc=nrm(4 * D, D), wproj=nrm(D, 4 * D))
        if has_ve(i, L):
            lt["ve"] = nrm(Vp, G * HD)
            lt["ve_gate"] = nrm(G, 12, dt=torch.float32)
        w["layers"].append(lt)
    den = max(L - 1, 1)
    w["resid"] = [float(np.float32(1.15 - 0.10 * i / den)) for i in range(L)]
    w["x0"] = [float(np.float32(0.20 - 0.15 * i / den)) for i in range(L)]
    w["smear_lambda"], w["backout_lambda"] = 0.5, float(np.float32(0.2))
    n = c.sequence_len
    inv = (1.0 / (np.float32(100000.0) ** (np.arange(0, HD, 2, dtype=np.float32) / np.float32(HD)))).astype(np.float32)
    f = np.outer(np.arange(n, dtype=np.float32), inv).astype(np.float32)
    w["cos"] = torch.from_numpy(np.cos(f)).cuda()
    w["sin"] = torch.from_numpy(np.sin(f)).cuda()
    return w


def _model(case, w, dtype):
    code = _lib.FC_BF16 if dtype == torch.bfloat16 else _lib.FC_F32
    mat = pack_operand if dtype == torch.bfloat16 else (lambda t: t)
    layers = [dict(lt, **{k: mat(lt[k]) for k in ("wqkv", "wo", "wfc", "wproj")}) for lt in w["layers"]]
    tensors = dict(wte=w["wte"], lm_head=mat(w["lm_head"]), layers=layers, rope_cos=w["cos"], rope_sin=w["sin"],
                   smear_gate=w["smear_gate"])
    scalars = dict(resid=w["resid"], x0=w["x0"], smear_lambda=w["smear_lambda"], backout_lambda=w["backout_lambda"])
    return DeviceModel(_config(case), code, torch.device("cuda", torch.cuda.current_device()), tensors, scalars)


def _ids(seed, n, vocab):
    return np.random.default_rng(seed).integers(0, vocab, n).astype(np.int32)


def _logits(g, rows, vocab):
    """Softcapped logits with a trained model's spread: a few likely tokens."""
    z = torch.randn(rows, vocab, device="cuda", generator=g) * 2.5
    return 15.0 * torch.tanh(z / 15.0)


def _chunk(case, seed, dtype):
    """A packed chunk on a filled cache."""
    n, start = _rows_of(case)
    off = np.zeros(case["batch"] + 1, np.int32)
    off[1:] = np.cumsum(n)
    ids = _ids(seed, int(off[-1]), case["vocab"])
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a, dtype=np.int32)).cuda()  # noqa: E731
    return n, start, off, ids, dev(ids), dev(off), dev(start)


def _fill_cache(case, seed, cache):
    g = _gen(seed + 1)
    # filled layer by layer: keys are 1.2 x unit-RMS after the QK norm
    for i in range(cache.k.shape[0]):
        cache.k[i] = torch.randn(cache.k[i].shape, device="cuda", generator=g) * 1.2
        cache.v[i] = torch.randn(cache.v[i].shape, device="cuda", generator=g) * 0.5
    cache.hist.copy_(torch.randn(cache.hist.shape, device="cuda", generator=g))


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("step", "prefill"):
        dt = torch.bfloat16
        dm = _model(case, _weights(case, seed, dt), dt)
        n, start, off, ids, tok, roff, st = _chunk(case, seed, dt)
        cache = DeviceCache(dm, case["batch"], int((start + n).max()) + 32)
        _fill_cache(case, seed, cache)
        n_out = case["q"] if kind == "step" else 1
        logits = torch.zeros(case["batch"], n_out, dm.V, device="cuda", dtype=torch.float32)
        nb = _lib.lib().fc_forward_workspace_bytes(ctypes.byref(dm.desc), case["batch"], tok.numel(), int(n.max()), 0)
        return dict(kind=kind, dm=dm, cache=cache, tok=tok, off=roff, start=st, mpr=int(n.max()), n_out=n_out,
                    logits=logits, ws=torch.zeros(nb, device="cuda", dtype=torch.uint8))
    if kind == "full":
        dt = torch.bfloat16 if case["dtype"] == "bf16" else torch.float32
        dm = _model(case, _weights(case, seed, dt), dt)
        return dict(kind=kind, dm=dm, ids=_ids(seed, (case["batch"], case["seq"]), case["vocab"]))
    if kind == "attention":
        q, k, v, n, start, off = _attention_inputs(case, seed)
        return dict(kind=kind, q=q, k=k, v=v, off=torch.from_numpy(off).cuda(),
                    start=torch.from_numpy(start.astype(np.int32)).cuda(), mpr=int(n.max()), window=case["window"])
    if kind == "linear":
        x, w = _linear_inputs(case, seed)
        return dict(kind=kind, x=x, w=w, softcap=case["softcap"])
    g = _gen(seed)
    z = _logits(g, case["rows"], case["vocab"])
    if kind == "loss":
        return dict(kind=kind, z=z, t=_targets(case, seed))
    if kind == "stats":
        return dict(kind=kind, z=z, T=case["temperature"], top_k=case["top_k"])
    B = case["rows"]
    i32 = dict(dtype=torch.int32, device="cuda")
    return dict(kind=kind, z=z, B=B, V=case["vocab"], T=case["temperature"], top_k=min(case["top_k"], case["vocab"]),
                seed=seed, forced=torch.full((B,), -1, **i32), gen=torch.zeros(B, 4096, **i32),
                pos=torch.full((B,), 100, **i32), step=torch.zeros(B, **i32), tok=torch.zeros(B, **i32),
                stats=torch.zeros(B, ctypes.sizeof(_lib.FcRowstat) // 4, **i32))


def _attention_inputs(case, seed):
    g = _gen(seed)
    n, start = _rows_of(case)
    off = np.zeros(case["batch"] + 1, np.int32)
    off[1:] = np.cumsum(n)
    cap = (int((start + n).max()) + 31) // 32 * 32
    dt = torch.bfloat16 if case["dtype"] == "bf16" else torch.float32
    B, G = case["batch"], case["kv"]
    q = (torch.randn(int(off[-1]), case["heads"], HD, device="cuda", generator=g) * 1.2).to(dt)
    k = torch.empty(B, G, cap, HD, device="cuda", dtype=dt)
    v = torch.empty(B, G, cap // 32, HD, 32, device="cuda", dtype=dt)
    for b in range(0, B, 16):
        k[b:b + 16] = torch.randn(k[b:b + 16].shape, device="cuda", generator=g) * 1.2
        v[b:b + 16] = torch.randn(v[b:b + 16].shape, device="cuda", generator=g) * 0.5
    return q, k, v, n, start, off


def _linear_inputs(case, seed):
    g = _gen(seed)
    dt = torch.bfloat16 if case["dtype"] == "bf16" else torch.float32
    x = torch.randn(case["m"], case["k"], device="cuda", generator=g).to(dt)
    w = (torch.randn(case["n"], case["k"], device="cuda", generator=g) * 0.02).to(dt)
    return x, w


def _targets(case, seed):
    t = _ids(seed, case["rows"], case["vocab"])
    t[np.random.default_rng(seed + 1).random(case["rows"]) < 0.1] = -1  # masked positions
    return torch.from_numpy(t).cuda()


# ---------------------------------------------------------------- the pass
def run(s):
    kind = s["kind"]
    if kind in ("step", "prefill"):
        dm, c = s["dm"], s["cache"]
        OPS.forward(ctypes.addressof(dm.desc), c.k, c.v, c.hist, s["tok"], s["off"], s["start"], s["mpr"], s["n_out"],
                    s["logits"], s["ws"])
        return dict(logits=s["logits"], k=c.k, v=c.v, hist=c.hist)
    if kind == "full":
        return gpt_forward(s["dm"], s["ids"])
    if kind == "attention":
        return OPS.attention(s["q"], s["k"], s["v"], s["off"], s["start"], s["mpr"], s["window"])
    if kind == "linear":
        return OPS.linear(s["x"], s["w"], s["softcap"])
    if kind == "loss":
        return OPS.cross_entropy(s["z"], s["t"])
    if kind == "stats":
        return list(OPS.row_stats(s["z"], s["T"], s["top_k"]))
    _lib.check(_lib.lib().fc_engine_sample(
        s["z"].data_ptr(), s["B"], s["V"], s["T"], s["top_k"], s["seed"], s["forced"].data_ptr(), s["gen"].data_ptr(),
        s["gen"].shape[1], s["pos"].data_ptr(), s["step"].data_ptr(), s["tok"].data_ptr(), s["stats"].data_ptr(),
        torch.cuda.current_stream().cuda_stream), "fc_engine_sample")
    f = s["stats"].view(torch.float32)
    return dict(token=s["tok"], gen=s["gen"], mx=f[:, 0], sum=f[:, 1], tau=f[:, 2], tie=s["stats"][:, 3],
                argmax=s["stats"][:, 4])


# ---------------------------------------------------------------- what a pass cannot do without
def _model_work(case, tokens, keys, pairs, n_logits, es):
    """tokens fed; keys: K/V positions read, and pairs: (query, key) pairs, each
    as (short, full) sums over rows; n_logits rows of logits."""
    D, G, L, V = case["width"], case["kv"], case["layers"], case["vocab"]
    per = (D + 2 * G * HD) * D + D * D + 8 * D * D
    n_ve = sum(1 for i in range(L) if has_ve(i, L))
    full = [w == 2048 for w, _ in compute_window_sizes(_config(case))]
    nb = L * per * es + tokens * D * es + n_ve * tokens * G * HD * es + 2 * tokens * D * 4
    fl = 2.0 * L * per * tokens
    for f in full:
        nb += (keys[int(f)] + tokens) * G * HD * 2 * es
        fl += 4.0 * pairs[int(f)] * D
    nb += (V * D * es + n_logits * V * 4) if n_logits else 0
    fl += 2.0 * n_logits * V * D
    return dict(bytes=float(nb), flops=float(fl))


def _pairs(n, start, window):
    """(distinct keys read, (query, key) pairs) of one row."""
    pos = np.arange(start, start + n)
    lo = np.maximum(0, pos - window) if window > 0 else np.zeros_like(pos)
    return int(pos[-1] + 1 - lo[0]), int((pos - lo + 1).sum())


def work(case):
    kind = case["kind"]
    if kind in ("step", "prefill"):
        n, start = _rows_of(case)
        sh = [_pairs(a, b, case["short"]) for a, b in zip(n, start)]
        fu = [_pairs(a, b, 0) for a, b in zip(n, start)]
        keys = [sum(x[0] for x in sh) - int(n.sum()), sum(x[0] for x in fu) - int(n.sum())]
        return _model_work(case, int(n.sum()), keys, [sum(x[1] for x in sh), sum(x[1] for x in fu)],
                           case["batch"] * (case["q"] if kind == "step" else 1), 2)
    if kind == "full":
        B, T = case["batch"], case["seq"]
        pr = [B * _pairs(T, 0, case["short"])[1], B * _pairs(T, 0, 0)[1]]
        w = _model_work(case, B * T, [0, 0], pr, B * T, 2 if case["dtype"] == "bf16" else 4)
        return w
    if kind == "attention":
        es = 2 if case["dtype"] == "bf16" else 4
        n, start = _rows_of(case)
        p = [_pairs(a, b, case["window"]) for a, b in zip(n, start)]
        qo = 2 * int(n.sum()) * case["heads"] * HD * es
        return dict(bytes=float(sum(x[0] for x in p) * case["kv"] * HD * 2 * es + qo),
                    flops=4.0 * sum(x[1] for x in p) * case["heads"] * HD)
    if kind == "linear":
        es = 2 if case["dtype"] == "bf16" else 4
        m, n, k = case["m"], case["n"], case["k"]
        return dict(bytes=float((m + n) * k * es + m * n * 4), flops=2.0 * m * n * k)
    nb = case["rows"] * case["vocab"] * 4.0
    return dict(bytes=nb + case["rows"] * (8 if kind == "loss" else 32), flops=3.0 * case["rows"] * case["vocab"])


# ---------------------------------------------------------------- tolerance
def tolerance(case):
    """About four times the distance to `exact` that the sizes above show:
    0.3% for bf16 models (0.2% for one attention layer), 1e-7 to 4e-7 for
    fp32 results and sums; the bf16 head's softcap is within 5e-6 of
    15 tanh(z / 15) in absolute value."""
    kind = case["kind"]
    if kind in ("step", "prefill") or (kind == "full" and case["dtype"] == "bf16"):
        return {"rel": 0.012}
    if kind == "attention" and case["dtype"] == "bf16":
        return {"rel": 0.0085}
    if kind == "linear" and case["softcap"]:
        return {"rel": 5e-6}
    return {"rel": 1.5e-6}


# ---------------------------------------------------------------- the same in 64 bits
def _plain_k(k):
    """[.. cap][128] keys of a bf16 cache layer: 32-key blocks, element (key
    kk, dim d) at ((2 (d / 32) + (kk / 4) % 2) 64 + 4 (kk / 8) + kk % 4 +
    16 ((d / 8) % 4)) 8 + d % 8."""
    shape = k.shape
    b = k.reshape(-1, 4, 2, 4, 4, 4, 8)        # block, d/32, (kk/4)%2, (d/8)%4, kk/8, kk%4, d%8
    return b.permute(0, 4, 2, 5, 1, 3, 6).reshape(shape)


def _plain_v(v):
    """[.. cap / 32][128][32] values as [.. cap][128]."""
    return v.transpose(-1, -2).reshape(*v.shape[:-3], -1, HD)


def _attend(q, k, v, start, window):
    """q [n][H][128] at positions start.., k / v [G][keys][128], all double."""
    n, H = q.shape[:2]
    rep = H // k.shape[0]
    pos = torch.arange(start, start + n, device=q.device)[:, None]
    key = torch.arange(k.shape[1], device=q.device)[None, :]
    see = key <= pos
    if window > 0:
        see &= pos - key <= window
    qg = q.transpose(0, 1).reshape(k.shape[0], rep * n, HD)             # [G][rep * n]
    s = torch.matmul(qg, k.transpose(1, 2).contiguous()) / math.sqrt(HD)
    s = s.masked_fill(~see.repeat(rep, 1), -math.inf)
    o = torch.matmul(torch.softmax(s, -1), v)
    return o.reshape(H, n, HD).transpose(0, 1).reshape(n, H * HD)


def _norm(x):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + 1e-6)


def _forward64(case, w, tok, n, start, hist, kv, full_smear, n_out):
    """Packed rows through the model in double; kv(layer, row) gives the plain
    cached keys and values below the row's first position. Softcapped logits
    of the last n_out tokens of every row."""
    c = _config(case)
    D, H, G, L = c.n_embd, c.n_head, c.n_kv_head, c.n_layer
    wins = [a for a, _ in compute_window_sizes(c)]
    off = np.concatenate([[0], np.cumsum(n)])
    dd = lambda t: t.double()  # noqa: E731
    emb = _norm(dd(w["wte"][tok]))
    gate = w["smear_lambda"] * torch.sigmoid(emb[:, :24] @ dd(w["smear_gate"]))
    x = torch.empty_like(emb)
    pos = torch.empty(len(tok), dtype=torch.long, device="cuda")
    for b in range(len(n)):
        prev = hist[b] if hist is not None else torch.zeros(D, dtype=torch.float64, device="cuda")
        pos[off[b]:off[b + 1]] = torch.arange(start[b], start[b] + n[b], device="cuda")
        if full_smear:
            e = emb[off[b]:off[b + 1]]
            x[off[b]:off[b + 1]] = e + gate[off[b]:off[b + 1], None] * torch.cat([prev[None], e[:-1]])
            continue
        for j in range(off[b], off[b + 1]):
            prev = emb[j] + gate[j] * prev
            x[j] = prev
    x0, xb = x, None
    cos, sin = dd(w["cos"])[pos][:, None], dd(w["sin"])[pos][:, None]

    def rope(t):
        a, b = t[..., :HD // 2], t[..., HD // 2:]
        return torch.cat([a * cos + b * sin, b * cos - a * sin], -1)

    for i in range(L):
        lt = w["layers"][i]
        x = w["resid"][i] * x + w["x0"][i] * x0
        h = _norm(x)
        qkv = h @ dd(lt["wqkv"]).t()
        q = _norm(rope(qkv[:, :H * HD].reshape(-1, H, HD))) * 1.2
        k = _norm(rope(qkv[:, H * HD:(H + G) * HD].reshape(-1, G, HD))) * 1.2
        v = qkv[:, (H + G) * HD:].reshape(-1, G, HD)
        if "ve" in lt:
            gv = 3 * torch.sigmoid(h[:, :12] @ dd(lt["ve_gate"]).t())
            v = v + gv[..., None] * dd(lt["ve"][tok]).reshape(-1, G, HD)
        y = torch.empty_like(x)
        for b in range(len(n)):
            a, e = off[b], off[b + 1]
            ck, cv = kv(i, b)
            kk = torch.cat([ck, k[a:e].transpose(0, 1)], 1)
            vv = torch.cat([cv, v[a:e].transpose(0, 1)], 1)
            y[a:e] = _attend(q[a:e], kk, vv, int(start[b]), wins[i])
        x = x + y @ dd(lt["wo"]).t()
        x = x + torch.relu(_norm(x) @ dd(lt["wfc"]).t()) ** 2 @ dd(lt["wproj"]).t()
        if i == L // 2:
            xb = x
    x = x - w["backout_lambda"] * xb
    last = np.concatenate([np.arange(off[b + 1] - n_out, off[b + 1]) for b in range(len(n))])
    z = _norm(x[torch.from_numpy(last).cuda()]) @ dd(w["lm_head"][:case["vocab"]]).t()
    return 15 * torch.tanh(z / 15)


def exact(case, seed):
    kind = case["kind"]
    if kind in ("step", "prefill"):
        dt = torch.bfloat16
        w = _weights(case, seed, dt)
        n, start, off, ids, tok, _, _ = _chunk(case, seed, dt)
        B, L, G = case["batch"], case["layers"], case["kv"]
        cap = (int((start + n).max()) + 32 + 31) // 32 * 32

        class Cache:  # the shapes and types of the engine's cache
            k = torch.empty(L, B, G, cap, HD, device="cuda", dtype=dt)
            v = torch.empty(L, B, G, cap // 32, HD, 32, device="cuda", dtype=dt)
            hist = torch.empty(B, cap, case["width"], device="cuda")

        _fill_cache(case, seed, Cache)

        def kv(i, b):
            return (_plain_k(Cache.k[i, b])[:, :start[b]].double(), _plain_v(Cache.v[i, b])[:, :start[b]].double())

        hist = [Cache.hist[b, start[b] - 1].double() if start[b] > 0 else
                torch.zeros(case["width"], device="cuda", dtype=torch.float64) for b in range(B)]
        n_out = case["q"] if kind == "step" else 1
        z = _forward64(case, w, tok.long(), n, start, hist, kv, False, n_out)
        return dict(logits=z.view(B, n_out, case["vocab"]), k=None, v=None, hist=None)
    if kind == "full":
        dt = torch.bfloat16 if case["dtype"] == "bf16" else torch.float32
        w = _weights(case, seed, dt)
        B, T, G = case["batch"], case["seq"], case["kv"]
        tok = torch.from_numpy(_ids(seed, (B, T), case["vocab"])).cuda().long().view(-1)
        none = torch.empty(G, 0, HD, device="cuda", dtype=torch.float64)
        z = _forward64(case, w, tok, np.full(B, T), np.zeros(B, int), None, lambda i, b: (none, none), True, T)
        return z.view(B, T, case["vocab"])
    if kind == "attention":
        q, k, v, n, start, off = _attention_inputs(case, seed)
        out = torch.empty(q.shape[0], q.shape[1] * HD, device="cuda", dtype=torch.float64)
        for b in range(case["batch"]):
            end = int(start[b] + n[b])
            kb = (_plain_k(k[b]) if case["dtype"] == "bf16" else k[b])[:, :end].double()
            vb = _plain_v(v[b])[:, :end].double()
            out[off[b]:off[b + 1]] = _attend(q[off[b]:off[b + 1]].double(), kb, vb, int(start[b]), case["window"])
        return out
    if kind == "linear":
        x, w = _linear_inputs(case, seed)
        z = x.double() @ w.double().t()
        return 15 * torch.tanh(z / 15) if case["softcap"] else z
    z = _logits(_gen(seed), case["rows"], case["vocab"])
    if kind == "loss":
        t = _targets(case, seed).long()
        zd = z.double()
        nll = torch.logsumexp(zd, -1) - zd.gather(1, t.clamp(min=0)[:, None])[:, 0]
        return torch.where(t >= 0, nll, torch.zeros_like(nll))
    T, top_k, V = case["temperature"], case["top_k"], case["vocab"]
    keep = z
    tau = torch.full((case["rows"],), -math.inf, device="cuda", dtype=torch.float64)
    if T > 0 and 0 < top_k < V:
        keep = torch.topk(z, top_k, dim=-1).values
        tau = keep[:, -1].double()
    if T > 0:
        y = keep.double() / T
        mx = y.amax(-1)
        total = torch.exp(y - mx[:, None]).sum(-1)
    else:
        mx, total = torch.zeros_like(tau), torch.ones_like(tau)
    if kind == "stats":
        return [mx, total, tau, None, None]
    return dict(token=None, gen=None, mx=mx, sum=total, tau=tau, tie=None, argmax=None)
