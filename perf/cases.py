"""Performance cases: the calls a user of the framework makes, over the range of sizes it serves.

Serving works on one set of weights for many requests, so a model's weights (seeded random
init, laid out once) are shared by all states of a case; tokens, caches, logits and gradients
come from the state's own seed.  ``exact`` restates every path in plain torch at 64 bits.
"""
import math

import numpy as np
import torch

from transformer_amd.configs import M306, TINY
from transformer_amd.fused_decode_nlayer import new_kv_packed, prepare_decode_weights_nlayer
from transformer_amd.generate import Sampler
from transformer_amd.multi_sm_decode import Decoder
from transformer_amd.paged import PAGE, PagedBatchDecoder, PagePool
from transformer_amd.prefill import Prefiller
from transformer_amd.speculative import Verifier
from transformer_amd.xent import fused_cross_entropy

# The model shapes of the package and of its shape tests.
MODELS = {
    "tiny": TINY,
    "d512": dict(vocab_size=32000, d_model=512, n_heads=8, n_kv_heads=8, n_layers=8, d_head=64, d_ff=1408,
                 context_len=256),
    "d768": dict(vocab_size=32000, d_model=768, n_heads=12, n_kv_heads=4, n_layers=12, d_head=64, d_ff=2048,
                 context_len=512),
    "306m": M306,
}
DEV = "cuda"


def listed():
    return [
        # one token of the smallest model: launch and exchange latency, nothing else
        dict(name="decode_tiny", kind="decode", model="tiny", pos=60),
        # one token of a chat or completion at batch 1, mid-context: the headline path
        dict(name="decode_306m", kind="decode", model="306m", pos=300),
        # a short greedy continuation (an autocompletion, a draft) in one launch
        dict(name="continue_306m_16", kind="continue", model="306m", pos=129, steps=16),
        # time to first token of an ordinary prompt
        dict(name="prefill_306m_128", kind="prefill", model="306m", tokens=128, every=False),
        # time to first token of a prompt that fills the context
        dict(name="prefill_306m_511", kind="prefill", model="306m", tokens=511, every=False),
        # scoring a text of odd length: the logits of every position
        dict(name="score_d768_203", kind="prefill", model="d768", tokens=203, every=True),
        # four drafted tokens and the last accepted one checked by the target model
        dict(name="verify_306m_5", kind="verify", model="306m", pos=211, tokens=5),
        # a small serving batch over the paged cache (one persistent launch)
        dict(name="batch_306m_8", kind="batch", model="306m", batch=8, longest=384),
        # a larger serving batch, past what the persistent launch takes
        dict(name="batch_306m_24", kind="batch", model="306m", batch=24, longest=384),
        # one draw from a trained model's peaked distribution with the usual sampling options
        dict(name="sample_32000", kind="sample", vocab=32000, temperature=0.7, top_p=0.95, penalty=1.2, spread=3.0),
        # the output layer of a training step of the 306M model (forward and both gradients)
        dict(name="loss_4096", kind="loss", rows=4096, vocab=32000, d=1024, chunk=4096, train=True, check=False),
        # the same layer of a small, ragged micro-batch with the default checks
        dict(name="loss_509_d768", kind="loss", rows=509, vocab=32000, d=768, chunk=4096, train=True, check=True),
    ]


def _log(rng, lo, hi):
    """An integer of lo..hi spread evenly over its logarithm."""
    return min(hi, max(lo, int(math.exp(rng.uniform(math.log(lo), math.log(hi + 1))))))


def draw(rng):
    kind = rng.choice(["decode", "continue", "prefill", "prefill", "verify", "batch", "batch", "sample", "loss", "loss"])
    if kind == "sample":
        return dict(kind=kind, vocab=_log(rng, 1000, 32768), temperature=rng.choice([0.0, 0.7, 1.0, 1.3]),
                    top_p=rng.choice([0.5, 0.9, 0.95, 1.0]), penalty=rng.choice([1.0, 1.2]),
                    spread=rng.choice([0.9, 2.0, 3.0, 4.0]))
    if kind == "loss":
        return dict(kind=kind, rows=_log(rng, 64, 4096), vocab=rng.choice([rng.randint(4000, 32000), 32000]),
                    d=rng.choice([256, 512, 768, 1024]), chunk=rng.choice([1000, 4096, 8192]),
                    train=rng.random() < 0.75, check=rng.random() < 0.5)
    model = rng.choice(["tiny", "d512", "d768", "306m", "306m"])
    ctx = MODELS[model]["context_len"]
    if kind == "decode":
        return dict(kind=kind, model=model, pos=_log(rng, 1, ctx - 1))
    if kind == "continue":
        steps = rng.randint(2, 12)
        return dict(kind=kind, model=model, pos=_log(rng, 1, ctx - steps), steps=steps)
    if kind == "prefill":
        tokens = _log(rng, 2, ctx - 1)
        return dict(kind=kind, model=model, tokens=tokens, every=tokens <= 256 and rng.random() < 0.3)
    if kind == "verify":
        tokens = rng.randint(2, 9)
        return dict(kind=kind, model=model, pos=_log(rng, 1, ctx - tokens), tokens=tokens)
    return dict(kind="batch", model=model, batch=_log(rng, 1, 24), longest=_log(rng, 32, min(ctx, 400) - 1))


# ---- weights -------------------------------------------------------------------------------

def _params(model):
    """Random-init parameters as the benchmark's (N(0, 0.02), residual projections scaled down),
    with RMSNorm scales spread around 1 as in a trained model."""
    c = MODELS[model]
    g = torch.Generator(device=DEV).manual_seed(1234)
    d, ff, L = c["d_model"], c["d_ff"], c["n_layers"]
    dkv = c["n_kv_heads"] * c["d_head"]
    res = 0.02 / math.sqrt(2 * L)

    def mat(a, b, s):
        return (torch.randn(a, b, generator=g, device=DEV) * s).to(torch.bfloat16)

    def scale():
        return (1 + 0.1 * torch.randn(d, generator=g, device=DEV)).to(torch.bfloat16)

    p = {"token_emb": mat(c["vocab_size"], d, 0.02), "ln_final.scale": scale()}
    for i in range(L):
        n = f"layer{i}"
        p.update({f"{n}.ln1.scale": scale(), f"{n}.ln2.scale": scale(), f"{n}.attn.q": mat(d, d, 0.02),
                  f"{n}.attn.k": mat(d, dkv, 0.02), f"{n}.attn.v": mat(d, dkv, 0.02),
                  f"{n}.attn.o": mat(d, d, res), f"{n}.ffn.gate": mat(d, ff, 0.02),
                  f"{n}.ffn.up": mat(d, ff, 0.02), f"{n}.ffn.down": mat(ff, d, res)})
    return p


_weights = {}


def _model(model):
    if model not in _weights:
        _weights[model] = prepare_decode_weights_nlayer(_params(model), MODELS[model], device=DEV)
    return _weights[model], MODELS[model]


# ---- inputs --------------------------------------------------------------------------------

def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed) % (1 << 62))


def _ids(n, vocab, g):
    return torch.randint(0, vocab, (n,), generator=g, device=DEV, dtype=torch.int32)


def _cache(shape, c, g):
    """Cached K and V rows at the magnitude this model's projections give."""
    s = 0.02 * math.sqrt(c["d_model"])
    return (torch.randn(shape, generator=g, device=DEV) * s).to(torch.bfloat16)


def _kv_shape(c):
    return (c["n_layers"], 2, c["n_kv_heads"], c["context_len"], c["d_head"])


def _cached(case, seed):
    """(token ids, cache) of a sequence that holds ``pos`` positions; later rows are zero."""
    c, g = MODELS[case["model"]], _gen(seed)
    kv = _cache(_kv_shape(c), c, g)
    kv[:, :, :, case["pos"]:] = 0
    return _ids(case.get("tokens", 1), c["vocab_size"], g), kv.reshape(-1)


def _batched(case, seed):
    """(tokens, positions, page rows, pool data): each sequence's pages from a shuffled pool."""
    c, g = MODELS[case["model"]], _gen(seed)
    B, r = case["batch"], np.random.RandomState(int(seed) % (1 << 31))
    pos = r.randint(max(1, case["longest"] // 8), case["longest"] + 1, B)
    need = -(-(pos + 1) // PAGE)
    n_pages = B * -(-(case["longest"] + 1) // PAGE)
    free = [int(x) for x in r.permutation(n_pages)]
    pages = [[free.pop() for _ in range(n)] for n in need]
    pool = _cache((c["n_layers"], 2, c["n_kv_heads"], n_pages * PAGE, c["d_head"]), c, g)
    return _ids(B, c["vocab_size"], g), pos.astype(np.int32), pages, pool, n_pages


def _logits(case, seed):
    g = _gen(seed)
    V = case["vocab"]
    lg = torch.randn(V, generator=g, device=DEV) * case["spread"]
    u = torch.rand(1, generator=g, device=DEV, dtype=torch.float64)
    seen = torch.randint(0, V, (200,), generator=g, device=DEV).unique()
    return lg, u, seen


def _loss_inputs(case, seed):
    g = _gen(seed)
    N, V, d = case["rows"], case["vocab"], case["d"]
    h = torch.randn(N, d, generator=g, device=DEV).to(torch.bfloat16)   # final-norm output: unit scale
    w = (torch.randn(V, d, generator=g, device=DEV) * 0.05).to(torch.bfloat16)
    t = torch.randint(0, V, (N,), generator=g, device=DEV)
    return h, w, t


def prepare(case, seed):
    k = case["kind"]
    if k == "sample":
        lg, u, seen = _logits(case, seed)
        smp = Sampler(case["vocab"], DEV)
        smp.reset(seen.tolist())
        return dict(case=case, smp=smp, logits=lg, u=u)
    if k == "loss":
        h, w, t = _loss_inputs(case, seed)
        if case["train"]:
            h.requires_grad_()
            w.requires_grad_()
        return dict(case=case, h=h, w=w, t=t)
    w, c = _model(case["model"])
    if k in ("decode", "continue"):
        tok, kv = _cached(case, seed)
        every = torch.empty((case.get("steps", 1), c["vocab_size"]), dtype=torch.float32, device=DEV)
        return dict(case=case, dec=Decoder(w, c, kv), tok=tok, every=every)
    if k == "verify":
        tok, kv = _cached(case, seed)
        return dict(case=case, ver=Verifier(w, c, max_tokens=case["tokens"]), tok=tok, kv=kv)
    if k == "prefill":
        T = case["tokens"]
        every = torch.empty((T, c["vocab_size"]), dtype=torch.float32, device=DEV) if case["every"] else None
        return dict(case=case, pf=Prefiller(w, c, max_tokens=T), tok=_ids(T, c["vocab_size"], _gen(seed)),
                    kv=new_kv_packed(c, DEV), every=every)
    tok, pos, pages, data, n_pages = _batched(case, seed)
    pool = PagePool(c, n_pages, device=DEV)
    pool.data.copy_(data.reshape(-1))
    bd = PagedBatchDecoder(w, c, pool, case["batch"])
    for b, pg in enumerate(pages):
        bd.set_pages(b, pg)
    return dict(case=case, bd=bd, tok=tok, pos=torch.from_numpy(pos).to(DEV))


def run(state):
    case = state["case"]
    k = case["kind"]
    if k == "decode":
        dec = state["dec"]
        out = dec.launch(state["tok"], case["pos"])
        return dict(logits=dec.logits, next=out, kv=dec.kv)
    if k == "continue":
        dec = state["dec"]
        out = dec.launch_steps(state["tok"], case["pos"], case["steps"], all_logits=True, logits=state["every"])
        return dict(logits=state["every"], next=out, kv=dec.kv)
    if k == "prefill":
        pf = state["pf"]
        out = pf.launch(state["tok"], state["kv"], logits_all=state["every"])
        return dict(logits=pf.logits if state["every"] is None else state["every"], next=out, kv=state["kv"])
    if k == "verify":
        logits, out = state["ver"].launch(state["tok"], case["pos"], state["kv"])
        return dict(logits=logits, next=out, kv=state["kv"])
    if k == "batch":
        bd = state["bd"]
        out = bd.launch(state["tok"], state["pos"])
        return dict(logits=bd.logits, next=out, kv=bd.pool.data)
    if k == "sample":
        smp = state["smp"]
        tok = smp.launch(state["logits"], case["temperature"], case["top_p"], case["penalty"], u=state["u"])
        return dict(token=tok, seen=smp.seen)
    loss = fused_cross_entropy(state["h"], state["w"], state["t"], case["chunk"], case["check"])
    if not case["train"]:
        return dict(loss=loss)
    gh, gw = torch.autograd.grad(loss, (state["h"], state["w"]))
    return dict(loss=loss.detach(), grad_h=gh, grad_w=gw)


# ---- what a pass cannot do without ---------------------------------------------------------

def work(case):
    k = case["kind"]
    if k == "sample":
        return {"bytes": 5 * case["vocab"], "flops": 10 * case["vocab"]}
    if k == "loss":
        N, V, d = case["rows"], case["vocab"], case["d"]
        one = 2.0 * N * V * d
        if case["train"]:
            return {"bytes": 4.0 * (N * d + V * d) + 8 * N, "flops": 3 * one}
        return {"bytes": 2.0 * (N * d + V * d) + 8 * N, "flops": one}
    c = MODELS[case["model"]]
    d, L, V, ff = c["d_model"], c["n_layers"], c["vocab_size"], c["d_ff"]
    dkv = c["n_kv_heads"] * c["d_head"]
    layer = 2 * d * d + 2 * d * dkv + 3 * d * ff            # one layer's projection weights
    row = 2 * 2 * L * dkv                                   # one position's K and V, bytes
    if k == "batch":
        rows, heads = case["batch"], case["batch"]
        cached = rows * case["longest"] * 9 // 16           # mean position of the draw
        attended = cached + rows
    else:
        rows = case.get("steps", case.get("tokens", 1))
        heads = 1 if k == "prefill" and not case["every"] else rows
        start = case.get("pos", 0)
        cached = sum(start + i for i in range(rows)) if k == "continue" else start
        attended = rows * start + rows * (rows + 1) // 2
    passes = rows if k == "continue" else 1
    nbytes = passes * 2 * (L * (layer + 2 * d) + V * d) + row * (cached + rows) + 4 * heads * V + 2 * rows * d
    flops = 2.0 * rows * L * layer + 2.0 * heads * V * d + 4.0 * L * d * attended
    return {"bytes": float(nbytes), "flops": flops}


def tolerance(case):
    k = case["kind"]
    if k == "sample":
        return "exact"
    if k == "loss":   # gradients of bf16 probabilities; the loss alone is a 32-bit sum
        return {"rel": 1e-2, "max": 3e-2} if case["train"] else {"rel": 1e-6, "max": 1e-6}
    # stored K and V may round the other way (one bf16 step each); the multi-row passes take their
    # inputs to about 2^-17, the one-row step in full f32
    rel = 2.5e-4 if k in ("decode", "continue") else 1e-3
    return {"rel": rel, "max": 2e-2, "differ": 0.0}


# ---- 64 bits -------------------------------------------------------------------------------

def _r16(x):
    return x.to(torch.bfloat16).double()


def _norm(x, s):
    return s.double() * (x / torch.sqrt((x * x).mean(-1, keepdim=True) + 1e-5))


def _rope(x, pos):
    """Rotate-half RoPE of x (n, heads, d_head) at positions ``pos`` (f32 angles, as specified)."""
    half = x.shape[-1] // 2
    i = np.arange(half, dtype=np.float32)
    freq = (np.float32(10000.0) ** (-i * np.float32(2.0) / np.float32(2 * half))).astype(np.float32)
    ang = (np.asarray(pos, dtype=np.float32)[:, None] * freq[None, :]).astype(np.float32)
    cos = torch.from_numpy(np.cos(ang)).to(DEV).double()[:, None]
    sin = torch.from_numpy(np.sin(ang)).to(DEV).double()[:, None]
    a, b = x[..., :half], x[..., half:]
    return torch.cat([a * cos - b * sin, a * sin + b * cos], -1)


def _forward(p, c, ids, start, cache, rounded):
    """Logits of ``ids`` at start.. after the cached rows, and their K/V rows (L, 2, n, KV, dh).
    ``rounded``: earlier rows of the call are attended as stored (bf16); else un-rounded."""
    H, KV, dh, n = c["n_heads"], c["n_kv_heads"], c["d_head"], len(ids)
    pos = np.arange(start, start + n)
    x = p["token_emb"][ids.long()].double()
    eye = torch.eye(n, dtype=torch.bool, device=DEV)
    later = torch.ones(n, n, dtype=torch.bool, device=DEV).triu(1)
    rows = []
    for l in range(c["n_layers"]):
        W = lambda name: p[f"layer{l}.{name}"].double()   # noqa: E731
        y = _norm(x, p[f"layer{l}.ln1.scale"])
        q = _rope((y @ W("attn.q")).view(n, H, dh), pos)
        k = _rope((y @ W("attn.k")).view(n, KV, dh), pos)
        v = (y @ W("attn.v")).view(n, KV, dh)
        rows.append(torch.stack([k, v]))
        q, k, v = q.transpose(0, 1), k.transpose(0, 1), v.transpose(0, 1)
        grp = lambda t: t.repeat_interleave(H // KV, 0).contiguous()   # noqa: E731
        kk, vv = grp(k), grp(v)
        ks, vs = (_r16(kk), _r16(vv)) if rounded else (kk, vv)
        s = torch.where(eye, (q * kk).sum(-1, keepdim=True), q @ ks.transpose(1, 2).contiguous())
        s = s.masked_fill(later, -math.inf)
        if start:
            ck, cv = (grp(cache[l, j][:, :start].double()) for j in range(2))
            s = torch.cat([q @ ck.transpose(1, 2).contiguous(), s], -1)
        a = torch.softmax(s / math.sqrt(dh), -1)
        new = a[..., start:]
        o = new.masked_fill(eye, 0.0) @ vs + torch.diagonal(new, dim1=1, dim2=2)[..., None] * vv
        if start:
            o = o + a[..., :start].contiguous() @ cv
        x = x + o.transpose(0, 1).reshape(n, H * dh) @ W("attn.o")
        y = _norm(x, p[f"layer{l}.ln2.scale"])
        g = y @ W("ffn.gate")
        x = x + (g * torch.sigmoid(g) * (y @ W("ffn.up"))) @ W("ffn.down")
    logits = _norm(x, p["ln_final.scale"]) @ p["token_emb"].double().t().contiguous()
    return logits, torch.stack(rows)


def exact(case, seed):
    k = case["kind"]
    if k == "sample":
        return None
    if k == "loss":
        h, w, t = _loss_inputs(case, seed)
        h, w, N = h.double(), w.double(), case["rows"]
        s = h @ w.t().contiguous()
        lse = torch.logsumexp(s, -1)
        loss = (lse - s.gather(1, t[:, None])[:, 0]).mean()
        if not case["train"]:
            return dict(loss=loss)
        s = torch.exp(s - lse[:, None])
        s[torch.arange(N, device=DEV), t] -= 1
        s /= N
        return dict(loss=loss, grad_h=s @ w, grad_w=s.t().contiguous() @ h)
    p, c = _params(case["model"]), MODELS[case["model"]]

    def store(kv, rows, at):   # rows (L, 2, n, KV, dh)
        kv[:, :, :, at:at + rows.shape[2]] = _r16(rows.transpose(2, 3))

    if k == "prefill":
        T = case["tokens"]
        logits, rows = _forward(p, c, _ids(T, c["vocab_size"], _gen(seed)), 0, None, False)
        kv = torch.zeros(_kv_shape(c), dtype=torch.float64, device=DEV)
        store(kv, rows, 0)
        return dict(logits=logits if case["every"] else logits[-1], next=None, kv=kv.reshape(-1))
    if k == "batch":
        tok, pos, pages, pool, _ = _batched(case, seed)
        pool, out = pool.double(), []
        for b in range(case["batch"]):
            n = int(pos[b])
            at = torch.tensor([pages[b][i // PAGE] * PAGE + i % PAGE for i in range(n + 1)], device=DEV)
            logits, rows = _forward(p, c, tok[b:b + 1], n, pool[:, :, :, at[:n]], True)
            pool[:, :, :, at[n]] = _r16(rows[:, :, 0])
            out.append(logits[0])
        return dict(logits=torch.stack(out), next=None, kv=pool.reshape(-1))
    tok, kv = _cached(case, seed)
    kv = kv.double().view(_kv_shape(c))
    out = []
    for i in range(case.get("steps", 1)):
        logits, rows = _forward(p, c, tok, case["pos"] + i, kv, True)
        store(kv, rows, case["pos"] + i)
        out.append(logits)
        tok = logits[-1:].argmax(-1)
    logits = torch.cat(out)
    return dict(logits=logits[0] if k == "decode" else logits, next=None, kv=kv.reshape(-1))
