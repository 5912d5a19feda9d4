"""The work a user of this framework has it do, as cases that can be timed and checked.

Six kinds, each through the package's public entry points:

  hard     lema_hard on projected q, k, v: the exact op of an evaluation (forward) or of training
           the value path through it (forward and backward); contiguous heads or the model's own
           [B, T, H * d] projection views
  codes    lema_from_codes on codes that are already packed, match indices wanted too
  match    latest_prev_match alone, int64 in and out as the code census and the traces call it
  store    LayerStore.exchange: one layer's retrieval step (T = 1), a chunk of a prompt, or a
           long prompt, against a table that already holds a context
  block    one transformer layer in bf16: dense over a window, or one token a stream with a store
  decoder  LemaDecoder.step: a whole model's token, every layer and the head in one graph

A run leaves its state so that the next run gives the same outputs: store keys are drawn apart
from the codes that queries expect to miss, and decode states have run until they repeat.
"""
import math

import torch
import torch.nn.functional as F

from latest_exact_match_attention_amd import latest_prev_match, lema_from_codes, lema_hard
from latest_exact_match_attention_amd.cache import HashStore, LayerStore, LemaCache
from latest_exact_match_attention_amd.decode import decoder
from latest_exact_match_attention_amd.model import Block, ModelConfig, Transformer

DTYPES = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}


def listed():
    return [
        # one short prompt of a small model: a handful of launches, nothing to amortise them
        dict(name="hard_tiny", kind="hard", B=1, H=8, T=200, d=24, dv=24, dtype="bf16",
             view=True, distinct=64, grad=False),
        # the dense op at B1 H8 T4096, 16-bit codes, fp32 values, with the gradient of v
        dict(name="hard_train_f32", kind="hard", B=1, H=8, T=4096, d=16, dv=64, dtype="f32",
             view=False, distinct=1024, grad=True),
        # a language-model layer's op in training, on projection views, ragged length
        dict(name="hard_train_lm", kind="hard", B=2, H=64, T=8001, d=24, dv=24, dtype="bf16",
             view=True, distinct=4096, grad=True),
        # a 100K-token window of the 0.8B geometry (24 heads of 64), without a store
        dict(name="hard_long", kind="hard", B=1, H=24, T=100003, d=64, dv=64, dtype="bf16",
             view=False, distinct=20000, grad=False),
        # prefill from codes: B8 H16 T16384, 24-bit Zipf codes, 64-wide bf16 values
        dict(name="codes_prefill", kind="codes", B=8, H=16, T=16384, bits=24, dv=64,
             dtype="bf16", distinct=4096),
        # the census of one 262,144-token stream: every head of a layer, int64 codes
        dict(name="match_census", kind="match", N=24, T=262144, bits=64, distinct=30000),
        # one decode step of 16 streams x 64 heads against a context of 32,768 tokens each
        dict(name="store_step", kind="store", B=16, H=64, T=1, ctx=32768, bits=32, dv=24,
             dtype="bf16", view=True),
        # a prompt fed in pieces: 4 streams x 24 heads, 200 positions a call, 64-bit codes
        dict(name="store_chunk", kind="store", B=4, H=24, T=200, ctx=8192, bits=64, dv=64,
             dtype="bf16", view=True),
        # a long prompt in one call: 24 heads x 16,384 positions, 64-bit codes
        dict(name="store_prompt", kind="store", B=1, H=24, T=16384, ctx=16384, bits=64, dv=64,
             dtype="bf16", view=True),
        # a layer of the LM's decode step, 16 streams
        dict(name="block_decode", kind="block", B=16, T=1, ctx=256, dim=1536, H=64, d=24, dv=24,
             ff=6144, store=True),
        # a layer of the LM over a window of 8,192 tokens
        dict(name="block_window", kind="block", B=1, T=8192, dim=1536, H=64, d=24, dv=24,
             ff=6144, store=False),
        # a token of the whole 0.8B-geometry model, one stream
        dict(name="decoder_token", kind="decoder", B=1, ctx=96, depth=24, dim=1536, H=24, d=64,
             dv=64, ff=4096, vocab=50304),
    ]


def _log(rng, lo, hi):
    """A whole number spread over [lo, hi] by its logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["hard", "hard", "hard", "codes", "match", "store", "store", "store",
                       "block", "block", "decoder"])
    if kind == "hard":
        H, T = rng.choice([1, 3, 8, 16, 24, 64]), _log(rng, 64, 131072)
        # a head's values and codes: at most 1.05M rows of at most 128 values
        return dict(kind=kind, B=max(1, min(rng.choice([1, 2, 4, 8]), (1 << 20) // (H * T))),
                    H=min(H, max(1, (1 << 22) // T)), T=T, d=rng.choice([8, 16, 24, 40, 64]),
                    dv=rng.choice([16, 24, 33, 64, 128]), dtype=rng.choice(["f32", "f16", "bf16"]),
                    view=rng.random() < 0.5, distinct=_log(rng, 16, 40000),
                    grad=rng.random() < 0.5)
    if kind == "codes":
        H, T = rng.choice([3, 8, 16, 64]), _log(rng, 100, 65536)
        return dict(kind=kind, B=max(1, min(rng.choice([1, 2, 8]), (1 << 21) // (H * T))),
                    H=min(H, max(1, (1 << 21) // T)), T=T, bits=rng.choice([16, 24, 64]),
                    dv=rng.choice([16, 24, 64]), dtype=rng.choice(["f32", "bf16"]),
                    distinct=_log(rng, 16, 4096))
    if kind == "match":
        T = _log(rng, 128, 262144)
        return dict(kind=kind, N=max(1, min(rng.choice([1, 8, 24, 64]), (1 << 22) // T)), T=T,
                    bits=rng.choice([32, 64]), distinct=_log(rng, 16, 60000))
    if kind == "store":
        T = rng.choice([1, _log(rng, 2, 1024), _log(rng, 1024, 16384)])
        B, H = rng.choice([1, 2, 4, 16]), rng.choice([8, 24, 64])
        B = max(1, min(B, (1 << 19) // (H * T)))
        return dict(kind=kind, B=B, H=H, T=T, ctx=_log(rng, 512, 16384),
                    bits=rng.choice([32, 64]), dv=rng.choice([24, 32, 64]),
                    dtype=rng.choice(["f16", "bf16", "f32"]), view=rng.random() < 0.7)
    geo = rng.choice([dict(dim=1536, H=64, d=24, dv=24, ff=6144),
                      dict(dim=1536, H=24, d=64, dv=64, ff=4096),
                      dict(dim=768, H=32, d=24, dv=24, ff=2048),
                      dict(dim=1024, H=16, d=64, dv=64, ff=2816)])
    if kind == "block":
        if rng.random() < 0.6:
            return dict(kind=kind, B=_log(rng, 1, 32), T=1, ctx=_log(rng, 40, 800), store=True,
                        **geo)
        return dict(kind=kind, B=1, T=_log(rng, 40, 8000), store=False, **geo)
    return dict(kind=kind, B=_log(rng, 1, 32), ctx=_log(rng, 40, 400),
                depth=rng.choice([2, 3, 6, 12]), vocab=50304, **geo)


# ------------------------------------------------------------------------------------ inputs

def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _zipf(g, shape, distinct, s=1.1):
    """Ranks 0..distinct-1 with p(r) ~ (r + 1)^-s."""
    p = torch.arange(1, distinct + 1, dtype=torch.float64, device="cuda") ** -s
    cdf = torch.cumsum(p / p.sum(), 0)
    u = torch.rand(shape, generator=g, device="cuda", dtype=torch.float64)
    return torch.searchsorted(cdf, u.reshape(-1)).view(shape).clamp_(max=distinct - 1)


def _ranks(g, rows, T, distinct):
    """Code ranks of queries and keys. Codes recur (Zipf over `distinct`), except that one
    query in four carries a code that no key has (rank >= distinct)."""
    kr, qr = _zipf(g, (rows, T), distinct), _zipf(g, (rows, T), distinct)
    lone = torch.rand((rows, T), generator=g, device="cuda") < 0.25
    own = distinct + torch.arange(T, device="cuda").expand(rows, T)
    return torch.where(lone, own, qr), kr


def _mix(x):
    """An invertible mixing of int64 words (odd multiplications and shifts)."""
    x = (x ^ ((x >> 31) & 0x1FFFFFFFF)) * 0x7FB5D329728EA185
    x = (x ^ ((x >> 27) & 0x1FFFFFFFFF)) * -0x7E25210B43D22BB3
    return x ^ ((x >> 33) & 0x7FFFFFFF)


def _signs(seed, ranks, d):
    """[rows, T] ranks -> [rows, T, d] of +-1: a rank's d pseudo-random signs in its row."""
    rows = torch.arange(ranks.shape[0], device="cuda").view(-1, 1)
    h = _mix((ranks * 8191 + rows) * 131 + seed)
    bits = (h.unsqueeze(-1) >> torch.arange(d, device="cuda")) & 1
    return bits * 2 - 1


def _preact(g, seed, ranks, B, H, T, d, dtype, view):
    """Projected queries or keys: the code's signs, magnitudes of a normal distribution."""
    z = torch.empty((B, T, H, d) if view else (B, H, T, d), dtype=dtype, device="cuda")
    out = z.transpose(1, 2) if view else z
    r = ranks.view(B, H, T)
    for b in range(B):
        for h in range(0, H, 8):
            s = _signs(seed + 1000 * b + h, r[b, h:h + 8], d)
            m = torch.randn(s.shape, generator=g, device="cuda").abs_() + 1e-3
            out[b, h:h + 8] = (s * m).to(dtype)
    return out


def _values(g, B, H, T, dv, dtype, view):
    z = torch.randn((B, T, H, dv) if view else (B, H, T, dv), generator=g,
                    device="cuda").to(dtype)
    return z.transpose(1, 2) if view else z


def _prepare_hard(c, seed):
    g, dt = _gen(seed), DTYPES[c["dtype"]]
    B, H, T = c["B"], c["H"], c["T"]
    qr, kr = _ranks(g, B * H, T, c["distinct"])
    q = _preact(g, seed, qr, B, H, T, c["d"], dt, c["view"])
    k = _preact(g, seed, kr, B, H, T, c["d"], dt, c["view"])
    v = _values(g, B, H, T, c["dv"], dt, c["view"])
    s = dict(kind="hard", q=q, k=k, v=v, grad=c["grad"])
    if c["grad"]:
        s["v"] = v.requires_grad_(True)
        s["gy"] = _values(g, B, H, T, c["dv"], dt, c["view"])
    return s


def _prepare_codes(c, seed):
    g, dt = _gen(seed), DTYPES[c["dtype"]]
    B, H, T = c["B"], c["H"], c["T"]
    ct, mask = (torch.int32, (1 << c["bits"]) - 1) if c["bits"] <= 32 else (torch.int64, -1)
    qr, kr = _ranks(g, B * H, T, c["distinct"])
    code = lambda r: (_mix(r * 131 + seed) & mask).to(ct).view(B, H, T)  # noqa: E731
    return dict(kind="codes", qc=code(qr), kc=code(kr),
                v=_values(g, B, H, T, c["dv"], dt, False))


def _prepare_match(c, seed):
    g = _gen(seed)
    mask = -1 if c["bits"] == 64 else (1 << c["bits"]) - 1
    qr, kr = _ranks(g, c["N"], c["T"], c["distinct"])
    return dict(kind="match", qc=_mix(qr * 131 + seed) & mask, kc=_mix(kr * 131 + seed) & mask)


def _store_ids(c, seed):
    """The call's (class, index) of every query and key, and the context rows queries read.
    Classes: 0 context codes that queries look up, 1 context codes that keys overwrite, 2 codes
    new with this call, 3 codes nothing holds."""
    g = _gen(seed)
    P, T, half = c["B"] * c["H"], c["T"], c["ctx"] // 2
    rnd = lambda n: torch.randint(0, n, (P, T), generator=g, device="cuda")  # noqa: E731
    uni = lambda: torch.rand((P, T), generator=g, device="cuda")  # noqa: E731
    old = uni() < 0.1
    kcls = torch.where(old, 1, 2)
    kidx = torch.where(old, rnd(half), rnd(max(1, 3 * T // 4)))
    pos = torch.arange(T, device="cuda").expand(P, T)
    back = (uni() * pos).long().clamp_(min=0)            # an earlier position of the call
    u = uni()
    ctx, copy = u < 0.3, (u >= 0.3) & (u < 0.5) & (pos > 0)
    qcls = torch.where(ctx, 0, torch.where(copy, kcls.gather(1, back), 3))
    qidx = torch.where(ctx, rnd(half), torch.where(copy, kidx.gather(1, back), rnd(1 << 29)))
    return qcls, qidx, kcls, kidx, g


def _store_code(c, seed, cls, idx):
    """Codes of (class, index): a class's indices give distinct codes, classes share none."""
    n = c["bits"] - 2
    h = (idx * 0x5851F42D4C957F2D + seed * 977) & ((1 << n) - 1)
    code = (h << 2) | cls
    if c["bits"] == 64:
        return code
    return torch.where(code >= 1 << 31, code - (1 << 32), code).to(torch.int32)


def _store_inputs(c, seed):
    dt = DTYPES[c["dtype"]]
    B, H, P, T, half = c["B"], c["H"], c["B"] * c["H"], c["T"], c["ctx"] // 2
    qcls, qidx, kcls, kidx, g = _store_ids(c, seed)
    v = _values(g, B, H, T, c["dv"], dt, c["view"])
    at = torch.arange(2 * half, device="cuda").expand(P, 2 * half)
    ctx = _store_code(c, seed, at // half, at % half)
    ctx_v = torch.randn((P, 2 * half, c["dv"]), generator=g, device="cuda", dtype=dt) \
        if dt != torch.float32 else torch.randn((P, 2 * half, c["dv"]), generator=g, device="cuda")
    qc = _store_code(c, seed, qcls, qidx).view(B, H, T)
    kc = _store_code(c, seed, kcls, kidx).view(B, H, T)
    return qc, kc, v, ctx, ctx_v, (qcls, qidx, kcls, kidx)


def _prepare_store(c, seed):
    qc, kc, v, ctx, ctx_v, _ = _store_inputs(c, seed)
    P, n = ctx.shape
    store = HashStore(c["dv"], groups=P, dtype=DTYPES[c["dtype"]],
                      capacity=2 * P * (n + c["T"]), device="cuda")
    store.exchange(None, ctx.reshape(-1), ctx_v.view(-1, c["dv"]), None, n, 0)
    return dict(kind="store", layer=LayerStore(store, 0, P), qc=qc, kc=kc, v=v)


def _config(c, depth=1):
    return ModelConfig(vocab_size=c.get("vocab", 128), depth=depth, dim=c["dim"],
                       num_heads=c["H"], d_qk=c["d"], d_v=c["dv"], dim_ff=c["ff"])


def _block(c, seed):
    """One layer with the model's initialisation; keys projected like queries, so that a token
    looks up the latest earlier one like it."""
    torch.manual_seed(seed)
    with torch.device("cuda"):
        blk = Block(_config(c))
    for m in blk.modules():
        if isinstance(m, torch.nn.Linear):
            torch.nn.init.normal_(m.weight, std=m.weight.shape[1] ** -0.5)
    with torch.no_grad():
        blk.attn.k_proj.weight.copy_(blk.attn.q_proj.weight)
    blk.attn.hard = True
    return blk.to(torch.bfloat16)


def _tokens(c, seed, n):
    """[B, n] token ids, Zipf over 4,096, and their bf16 embedding rows."""
    g = _gen(seed)
    emb = torch.randn((4096, c["dim"]), generator=g, device="cuda").to(torch.bfloat16)
    ids = _zipf(g, (c["B"], n), 4096)
    return ids, emb[ids]


@torch.no_grad()
def _prepare_block(c, seed):
    blk = _block(c, seed)
    if not c["store"]:
        return dict(kind="block", blk=blk, x=_tokens(c, seed, c["T"])[1], layer=None)
    n = c["ctx"]
    x = _tokens(c, seed, n + 1)[1]
    layer = LemaCache(_config(c), max_cache_len=2 * n, batch=c["B"], device="cuda").layer(0)
    blk(x[:, :n].contiguous(), store=layer)
    s = dict(kind="block", blk=blk, x=x[:, n:].contiguous(), layer=layer)
    for _ in range(2):  # the token itself is then the latest of its code
        run(s)
    return s


@torch.no_grad()
def _decoder_model(c, seed):
    """A model whose even layers look the token up (keys projected like queries) and whose odd
    layers find nothing."""
    torch.manual_seed(seed)
    with torch.device("cuda"):
        model = Transformer(_config(c, c["depth"]))
    for b in model.blocks[::2]:
        b.attn.k_proj.weight.copy_(b.attn.q_proj.weight)
    model.set_hard(True)
    model.requires_grad_(False)
    prompt = torch.randint(0, c["vocab"], (c["B"], c["ctx"] + 1), generator=_gen(seed),
                           device="cuda")
    return model.to(torch.bfloat16), prompt


@torch.no_grad()
def _prepare_decoder(c, seed):
    model, prompt = _decoder_model(c, seed)
    cache = model.new_cache("hbm", max_cache_len=2 * c["ctx"], batch=c["B"])
    model(prompt[:, :-1], cache=cache, return_logits=False)
    tok = prompt[:, -1:].contiguous()
    s = dict(kind="decoder", dec=decoder(model, cache, tok=tok), tok=tok)
    for _ in range(c["depth"] + 3):  # until every layer's latest entry is the token's own
        run(s)
    cache.store.check_full()
    return s


def prepare(case, seed):
    return {"hard": _prepare_hard, "codes": _prepare_codes, "match": _prepare_match,
            "store": _prepare_store, "block": _prepare_block,
            "decoder": _prepare_decoder}[case["kind"]](case, seed)


# --------------------------------------------------------------------------------------- run

def run(state):
    kind = state["kind"]
    if kind == "hard":
        y = lema_hard(state["q"], state["k"], state["v"])
        if not state["grad"]:
            return y
        (gv,) = torch.autograd.grad(y, state["v"], state["gy"])
        return y, gv
    if kind == "codes":
        return lema_from_codes(state["qc"], state["kc"], state["v"], return_src=True)
    if kind == "match":
        return latest_prev_match(state["qc"], state["kc"])
    if kind == "store":
        got = state["layer"].exchange(state["qc"], state["kc"], state["v"], check=False)
        return got, state["layer"].store.counts_device
    if kind == "block":
        blk, x, layer = state["blk"], state["x"], state["layer"]
        with torch.no_grad():
            if layer is None:
                return blk(x)
            qc, kc, v = blk.gpu_pre(x)
            return blk.gpu_post(x, layer.exchange(qc, kc, v, check=False))
    dec = state["dec"]
    dec.tok.copy_(state["tok"])
    dec.step(check=False)
    return dec.logits


# --------------------------------------------------------------------------- work, tolerance

def work(case):
    c, kind = case, case["kind"]
    es = {"f32": 4, "f16": 2, "bf16": 2}.get(c.get("dtype"), 2)
    if kind == "hard":
        n = c["B"] * c["H"] * c["T"]
        rows = 2 * c["d"] + 2 * c["dv"] + (2 * c["dv"] if c["grad"] else 0)
        return dict(bytes=n * es * rows, flops=n * c["dv"] if c["grad"] else 0)
    if kind == "codes":
        n = c["B"] * c["H"] * c["T"]
        return dict(bytes=n * (2 * (4 if c["bits"] <= 32 else 8) + 4 + 2 * c["dv"] * es), flops=0)
    if kind == "match":
        return dict(bytes=c["N"] * c["T"] * 24, flops=0)
    if kind == "store":
        n, vb = c["B"] * c["H"] * c["T"], c["dv"] * es
        # both codes, the value in, the value out, the slot looked up and the slot written
        return dict(bytes=n * (2 * c["bits"] // 8 + 2 * vb + 2 * (16 + vb)), flops=0)
    M = c["B"] * c.get("T", 1)
    qk, vv = c["H"] * c["d"], c["H"] * c["dv"]
    per = c["dim"] * (2 * qk + 2 * vv + 3 * c["ff"])
    if kind == "block":
        slots = M * c["H"] * 2 * (16 + 2 * c["dv"]) if c["store"] else 0
        return dict(bytes=2 * per + 2 * 2 * M * c["dim"] + slots, flops=2 * M * per)
    head = c["dim"] * c["vocab"]
    slots = c["depth"] * M * c["H"] * 2 * (16 + 2 * c["dv"])
    return dict(bytes=2 * (c["depth"] * per + head) + 2 * M * (c["vocab"] + c["dim"]) + slots,
                flops=2 * M * (c["depth"] * per + head))


def tolerance(case):
    kind = case["kind"]
    if kind == "hard" and case["grad"]:
        # the gradient's rows are sums: 32-bit sums in another order, or 16-bit results (bf16
        # is 1.8e-3 from 64 bits with every partial sum rounded, f16 an eighth of that)
        return {"f32": dict(rel=1e-5), "f16": dict(rel=1e-3, max=0.03),
                "bf16": dict(rel=7e-3, max=0.2)}[case["dtype"]]
    if kind == "block":  # 0.4e-2 from 64 bits
        return dict(rel=1.5e-2, max=0.2)
    if kind == "decoder":  # 1.7e-2 from 64 bits over 24 layers of bf16
        return dict(rel=3e-2, max=0.4)
    return "exact"


# ------------------------------------------------------------------------------------- exact

def _match(qc, kc):
    """[N, T] codes -> the latest j < i with kc[j] == qc[i], else -1, by one stable sort."""
    N, T = qc.shape
    both = torch.stack([qc, kc], -1).reshape(N, 2 * T)  # a position's query before its key
    code, at = torch.sort(both, dim=1, stable=True)
    place = torch.arange(2 * T, device=qc.device).expand(N, 2 * T)
    last = torch.where(at % 2 == 1, place, -1).cummax(1).values
    hit = (last >= 0) & (code.gather(1, last.clamp(min=0)) == code)
    src = torch.where(hit, at.gather(1, last.clamp(min=0)) // 2, -1)
    out = torch.empty_like(src).scatter_(1, at, src)
    return out.view(N, T, 2)[:, :, 0].contiguous()


def _pack(z):
    w = (z >= 0).long() << torch.arange(z.shape[-1], device=z.device)
    return w.sum(-1)


def _take(v, src):
    """[N, T, dv] rows at src, zeros where it is -1, in 64 bits."""
    i = src.clamp(min=0).unsqueeze(-1).expand(v.shape)
    return v.double().gather(1, i) * (src >= 0).unsqueeze(-1)


def _norm(x, eps=1e-5):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps)


def _mlp(blk, x):
    m = blk.mlp
    h = _norm(x) * blk.norm2.weight.double()
    a = F.silu(h @ m.gate.weight.double().t()) * (h @ m.up.weight.double().t())
    return x + a @ m.down.weight.double().t()


def _looked_up(blk, x, hit):
    """A layer whose tokens read the value of an equal one (where `hit`) or nothing."""
    h = _norm(x) * blk.norm1.weight.double()
    y = (h @ blk.attn.v_proj.weight.double().t()) * hit
    return _mlp(blk, x + y @ blk.attn.o_proj.weight.double().t())


@torch.no_grad()
def exact(case, seed):
    c, kind = case, case["kind"]
    if kind == "hard":
        s = prepare(c, seed)
        B, H, T, dv = s["v"].shape
        src = torch.cat([_match(_pack(s["q"][b]), _pack(s["k"][b])) for b in range(B)])
        y = _take(s["v"].reshape(B * H, T, dv), src).view(B, H, T, dv)
        if not c["grad"]:
            return y
        gv = torch.zeros((B * H, T, dv), dtype=torch.float64, device="cuda")
        gy = s["gy"].reshape(B * H, T, dv).double() * (src >= 0).unsqueeze(-1)
        gv.scatter_add_(1, src.clamp(min=0).unsqueeze(-1).expand(B * H, T, dv), gy)
        return y, gv.view(B, H, T, dv)
    if kind == "codes":
        s = prepare(c, seed)
        B, H, T, dv = s["v"].shape
        src = _match(s["qc"].view(B * H, T).long(), s["kc"].view(B * H, T).long())
        return _take(s["v"].view(B * H, T, dv), src).view(B, H, T, dv), src.view(B, H, T).int()
    if kind == "match":
        s = prepare(c, seed)
        return _match(s["qc"], s["kc"])
    if kind == "store":
        qc, _, v, _, ctx_v, (qcls, qidx, kcls, kidx) = _store_inputs(c, seed)
        B, H, T, dv = v.shape
        src = _match((qcls << 40) + qidx, (kcls << 40) + kidx)
        got = _take(v.reshape(B * H, T, dv), src)
        row = qidx.clamp(max=c["ctx"] // 2 - 1).unsqueeze(-1).expand(B * H, T, dv)
        got = torch.where((qcls == 0).unsqueeze(-1), ctx_v.gather(1, row).double(), got)
        return got.view(B, H, T, dv), None
    if kind == "block":
        blk = _block(c, seed)
        if c["store"]:
            return _looked_up(blk, _tokens(c, seed, c["ctx"] + 1)[1][:, -1:].double(), 1.0)
        ids, x = _tokens(c, seed, c["T"])
        seen = (_match(ids, ids) >= 0).unsqueeze(-1)
        return _looked_up(blk, x.double(), seen)
    model, prompt = _decoder_model(c, seed)
    x = model.tok_emb.weight[prompt[:, -1:]].double()
    for i, blk in enumerate(model.blocks):
        x = _looked_up(blk, x, 1.0 if i % 2 == 0 else 0.0)
    return (_norm(x) * model.norm_f.weight.double()) @ model.lm_head.weight.double().t()
