"""The work that programs have this package do, as cases to measure.

Each case names a path (`kind`) and its sizes:

  attn     one decode step's attention of one layer, decode_attention(q, k_cache, v_cache),
           over the compressed caches or the plain bf16 ones, whole context or a window
  steps    a batch's cache work in one layer: prefill of every slot, then decode steps
           (append to K and V, attention, check_overflow at page ends), contiguous caches
  paged    the same for sequences of different lengths over a pool of pages, through
           PageTable: join, decode together, leave, pool compacted
  prefill  one layer's prompt K and V into a cache slot, read in the attention module's
           [1, H, T, D] layout (what Engine.prefill does per layer and prompt)
  codec    encode_reference, then decode_reference
  wire     sequences packed into blobs and unpacked into another cache (offload, migration)
  engine   Engine over a small decoder: prompts prefilled, then decode steps with given
           next tokens, logits of every step

Keys and values follow the package's synthetic recipe (per-channel scales, rotary
embedding on keys, 0.04% exact zeros, 0.3% of token rows with an outlier that makes them
raw), made on the GPU so that preparing is quick."""
import math

import torch
import torch.nn.functional as F

import exactkv_amd as exactkv
from exactkv_amd import wire

DEV = "cuda"
PAGE = 16
RAW_ROWS, ZEROS = 3e-3, 4e-4
POOL = 0.04          # raw rows reserved, a share of all: above what the data has, so pools keep their size


# ---------------------------------------------------------------- the cases

def listed():
    return [
        # the smallest call: one chat sequence of about a thousand tokens; latency
        dict(name="attn_short", kind="attn", cache="compressed", B=1, T=997, Hq=32, Hkv=8, D=128, window=0),
        # one long document in a 28q/4kv model, an odd length just under 32K
        dict(name="attn_one_32k", kind="attn", cache="compressed", B=1, T=32763, Hq=28, Hkv=4, D=128, window=0),
        # the benchmark's headline shape: 8 sequences of 8K
        dict(name="attn_8x8k", kind="attn", cache="compressed", B=8, T=8192, Hq=32, Hkv=8, D=128, window=0),
        # a serving batch: the largest, all bandwidth
        dict(name="attn_serving", kind="attn", cache="compressed", B=128, T=4339, Hq=32, Hkv=8, D=128, window=0),
        # the uncompressed cache, the option a user compares with
        dict(name="attn_bf16", kind="attn", cache="bf16", B=8, T=8185, Hq=32, Hkv=8, D=128, window=0),
        # a small model's head dim at a medium batch, ragged last page
        dict(name="attn_d64", kind="attn", cache="compressed", B=24, T=4093, Hq=32, Hkv=8, D=64, window=0),
        # a short answer for a batch of eight: prompts of 500, 40 tokens, two page ends
        dict(name="steps_batch8", kind="steps", B=8, T=501, N=40, Hq=32, Hkv=8, D=128),
        # continuous batching: twelve sequences of mixed lengths, 24 tokens
        dict(name="paged_mixed12", kind="paged", B=12, T=1500, N=24, Hq=32, Hkv=8, D=128),
        # one prompt of about 4K tokens, one layer
        dict(name="prefill_4k", kind="prefill", T=4091, Hkv=8, D=128),
        # a whole prefill batch through the codec
        dict(name="codec_batch", kind="codec", B=16, T=4096, Hkv=8, D=128),
        # eight sequences moved to another cache
        dict(name="wire_move8", kind="wire", B=8, T=4101, Hkv=8, D=128),
        # four prompts of 300 tokens and 40 decode steps of a two-layer model
        dict(name="engine_small", kind="engine", B=4, T=300, N=40, Hq=16, Hkv=4, D=128, hidden=2048),
    ]


def _spread(rng, lo, hi):
    """A whole number from lo to hi, even over its logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


_HEADS = [(32, 8), (28, 4), (32, 32), (16, 2), (14, 2), (40, 8), (24, 6), (8, 1), (64, 8)]


def draw(rng):
    kind = rng.choice(["attn"] * 6 + ["steps", "paged", "prefill", "prefill", "codec", "wire", "engine"])
    Hq, Hkv = rng.choice(_HEADS[:2] * 3 + _HEADS)
    D = rng.choice([128, 128, 128, 128, 64, 256])
    if kind == "attn":
        T = _spread(rng, 33, 32768)
        most = 128 * 4339 * 8 * 128 // (T * Hkv * D)          # no more than the serving batch reads
        B = _spread(rng, 1, max(1, min(128, most)))
        window = rng.choice([0, 0, 0, 0, _spread(rng, 256, 4096)])
        cache = rng.choice(["compressed"] * 4 + ["bf16"])
        return dict(kind=kind, cache=cache, B=B, T=T, Hq=Hq, Hkv=Hkv, D=D, window=window if window < T else 0)
    if kind in ("steps", "paged"):
        top = 8 if kind == "steps" else 12
        return dict(kind=kind, B=rng.randint(1, top), T=_spread(rng, 20, 500 if kind == "steps" else 1500),
                    N=rng.randint(3, 40 if kind == "steps" else 24), Hq=Hq, Hkv=min(Hkv, 8), D=min(D, 128)) | (
                        {"Hq": 32} if Hkv > 8 else {})
    if kind == "prefill":
        return dict(kind=kind, T=_spread(rng, 17, 16384), Hkv=min(Hkv, 8), D=D)
    if kind == "codec":
        B = rng.randint(1, 16)
        return dict(kind=kind, B=B, T=PAGE * _spread(rng, 1, 256), Hkv=min(Hkv, 8), D=min(D, 128))
    if kind == "wire":
        return dict(kind=kind, B=rng.randint(1, 8), T=_spread(rng, 20, 4101), Hkv=min(Hkv, 8), D=128)
    return dict(kind=kind, B=rng.randint(1, 4), T=_spread(rng, 20, 300), N=rng.randint(3, 40), Hq=16, Hkv=4, D=128,
                hidden=2048)


# ---------------------------------------------------------------- inputs

def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _rotate(x, pos, theta):
    """Rotary embedding (half-split) of x [n, H, D] in fp32 at positions pos [n]."""
    half = x.shape[-1] // 2
    inv = theta ** (-torch.arange(half, device=DEV, dtype=torch.float64) / half)
    ang = pos.double()[:, None] * inv
    c, s = ang.cos().float()[:, None, :], ang.sin().float()[:, None, :]
    a, b = x[..., :half], x[..., half:]
    return torch.cat([a * c - b * s, b * c + a * s], dim=-1)


def _kv(B, T, H, D, keys, g):
    """Keys or values [B, T, H, D] bf16: the recipe of exactkv_amd.synthetic on the GPU."""
    scale = torch.exp(torch.randn(H, D, generator=g, device=DEV) * (1.5 if keys else 0.5))
    out = torch.empty(B, T, H, D, dtype=torch.bfloat16, device=DEV)
    for b in range(B):
        x = torch.randn(T, H, D, generator=g, device=DEV) * scale
        if keys:
            x = _rotate(x, torch.arange(T, device=DEV), 1e6)
        x = x.bfloat16()
        x[torch.rand(T, H, D, generator=g, device=DEV) < ZEROS] = 0
        raw = torch.rand(T, H, 1, generator=g, device=DEV) < RAW_ROWS
        at = torch.randint(0, D, (T, H, 1), generator=g, device=DEV) == torch.arange(D, device=DEV)
        out[b] = torch.where(raw & at, x * 2.0 ** -20, x)
    return out


def _inputs(c, seed):
    """(q, k, v) of an attn, steps or paged case: k, v [B, T + N, Hkv, D]; q [B, Hq, D], or one for
    each of the N steps."""
    g = _gen(seed)
    N = c.get("N", 0)
    k = _kv(c["B"], c["T"] + N, c["Hkv"], c["D"], True, g)
    v = _kv(c["B"], c["T"] + N, c["Hkv"], c["D"], False, g)
    shape = (c["B"], c["Hq"], c["D"]) if N == 0 else (N, c["B"], c["Hq"], c["D"])
    return torch.randn(shape, generator=g, device=DEV).bfloat16(), k, v


def _lengths(c):
    """Prompt lengths of a paged case: from a third of T up to T, in no order."""
    return [c["T"] - (i * 7 % c["B"]) * (c["T"] * 2 // 3) // c["B"] for i in range(c["B"])]


def _round_up(n, m):
    return -(-n // m) * m


# ---------------------------------------------------------------- a decoder with the layout of
# the Hugging Face Llama modules, which Engine drives

def apply_rotary_pos_emb(q, k, cos, sin):
    def turn(x):
        half = x.shape[-1] // 2
        return torch.cat((-x[..., half:], x[..., :half]), dim=-1)
    cos, sin = cos.unsqueeze(1), sin.unsqueeze(1)
    return q * cos + turn(q) * sin, k * cos + turn(k) * sin


class _Config:
    model_type = "llama"

    def __init__(self, c, layers=2, vocab=4096):
        self.num_hidden_layers, self.vocab = layers, vocab
        self.hidden_size, self.inner = c["hidden"], 2 * c["hidden"]
        self.num_attention_heads, self.num_key_value_heads, self.head_dim = c["Hq"], c["Hkv"], c["D"]


class _Norm(torch.nn.Module):
    def __init__(self, n):
        super().__init__()
        self.weight = torch.nn.Parameter(torch.ones(n))

    def forward(self, x):
        y = x if x.dtype == torch.float64 else x.float()
        return self.weight * (y * torch.rsqrt(y.square().mean(-1, keepdim=True) + 1e-5)).to(x.dtype)


class _Attention(torch.nn.Module):
    def __init__(self, cfg, index):
        super().__init__()
        self.cfg, self.index = cfg, index
        n, kv = cfg.num_attention_heads * cfg.head_dim, cfg.num_key_value_heads * cfg.head_dim
        lin = torch.nn.Linear
        self.q_proj = lin(cfg.hidden_size, n, bias=False)
        self.k_proj = lin(cfg.hidden_size, kv, bias=False)
        self.v_proj = lin(cfg.hidden_size, kv, bias=False)
        self.o_proj = lin(n, cfg.hidden_size, bias=False)

    def forward(self, x, cos, sin, past):
        cfg, (B, T, _) = self.cfg, x.shape
        q = self.q_proj(x).view(B, T, cfg.num_attention_heads, cfg.head_dim).transpose(1, 2)
        k = self.k_proj(x).view(B, T, cfg.num_key_value_heads, cfg.head_dim).transpose(1, 2)
        v = self.v_proj(x).view(B, T, cfg.num_key_value_heads, cfg.head_dim).transpose(1, 2)
        q, k = apply_rotary_pos_emb(q, k, cos, sin)
        if past is not None:
            k, v = past.update(k, v, self.index)
        G = cfg.num_attention_heads // cfg.num_key_value_heads
        k, v = k.repeat_interleave(G, dim=1), v.repeat_interleave(G, dim=1)
        if x.dtype == torch.float64:
            s = torch.matmul(q, k.transpose(2, 3).contiguous()) * cfg.head_dim ** -0.5
            s = s.masked_fill(torch.ones(T, T, dtype=torch.bool, device=x.device).triu(1), -math.inf)
            o = torch.matmul(s.softmax(-1), v)
        else:
            o = F.scaled_dot_product_attention(q, k, v, is_causal=True)
        return self.o_proj(o.transpose(1, 2).reshape(B, T, -1))


class _MLP(torch.nn.Module):
    def __init__(self, cfg):
        super().__init__()
        self.gate_proj = torch.nn.Linear(cfg.hidden_size, cfg.inner, bias=False)
        self.up_proj = torch.nn.Linear(cfg.hidden_size, cfg.inner, bias=False)
        self.down_proj = torch.nn.Linear(cfg.inner, cfg.hidden_size, bias=False)

    def forward(self, x):
        return self.down_proj(F.silu(self.gate_proj(x)) * self.up_proj(x))


class _Layer(torch.nn.Module):
    def __init__(self, cfg, index):
        super().__init__()
        self.self_attn, self.mlp = _Attention(cfg, index), _MLP(cfg)
        self.input_layernorm, self.post_attention_layernorm = _Norm(cfg.hidden_size), _Norm(cfg.hidden_size)


class _Rotary(torch.nn.Module):
    def __init__(self, cfg):
        super().__init__()
        half = cfg.head_dim // 2
        self.inv = 5e5 ** (-torch.arange(half, device=DEV, dtype=torch.float64) / half)

    def forward(self, x, pos):
        ang = pos.double()[..., None] * self.inv
        ang = torch.cat((ang, ang), dim=-1)
        return ang.cos().to(x.dtype), ang.sin().to(x.dtype)


class _Output:
    def __init__(self, hidden):
        self.last_hidden_state = hidden


class _Body(torch.nn.Module):
    def __init__(self, cfg):
        super().__init__()
        self.embed_tokens = torch.nn.Embedding(cfg.vocab, cfg.hidden_size)
        self.layers = torch.nn.ModuleList([_Layer(cfg, i) for i in range(cfg.num_hidden_layers)])
        self.norm, self.rotary_emb = _Norm(cfg.hidden_size), _Rotary(cfg)

    def forward(self, ids, use_cache=True, past_key_values=None):
        h = self.embed_tokens(ids)
        cos, sin = self.rotary_emb(h, torch.arange(ids.shape[1], device=ids.device)[None])
        for layer in self.layers:
            h = h + layer.self_attn(layer.input_layernorm(h), cos, sin, past_key_values)
            h = h + layer.mlp(layer.post_attention_layernorm(h))
        return _Output(self.norm(h))


class _Decoder(torch.nn.Module):
    def __init__(self, cfg):
        super().__init__()
        self.config, self.model = cfg, _Body(cfg)
        self.lm_head = torch.nn.Linear(cfg.hidden_size, cfg.vocab, bias=False)


def _decoder(c, seed):
    """(bf16 decoder with random weights, prompt ids [B, T], next tokens [N, B])."""
    g = _gen(seed)
    cfg = _Config(c)
    with torch.device(DEV):
        m = _Decoder(cfg).bfloat16().eval().requires_grad_(False)
    for p in m.parameters():
        if p.dim() == 2:
            p.copy_(torch.randn(p.shape, generator=g, device=DEV) * (1.0 if p is m.model.embed_tokens.weight else 0.02))
    ids = torch.randint(0, cfg.vocab, (c["B"], c["T"]), generator=g, device=DEV)
    return m, ids, torch.randint(0, cfg.vocab, (c["N"], c["B"]), generator=g, device=DEV)


# ---------------------------------------------------------------- prepare and run

def prepare(case, seed):
    return _KINDS[case["kind"]][0](case, seed)


def run(state):
    return _KINDS[state["case"]["kind"]][1](state)


def _prepare_attn(c, seed):
    q, k, v = _inputs(c, seed)
    cls = exactkv.CompressedKV if c["cache"] == "compressed" else exactkv.BF16KV
    TS = _round_up(c["T"] + 1, PAGE)
    kc, vc = (cls(c["B"], TS, c["Hkv"], c["D"]) for _ in range(2))
    for b in range(c["B"]):
        kc.prefill_slot(b, k[b:b + 1])
        vc.prefill_slot(b, v[b:b + 1])
    return dict(case=c, q=q, kc=kc, vc=vc)


def _run_attn(s):
    w = s["case"]["window"]
    return exactkv.decode_attention(s["q"], s["kc"], s["vc"], **({"window": w} if w else {}))


def _cache_arrays(c):
    """A cache's arrays (raw rows as bit patterns)."""
    return dict(sm=c.sm, code=c.code, base=c.base, rowmask=c.rowmask, rowoff=c.rowoff, cnt=c.cnt,
                raw=c.raw.view(torch.int16))


def _prepare_steps(c, seed):
    q, k, v = _inputs(c, seed)
    TS = _round_up(c["T"] + c["N"] + 1, PAGE)
    kc, vc = (exactkv.CompressedKV(c["B"], TS, c["Hkv"], c["D"], reserve=POOL) for _ in range(2))
    T = c["T"]
    return dict(case=c, q=q, kc=kc, vc=vc, kp=k[:, :T].contiguous(), vp=v[:, :T].contiguous(),
                ks=k[:, T:].transpose(0, 1).contiguous(), vs=v[:, T:].transpose(0, 1).contiguous())


def _run_steps(s):
    kc, vc, c = s["kc"], s["vc"], s["case"]
    kc.cnt.zero_()                                     # a new batch: its raw rows from the pool's start
    vc.cnt.zero_()
    for b in range(c["B"]):
        kc.prefill_slot(b, s["kp"][b:b + 1])
        vc.prefill_slot(b, s["vp"][b:b + 1])
    out = []
    for n in range(c["N"]):
        kc.append(s["ks"][n])
        vc.append(s["vs"][n])
        out.append(exactkv.decode_attention(s["q"][n], kc, vc))
        if kc.T % PAGE == 0:
            exactkv.check_overflow([kc, vc])
    return dict(o=torch.stack(out), k=_cache_arrays(kc), v=_cache_arrays(vc))


def _prepare_paged(c, seed):
    q, k, v = _inputs(c, seed)
    lens, N = _lengths(c), c["N"]
    per = -(-(c["T"] + N + 1) // PAGE) + 1
    table = exactkv.PageTable(c["B"] * per, c["B"], per)
    kc, vc = (exactkv.PagedCompressedKV(table, c["Hkv"], D=c["D"], reserve=POOL) for _ in range(2))
    rows = [torch.arange(N, device=DEV) + L for L in lens]
    return dict(case=c, q=q, kc=kc, vc=vc, table=table, lens=lens,
                kp=[k[b:b + 1, :L].contiguous() for b, L in enumerate(lens)],
                vp=[v[b:b + 1, :L].contiguous() for b, L in enumerate(lens)],
                ks=torch.stack([k[b, r] for b, r in enumerate(rows)], dim=1),
                vs=torch.stack([v[b, r] for b, r in enumerate(rows)], dim=1))


def _run_paged(s):
    kc, vc, table, c = s["kc"], s["vc"], s["table"], s["case"]
    for b, L in enumerate(s["lens"]):
        slot = table.add(L)
        kc.prefill(slot, s["kp"][b])
        vc.prefill(slot, s["vp"][b])
    out = []
    for n in range(c["N"]):
        table.begin_step()
        kc.append(s["ks"][n])
        vc.append(s["vs"][n])
        out.append(exactkv.decode_attention(s["q"][n], kc, vc))
        if table.filled_in_step():
            exactkv.check_overflow([kc, vc])
    for b in range(c["B"]):
        table.release(b)
    kc.compact()                                       # no sequence left: the raw pools start anew
    vc.compact()
    return dict(o=torch.stack(out), lens=table.lens)


def _prepare_prefill(c, seed):
    g = _gen(seed)
    T, TS = c["T"], _round_up(c["T"] + 1, PAGE)
    k, v = (_kv(1, T, c["Hkv"], c["D"], keys, g).transpose(1, 2).contiguous() for keys in (True, False))
    kc, vc = (exactkv.CompressedKV(1, TS, c["Hkv"], c["D"], reserve=POOL) for _ in range(2))
    return dict(case=c, k=k, v=v, kc=kc, vc=vc)


def _run_prefill(s):
    kc, vc = s["kc"], s["vc"]
    kc.cnt.zero_()
    vc.cnt.zero_()
    kc.prefill_slot(0, s["k"].transpose(1, 2))
    vc.prefill_slot(0, s["v"].transpose(1, 2))
    return dict(k=_cache_arrays(kc), v=_cache_arrays(vc))


def _prepare_codec(c, seed):
    return dict(case=c, x=_kv(c["B"], c["T"], c["Hkv"], c["D"], True, _gen(seed)))


def _run_codec(s):
    enc = exactkv.encode_reference(s["x"])
    dec = exactkv.decode_reference(enc)
    out = {k: enc[k] for k in ("sm", "code", "base", "rowmask", "rowoff")}
    return dict(out, decoded=dec)                      # the raw rows (as many as the inputs have) are in it


def _prepare_wire(c, seed):
    B, T, H, D = c["B"], c["T"], c["Hkv"], c["D"]
    x = _kv(B, T, H, D, True, _gen(seed))
    TS = _round_up(T + 1, PAGE)
    src, dst = (exactkv.CompressedKV(B, TS, H, D, reserve=POOL) for _ in range(2))
    for b in range(B):
        src.prefill_slot(b, x[b:b + 1])
    return dict(case=c, src=src, dst=dst)


def _run_wire(s):
    src, dst, B = s["src"], s["dst"], s["case"]["B"]
    blobs = wire.pack_many(src, range(B))
    dst.cnt.zero_()
    wire.unpack_many(blobs, dst, range(B))
    return dict(sizes=[b.numel() for b in blobs], to=_cache_arrays(dst))   # the blobs' contents, unpacked


def _prepare_engine(c, seed):
    m, ids, forced = _decoder(c, seed)
    return dict(case=c, ids=ids, forced=forced, engine=exactkv.Engine(m, c["B"], c["T"] + c["N"] + 1))


def _run_engine(s):
    e = s["engine"]
    for kc, vc in e.kv:                                # a new batch on the same engine
        kc.cnt.zero_()
        vc.cnt.zero_()
    e.prefill(s["ids"])
    return torch.stack([e.step(tok) for tok in s["forced"]])


_KINDS = dict(attn=(_prepare_attn, _run_attn), steps=(_prepare_steps, _run_steps), paged=(_prepare_paged, _run_paged),
              prefill=(_prepare_prefill, _run_prefill), codec=(_prepare_codec, _run_codec),
              wire=(_prepare_wire, _run_wire), engine=(_prepare_engine, _run_engine))


# ---------------------------------------------------------------- what a pass cannot do without

def _row_bytes(D, compressed=True):
    """Bytes of one (token, KV head) row of one cache, its share of raw rows among them."""
    return 1.5 * D + D / PAGE + 0.5 + RAW_ROWS * 2 * D if compressed else 2.0 * D


def _attn_work(rows_k, B, Hq, Hkv, D, compressed=True):
    """One attention call over rows_k (token, KV head) rows of K and as many of V, q and out."""
    return 2 * rows_k * _row_bytes(D, compressed) + 4 * B * Hq * D, 4.0 * rows_k * (Hq / Hkv) * D


def work(case):
    c = case
    H, D, T = c["Hkv"], c["D"], c["T"]
    row = _row_bytes(D)
    if c["kind"] == "attn":
        span = min(T, c["window"]) if c["window"] else T
        b, f = _attn_work(c["B"] * span * H, c["B"], c["Hq"], H, D, c["cache"] == "compressed")
        return {"bytes": b, "flops": f}
    if c["kind"] in ("steps", "paged"):
        lens = [T] * c["B"] if c["kind"] == "steps" else _lengths(c)
        b = 2 * sum(lens) * H * (2 * D + row)          # the prompts of K and V read, their pages written
        f = 0.0
        for n in range(c["N"]):
            bn, fn = _attn_work((sum(lens) + (n + 1) * c["B"]) * H, c["B"], c["Hq"], H, D)
            b, f = b + bn + 2 * c["B"] * H * 4 * D, f + fn
        return {"bytes": b, "flops": f}
    if c["kind"] == "prefill":
        return {"bytes": 2 * T * H * (2 * D + row), "flops": 0}
    if c["kind"] == "codec":
        return {"bytes": c["B"] * T * H * 2 * (2 * D + row), "flops": 0}   # x read, pages written; and back
    if c["kind"] == "wire":
        return {"bytes": c["B"] * T * H * 4 * row, "flops": 0}             # read and written, twice
    cfg = _Config(c)
    per = cfg.hidden_size * D * 2 * (c["Hq"] + H) + 3 * cfg.hidden_size * cfg.inner
    weights = cfg.num_hidden_layers * per + cfg.vocab * cfg.hidden_size
    tokens = c["B"] * (T + c["N"])
    kv = sum(_attn_work(c["B"] * (T + n + 1) * H, c["B"], c["Hq"], H, D)[0] for n in range(c["N"]))
    return {"bytes": 2 * weights * (c["N"] + 1) + cfg.num_hidden_layers * kv, "flops": 2.0 * weights * tokens}


def tolerance(case):
    if case["kind"] in ("prefill", "codec", "wire"):
        return "exact"
    if case["kind"] == "engine":
        return {"rel": 2e-2}                           # bf16 rounding through two layers
    return {"rel": 1e-2}                               # bf16 outputs, softmax weights in bf16


# ---------------------------------------------------------------- the same in 64 bits

def _attention64(q, k, v, window=0):
    """q [Hq, D] over k, v [T, Hkv, D] of one sequence, in float64 -> [Hq, D]."""
    if window:
        k, v = k[-window:], v[-window:]
    Hkv, D = k.shape[1:]
    qd = q.double().view(Hkv, -1, D)
    s = torch.matmul(qd, k.double().permute(1, 2, 0).contiguous()) * D ** -0.5
    return torch.matmul(s.softmax(-1), v.double().transpose(0, 1).contiguous()).reshape(-1, D)


def exact(case, seed):
    c, none = case, dict(sm=None, code=None, base=None, rowmask=None, rowoff=None, cnt=None, raw=None)
    if c["kind"] == "attn":
        q, k, v = _inputs(c, seed)
        return torch.stack([_attention64(q[b], k[b], v[b], c["window"]) for b in range(c["B"])])
    if c["kind"] in ("steps", "paged"):
        q, k, v = _inputs(c, seed)
        lens = [c["T"]] * c["B"] if c["kind"] == "steps" else _lengths(c)
        o = torch.stack([torch.stack([_attention64(q[n, b], k[b, :L + n + 1], v[b, :L + n + 1])
                                      for b, L in enumerate(lens)]) for n in range(c["N"])])
        return dict(o=o, k=none, v=none) if c["kind"] == "steps" else dict(o=o, lens=None)
    if c["kind"] == "codec":
        x = _kv(c["B"], c["T"], c["Hkv"], c["D"], True, _gen(seed))
        return dict(sm=None, code=None, base=None, rowmask=None, rowoff=None, decoded=x.double())
    if c["kind"] == "engine":
        m, ids, forced = _decoder(c, seed)
        m = m.double()
        h = m.model(torch.cat([ids, forced.t()], dim=1)).last_hidden_state
        return m.lm_head(h[:, c["T"]:]).transpose(0, 1).contiguous()
    return None
