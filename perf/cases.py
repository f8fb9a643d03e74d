"""The calls a server makes on the attention path, as measurable cases.

Five families, one engine step each, all through vm_c_amd.capi (the C ABI's
entry points), inputs resident in GPU memory:

  decode  one new token per sequence: append its K/V to the cache, then split
          decode attention over every sequence's whole context, with the
          workspace a server allocates once.  f16 / bf16 / q8_0 / q4_0 pages
          or TurboQuant slots; head_dim 64, 128 and 256.
  prefill the prompts of new requests: causal attention over the step's own
          K/V, which are written to the cache on the way (pages), or by the
          TurboQuant store beside it.
  chunk   chunked prefill: append this step's tokens, then attend the cached
          prefix and the tokens themselves through the block tables.
  append  Q/K RMSNorm + RoPE + quantize-on-append, in place, of one step's
          tokens.

Values are N(0, 1) before quantization, as the repository's configurations
say; block tables are permutations of a shared pool.  The pools are filled
here, in plain torch, with the codes that such values quantize to.
"""
import math

import numpy as np
import torch

from vm_c_amd import capi

BS = 16  # tokens per page
TQ = ("turboquant_3bit_nc", "turboquant_4bit_nc", "turboquant_k3v4_nc")
_DT = {"f16": torch.float16, "bf16": torch.bfloat16}


# ------------------------------------------------------------------ the cases

def listed():
    return [
        # A single user's decode over fp16 pages: the smallest call, bound by launches and latency.
        _decode("decode_f16_b1", fmt="fp16", batch=1, lo=2048, hi=2048),
        # A small server's batch over GGUF q8_0 pages, contexts of 512 to 4096 tokens.
        _decode("decode_q8_0_b16", fmt="q8_0", batch=16, lo=512, hi=4096, spread="uniform", len_seed=1),
        # A full batch at one context length over 4-bit TurboQuant slots.
        _decode("decode_tq4_b32_8k", fmt="turboquant_4bit_nc", batch=32, lo=8192, hi=8192),
        # The long-context headline: ragged contexts to 32768, 3-bit slots, 64 / 8 heads.
        _decode("decode_tq3_b64_32k", fmt="turboquant_3bit_nc", batch=64, hq=64, lo=1024, hi=32768, len_seed=4),
        # The head_dim 256 deployment (16 / 2 heads, 262-byte slots), bf16 activations.
        _decode("decode_tq4_d256_b32", fmt="turboquant_4bit_nc", batch=32, hq=16, hkv=2, d=256, dtype="bf16",
                lo=4096, hi=32768, len_seed=3),
        # A small model's batch: head_dim 64, bf16 pages, short and long contexts together.
        _decode("decode_bf16_d64_b32", fmt="bf16", batch=32, d=64, dtype="bf16", lo=256, hi=8192, len_seed=5),
        # Long prompts: 4 x 4096 tokens, bf16, q8_0 pages written in the same launch.
        _prefill("prefill_bf16_4x4096", fmt="q8_0", batch=4, lo=4096, hi=4096),
        # Chat prompts: a few hundred tokens each, odd lengths, fp16 activations and pages.
        _prefill("prefill_f16_short", fmt="fp16", dtype="f16", batch=8, lo=32, hi=1024, len_seed=6),
        # Prompts of the head_dim 256 deployment: TurboQuant store and causal attention.
        _prefill("prefill_bf16_d256", fmt="turboquant_4bit_nc", batch=4, hq=16, hkv=2, d=256, lo=500, hi=4096,
                 len_seed=7),
        # Chunked prefill of a long document over q8_0 pages.
        _chunk("chunk_q8_0_2k_30k", fmt="q8_0", batch=1, new=2048, lo=30720, hi=30720),
        # The same over 3-bit TurboQuant slots.
        _chunk("chunk_tq3_2k_30k", fmt="turboquant_3bit_nc", batch=1, new=2048, lo=30720, hi=30720),
        # Norm, RoPE and append of a 16384-token prefill step.
        _append("append_q8_0_16k", fmt="q8_0", tokens=16384),
    ]


def _decode(name, *, fmt, batch, lo, hi, hq=32, hkv=8, d=128, dtype="f16", layout="nhd", spread="log", len_seed=0):
    return _named(name, kind="decode", fmt=fmt, batch=batch, hq=hq, hkv=hkv, d=d, dtype=dtype, layout=layout, lo=lo,
                  hi=hi, spread=spread, len_seed=len_seed)


def _prefill(name, *, fmt, batch, lo, hi, hq=32, hkv=8, d=128, dtype="bf16", layout="nhd", spread="log", len_seed=0):
    return _named(name, kind="prefill", fmt=fmt, batch=batch, hq=hq, hkv=hkv, d=d, dtype=dtype, layout=layout, lo=lo,
                  hi=hi, spread=spread, len_seed=len_seed)


def _chunk(name, *, fmt, batch, new, lo, hi, hq=32, hkv=8, d=128, dtype="f16", layout="nhd", spread="log",
           len_seed=0):
    return _named(name, kind="chunk", fmt=fmt, batch=batch, new=new, hq=hq, hkv=hkv, d=d, dtype=dtype, layout=layout,
                  lo=lo, hi=hi, spread=spread, len_seed=len_seed)


def _append(name, *, fmt, tokens, hq=32, hkv=8, dtype="bf16", layout="nhd", neox=True):
    return _named(name, kind="append", fmt=fmt, tokens=tokens, hq=hq, hkv=hkv, d=128, dtype=dtype, layout=layout,
                  neox=neox)


def _named(name, **case):
    return dict(case, name=name) if name else case


def draw(rng):
    """Another step of the same families.  Lengths and batches are spread over
    their logarithm; a batch whose work would pass the largest listed case's
    of its family is cut."""
    kind = rng.choice(["decode", "decode", "decode", "prefill", "prefill", "chunk", "append"])
    pages = ["fp16", "bf16", "q8_0", "q4_0"]
    layout = rng.choice(["nhd", "nhd", "hnd"])
    log = lambda a, b: int(round(math.exp(rng.uniform(math.log(a), math.log(b)))))  # noqa: E731
    len_seed = rng.randrange(1 << 20)

    def dt_of(fmt):
        return {"fp16": "f16", "bf16": "bf16"}.get(fmt) or rng.choice(["f16", "bf16"])

    if kind == "decode":
        if rng.random() < 0.5:  # TurboQuant slots
            d = rng.choice([128, 128, 256])
            heads = [(16, 2), (8, 1), (16, 4)] if d == 256 else [(32, 8), (64, 8), (32, 4), (16, 2)]
            fmt, layout = rng.choice(TQ if d == 128 else TQ[:2]), "nhd"
        else:
            d = rng.choice([64, 128, 128, 256])
            heads = {64: [(32, 8), (14, 2)], 128: [(32, 8), (64, 8), (32, 4), (16, 2)], 256: [(16, 2), (8, 4)]}[d]
            fmt = rng.choice(pages)
        hq, hkv = rng.choice(heads)
        hi = log(64, 32768)
        lo = max(1, log(max(1, hi // 16), hi))
        batch = log(1, 64)
        # no more bytes than 150k tokens of 8 heads x 128 dims x 2 bytes x 2
        batch = max(1, min(batch, int(150_000 * 1024 * 4 / (hi * hkv * d * 4))))
        return _decode("", fmt=fmt, batch=batch, lo=lo, hi=hi, hq=hq, hkv=hkv, d=d, dtype=dt_of(fmt), layout=layout,
                       len_seed=len_seed)
    if kind == "prefill":
        d = rng.choice([64, 128, 128, 256])
        hq, hkv = rng.choice({64: [(32, 8), (14, 2)], 128: [(32, 8), (64, 8), (28, 4)], 256: [(16, 2), (8, 4)]}[d])
        fmt = rng.choice(pages + ["turboquant_4bit_nc", "turboquant_3bit_nc"])
        if fmt in TQ:
            layout = "nhd"
        hi = log(16, 4096)
        lo = max(1, log(max(1, hi // 16), hi))
        batch = max(1, min(log(1, 8), 12288 // hi))
        return _prefill("", fmt=fmt, batch=batch, lo=lo, hi=hi, hq=hq, hkv=hkv, d=d, dtype=dt_of(fmt), layout=layout,
                        len_seed=len_seed)
    if kind == "chunk":
        fmt = rng.choice(pages + ["turboquant_4bit_nc", "turboquant_3bit_nc"])
        if fmt in TQ:
            layout = "nhd"
        hq, hkv = rng.choice([(32, 8), (64, 8), (28, 4)])
        hi = log(64, 30720)
        lo = max(1, log(max(1, hi // 8), hi))
        new = log(17, 2048)
        batch = max(1, min(log(1, 4), 32768 * 2048 * 32 // ((hi + new) * new * hq)))
        if hq == 64:
            new = max(17, new // 2)
        return _chunk("", fmt=fmt, batch=batch, new=new, lo=lo, hi=hi, hq=hq, hkv=hkv, dtype=dt_of(fmt),
                      layout=layout, len_seed=len_seed)
    fmt = rng.choice(pages + ["turboquant_4bit_nc", "turboquant_3bit_nc"])
    hq, hkv = rng.choice([(32, 8), (64, 8), (28, 4)])
    tokens = log(1, 16384 if hq < 64 else 8192)
    return _append("", fmt=fmt, tokens=tokens, hq=hq, hkv=hkv, dtype=dt_of(fmt),
                   layout="nhd" if fmt in TQ else layout, neox=rng.random() < 0.75)


def _lens(c):
    """The sequences' lengths: prompt lengths, contexts or cached prefixes."""
    rng = np.random.default_rng(c["len_seed"])
    if c["spread"] == "uniform":
        lens = rng.integers(c["lo"], c["hi"] + 1, c["batch"])
    else:
        lens = np.exp(rng.uniform(math.log(c["lo"]), math.log(c["hi"]), c["batch"])).astype(np.int64)
        lens[0] = c["hi"]
    return np.clip(lens, c["lo"], c["hi"]).astype(np.int64)


# ------------------------------------------------------------------ formats, in plain torch

def _entry_bytes(fmt, d):
    """Bytes of one (token, head): K or V of a page format, or a whole slot."""
    if fmt in TQ:
        kb, vb = _bits(fmt)
        return d * kb // 8 + 2 + d * vb // 8 + 4
    return {"fp16": 2 * d, "bf16": 2 * d, "q8_0": 34 * (d // 32), "q4_0": 18 * (d // 32)}[fmt]


def _bits(fmt):
    return {TQ[0]: (3, 3), TQ[1]: (4, 4), TQ[2]: (3, 4)}[fmt]


_TABLES = {}


def _centroids(d, bits):
    """Lloyd-Max levels for N(0, 1/d): trapezoid rule over cells that end at
    3 x 3.5 sigma, 200 rounds."""
    if (d, bits) not in _TABLES:
        n, s2 = 1 << bits, 1.0 / d
        hi = 3.5 * math.sqrt(s2)
        c = -hi + 2 * hi * (np.arange(n) + 0.5) / n
        w = np.ones(201)
        w[[0, -1]] = 0.5
        for _ in range(200):
            e = np.concatenate([[-3 * hi], (c[:-1] + c[1:]) / 2, [3 * hi]])
            x = e[:-1, None] + (e[1:] - e[:-1])[:, None] * np.arange(201) / 200
            p = w * np.exp(-x * x / (2 * s2))
            c = (p * x).sum(1) / p.sum(1)
        _TABLES[d, bits] = np.sort(c)
    return _TABLES[d, bits]


def _hadamard(d, dev):
    h = torch.ones(1, 1, dtype=torch.float64, device=dev)
    while h.shape[0] < d:
        h = torch.cat([torch.cat([h, h], 1), torch.cat([h, -h], 1)], 0)
    return h / math.sqrt(d)


def _b16(x, dtype):
    """16-bit values as two bytes each, in a new last dimension."""
    return x.to(_DT[dtype]).unsqueeze(-1).view(torch.uint8)


def _pack(codes, bits):
    """[.., d] codes -> bytes: two per byte, or eight per three bytes."""
    if bits == 4:
        p = codes.view(*codes.shape[:-1], -1, 2)
        return (p[..., 0] | (p[..., 1] << 4)).to(torch.uint8)
    p = codes.view(*codes.shape[:-1], -1, 8)
    w = p[..., 0].clone()
    for i in range(1, 8):
        w |= p[..., i] << (3 * i)
    return torch.stack([w & 255, (w >> 8) & 255, w >> 16], -1).to(torch.uint8).flatten(-2)


def _unpack(b, bits, d):
    b = b.to(torch.int32)
    if bits == 4:
        return torch.stack([b & 15, b >> 4], -1).flatten(-2)
    b = b.view(*b.shape[:-1], d // 8, 3)
    w = b[..., 0] | (b[..., 1] << 8) | (b[..., 2] << 16)
    return torch.stack([(w >> (3 * i)) & 7 for i in range(8)], -1).flatten(-2)


def _encode_slot(y, norm, v, fmt, dtype):
    """Rotated unit keys y, their norms and values v [.., d] -> slots."""
    d = v.shape[-1]
    kb, vb = _bits(fmt)
    c = torch.from_numpy(_centroids(d, kb)).to(y)
    codes = torch.bucketize(y, (c[1:] + c[:-1]) / 2, right=True, out_int32=True)
    lo, hi = v.amin(-1, keepdim=True), v.amax(-1, keepdim=True)
    q = (1 << vb) - 1
    scale = ((hi - lo) / q).clamp_min(1e-8)
    vc = torch.round((v - lo) / scale).clamp_(0, q).to(torch.int32)
    return torch.cat([_pack(codes, kb), _b16(norm, dtype), _pack(vc, vb), _b16(scale[..., 0], dtype),
                      _b16(lo[..., 0], dtype)], -1)


def _decode_slot(s, fmt, d, dtype):
    """Slots -> K in the rotated basis and V, in 64 bits."""
    kb, vb = _bits(fmt)
    nk, nv = d * kb // 8, d * vb // 8
    half = lambda o: s[..., o:o + 2].contiguous().view(_DT[dtype]).double()  # noqa: E731
    c = torch.from_numpy(_centroids(d, kb)).to(s.device)
    k = c[_unpack(s[..., :nk], kb, d).long()]
    k = k / k.norm(dim=-1, keepdim=True) * half(nk)
    v = _unpack(s[..., nk + 2:nk + 2 + nv], vb, d).double() * half(nk + 2 + nv) + half(nk + 4 + nv)
    return k, v


def _encode_page(x, fmt):
    """[.., d] values -> page entries."""
    if fmt in ("fp16", "bf16"):
        return _b16(x, "f16" if fmt == "fp16" else "bf16").flatten(-2)
    x = x.view(*x.shape[:-1], -1, 32)
    if fmt == "q8_0":
        s = x.abs().amax(-1, keepdim=True) / 127
        q = torch.round(x / s.clamp_min(1e-30)).to(torch.int8).view(torch.uint8)
    else:
        big = x.gather(-1, x.abs().argmax(-1, keepdim=True))
        s = big / -8
        q = (x / torch.where(s == 0, torch.ones_like(s), s) + 8.5).to(torch.int32).clamp_(0, 15)
        q = (q[..., :16] | (q[..., 16:] << 4)).to(torch.uint8)
    return torch.cat([_b16(s[..., 0], "f16"), q], -1).flatten(-2)


def _decode_page(b, fmt):
    if fmt in ("fp16", "bf16"):
        return b.contiguous().view(_DT["f16" if fmt == "fp16" else "bf16"]).double()
    b = b.view(*b.shape[:-1], -1, 34 if fmt == "q8_0" else 18)
    s = b[..., :2].contiguous().view(torch.float16).double()
    if fmt == "q8_0":
        return (b[..., 2:].contiguous().view(torch.int8).double() * s).flatten(-2)
    q = torch.cat([b[..., 2:] & 15, b[..., 2:] >> 4], -1).double() - 8
    return (q * s).flatten(-2)


# ------------------------------------------------------------------ inputs

def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _randn(g, *shape, dtype=torch.float32):
    return torch.randn(shape, generator=g, device="cuda").to(dtype)


def _pool(g, c, pages):
    """Page pools with every token's entries: (K pool, V pool), or (slots, None)."""
    n, d, fmt, e = pages * BS * c["hkv"], c["d"], c["fmt"], _entry_bytes(c["fmt"], c["d"])
    out = [torch.empty((n, e), dtype=torch.uint8, device="cuda") for _ in range(1 if fmt in TQ else 2)]
    for s in range(0, n, 1 << 19):
        m = min(1 << 19, n - s)
        if fmt in TQ:  # the rotation of a normal vector is another one
            x, v = _randn(g, m, d), _randn(g, m, d)
            norm = x.norm(dim=-1)
            out[0][s:s + m] = _encode_slot(x / norm[:, None], norm, v, fmt, c["dtype"])
        else:
            for p in out:
                p[s:s + m] = _encode_page(_randn(g, m, d), fmt)
    return out[0].view(-1), out[1].view(-1) if len(out) > 1 else None


def _table(g, lens):
    """A block table over a shuffled pool: [batch][most pages], -1 past each end."""
    n = torch.from_numpy((lens + BS - 1) // BS).cuda()
    perm = torch.randperm(int(n.sum()), generator=g, device="cuda").to(torch.int32)
    at = torch.arange(int(n.max()), device="cuda")[None, :]
    bt = torch.full((len(lens), int(n.max())), -1, dtype=torch.int32, device="cuda")
    bt[at < n[:, None]] = perm
    return bt


def _slots(bt, seq, pos):
    return (bt[seq, pos // BS].long() * BS + pos % BS).contiguous()


def _rows(lens, new):
    """(sequence, position) of each of a step's tokens: the last new[b] of lens[b]."""
    seq = np.repeat(np.arange(len(lens)), new)
    pos = np.concatenate([np.arange(n - k, n) for n, k in zip(lens, new)])
    return torch.from_numpy(seq).cuda(), torch.from_numpy(pos).cuda()


def prepare(case, seed):
    c, g = case, _gen(seed)
    dt, s = _DT[c["dtype"]], {"case": case}
    hq, hkv, d, fmt = c["hq"], c["hkv"], c["d"], c["fmt"]
    s["layout"] = capi.LAYOUT_HND if c["layout"] == "hnd" else capi.LAYOUT_NHD
    s["cfg"] = capi.tq_config(d, fmt) if fmt in TQ else None
    s["fmt"] = None if fmt in TQ else capi.KV_FORMATS[fmt]
    s["scale"] = 1.0 / math.sqrt(d)
    if c["kind"] in ("decode", "chunk"):
        lens = _lens(c)
        new = np.ones_like(lens) if c["kind"] == "decode" else np.full_like(lens, c["new"])
        lens = lens if c["kind"] == "decode" else lens + new
        s["bt"] = _table(g, lens)
        s["k_pool"], s["v_pool"] = _pool(g, c, int(((lens + BS - 1) // BS).sum()))
        s["lens"] = torch.from_numpy(lens).to(torch.int32).cuda()
        seq, pos = _rows(lens, new)
        s["slots"] = _slots(s["bt"], seq, pos)
        s["seq"], s["pos"] = seq.to(torch.int32), pos.to(torch.int32)
        t = len(pos)
    else:
        if c["kind"] == "prefill":
            lens = _lens(c)
            seq, pos = _rows(lens, lens)
        else:  # decode tokens and prompt chunks alike: every token at a position of its own
            lens = np.full(1, c["tokens"])
            seq, pos = torch.zeros(c["tokens"], dtype=torch.long, device="cuda"), \
                torch.randint(0, 8192, (c["tokens"],), generator=g, device="cuda")
        t = int(lens.sum())
        s["pos"] = pos.to(torch.int32 if c["kind"] == "prefill" else torch.int64)
        at = pos if c["kind"] == "prefill" else torch.arange(t, device="cuda")
        bt = _table(g, lens)
        s["slots"] = _slots(bt, seq, at)
        n = int(((lens + BS - 1) // BS).sum()) * BS * hkv * _entry_bytes(fmt, d)
        s["k_pool"] = torch.zeros(n, dtype=torch.uint8, device="cuda")
        s["v_pool"] = None if fmt in TQ else torch.zeros_like(s["k_pool"])
    s["q"] = _randn(g, t, hq, d, dtype=dt)
    s["k"], s["v"] = _randn(g, t, hkv, d, dtype=dt), _randn(g, t, hkv, d, dtype=dt)
    s["out"] = torch.empty_like(s["q"])
    ws = 0
    if c["kind"] == "decode":
        size = capi.turboquant_decode_workspace_size if fmt in TQ else capi.paged_decode_workspace_size
        ws = size(c["batch"], hq, hkv, d, s["bt"].shape[1], BS)
    elif c["kind"] == "prefill":
        ws = capi.flash_attention_prefill_workspace_size(t, hkv, d)
    elif c["kind"] == "append":
        s["qw"] = (1 + 0.1 * _randn(g, hq * d)).to(dt)
        s["kw"] = (1 + 0.1 * _randn(g, hkv * d)).to(dt)
        ang = torch.arange(8192, device="cuda", dtype=torch.float64)[:, None] * \
            10000.0 ** (-torch.arange(d // 2, device="cuda", dtype=torch.float64) * 2 / d)
        s["rope"] = torch.cat([ang.cos(), ang.sin()], 1).to(dt)
    s["ws"] = torch.empty(max(16, ws), dtype=torch.uint8, device="cuda")
    return s


# ------------------------------------------------------------------ one step

def run(state):
    s, c = state, state["case"]
    hkv, fmt, cfg = c["hkv"], c["fmt"], s["cfg"]
    if c["kind"] == "append":
        capi.fused_qk_norm_rope_store(s["q"], s["k"], s["v"], s["qw"], s["kw"], s["rope"], s["pos"], s["k_pool"],
                                      s["v_pool"], s["slots"], BS, eps=1e-6, is_neox=c["neox"],
                                      kv_format=s["fmt"] or 0, layout=s["layout"], tq_cfg=cfg)
        return _outputs(s, s["q"], s["k"])
    if c["kind"] == "prefill":
        pages = {}
        if fmt in TQ:
            capi.turboquant_store(s["k"], s["v"], s["k_pool"], s["slots"], BS, cfg)
        else:
            pages = dict(key_cache=s["k_pool"], value_cache=s["v_pool"], slot_mapping=s["slots"], block_size=BS,
                         kv_format=s["fmt"], layout=s["layout"])
        capi.flash_attention_prefill(s["out"], s["q"], s["k"], s["v"], s["pos"], hkv, s["scale"], workspace=s["ws"],
                                     **pages)
        return _outputs(s, s["out"])
    if fmt in TQ:
        capi.turboquant_store(s["k"], s["v"], s["k_pool"], s["slots"], BS, cfg)
    else:
        capi.reshape_and_cache(s["k"], s["v"], s["k_pool"], s["v_pool"], s["slots"], BS, kv_format=s["fmt"],
                               layout=s["layout"])
    if c["kind"] == "decode":
        if fmt in TQ:
            capi.turboquant_decode_attention(s["out"], s["q"], s["k_pool"], s["bt"], s["lens"], hkv, s["scale"], cfg,
                                             BS, workspace=s["ws"])
        else:
            capi.paged_attention_decode(s["out"], s["q"], s["k_pool"], s["v_pool"], s["bt"], s["lens"], hkv,
                                        s["scale"], block_size=BS, kv_format=s["fmt"], layout=s["layout"],
                                        workspace=s["ws"])
    elif fmt in TQ:
        capi.turboquant_prefill_attention(s["out"], s["q"], s["k_pool"], s["bt"], s["seq"], s["pos"], hkv, s["scale"],
                                          cfg, block_size=BS)
    else:
        capi.flash_attention_prefill_v2(s["out"], s["q"], s["k_pool"], s["v_pool"], s["bt"], s["seq"], s["pos"], hkv,
                                        s["scale"], block_size=BS, kv_format=s["fmt"], layout=s["layout"],
                                        seq_lens=s["lens"])
    return _outputs(s, s["out"])


def _outputs(s, *values):
    return [*values, s["k_pool"]] + ([] if s["v_pool"] is None else [s["v_pool"]])


# ------------------------------------------------------------------ what it costs, and what it should give

def work(case):
    c = case
    hq, hkv, d, e = c["hq"], c["hkv"], c["d"], _entry_bytes(c["fmt"], c["d"])
    kv = e * (1 if c["fmt"] in TQ else 2)  # cache bytes of one (token, head)
    if c["kind"] == "append":
        t = c["tokens"]
        return {"bytes": t * (4 * (hq + hkv) * d + 2 * hkv * d + hkv * kv + 2 * d + 16) + 2 * (hq + hkv) * d,
                "flops": t * (hq + hkv) * d * 8.0}
    lens = _lens(c)
    new = {"decode": np.ones_like(lens), "prefill": lens, "chunk": np.full_like(lens, c.get("new", 0))}[c["kind"]]
    total = lens + new if c["kind"] == "chunk" else lens
    t = float(new.sum())
    pairs = float((new * total - new * (new - 1) // 2).sum())  # (query, key) pairs under the causal mask
    step = t * (4 * hq * d + 4 * hkv * d + hkv * kv + 16)  # q in, out, the new K/V in and their entries out
    old = 0.0 if c["kind"] == "prefill" else float((total - new).sum()) * hkv * kv
    return {"bytes": step + old, "flops": 4.0 * hq * d * pairs}


def tolerance(case):
    # Four times what was seen against exact(): bf16 outputs 1.6e-3 to 2.3e-3, fp16 outputs over
    # TurboQuant slots 0.6e-3 to 1.2e-3 (16-bit level tables), over pages and this step's K/V
    # 0.2e-3 to 0.5e-3.  Page bytes and slots are whole numbers and stay the same.
    return {"rel": 8e-3 if case["dtype"] == "bf16" else 4e-3 if case["fmt"] in TQ else 2e-3}


def _attend(q, k, v, scale, first):
    """q [n][hq][d] at positions first .. first + n - 1, k, v [m][hkv][d], all in 64 bits."""
    n, hq, d = q.shape
    m, hkv, _ = k.shape
    out = torch.empty_like(q)
    late = torch.arange(m, device=q.device)[None, :] > first + torch.arange(n, device=q.device)[:, None]
    for h in range(hq):
        g = h // (hq // hkv)
        p = (q[:, h] @ k[:, g].t() * scale).masked_fill_(late, -math.inf).softmax(-1)
        out[:, h] = p @ v[:, g]
    return out


def exact(case, seed):
    c, s = case, prepare(case, seed)
    hq, hkv, d, fmt = c["hq"], c["hkv"], c["d"], c["fmt"]
    q, k, v = s["q"].double(), s["k"].double(), s["v"].double()
    rest = [None] * (1 if fmt in TQ else 2)
    if c["kind"] == "append":
        cs = s["rope"].double()[s["pos"]][:, None, :]
        cos, sin = cs[..., :d // 2], cs[..., d // 2:]

        def turned(x, w):
            x = x / (x.square().mean(-1, keepdim=True) + 1e-6).sqrt() * w.double().view(-1, d)
            if c["neox"]:
                a, b = x[..., :d // 2], x[..., d // 2:]
                return torch.cat([a * cos - b * sin, b * cos + a * sin], -1)
            a, b = x[..., 0::2], x[..., 1::2]
            return torch.stack([a * cos - b * sin, b * cos + a * sin], -1).flatten(-2)

        return [turned(q, s["qw"]), turned(k, s["kw"])] + rest
    out = torch.empty_like(q)
    if c["kind"] == "prefill":
        at = 0
        for n in _lens(c).tolist():
            out[at:at + n] = _attend(q[at:at + n], k[at:at + n], v[at:at + n], s["scale"], 0)
            at += n
        return [out] + rest
    # the new tokens' entries, then every sequence's pages, back to 64 bits
    e = _entry_bytes(fmt, d)
    if fmt in TQ:
        h = _hadamard(d, q.device)
        q = q @ h
        norm = k.norm(dim=-1)
        fresh = [_encode_slot((k @ h) / norm[..., None], norm, v, fmt, c["dtype"])]
    else:
        fresh = [_encode_page(k, fmt), _encode_page(v, fmt)]
    at = 0
    for b, n in enumerate(s["lens"].tolist()):
        new = 1 if c["kind"] == "decode" else c["new"]
        table = s["bt"][b, :(n + BS - 1) // BS].long()
        parts = []
        for pool, f in zip((s["k_pool"], s["v_pool"]), fresh):
            p = pool.view(-1, BS * hkv * e)[table]
            p = p.view(-1, BS, hkv, e) if c["layout"] == "nhd" else p.view(-1, hkv, BS, e).transpose(1, 2)
            p = p.reshape(-1, hkv, e)[:n]
            parts.append(torch.cat([p[:n - new], f[at:at + new]]))
        kk, vv = _decode_slot(parts[0], fmt, d, c["dtype"]) if fmt in TQ else [_decode_page(p, fmt) for p in parts]
        out[at:at + new] = _attend(q[at:at + new], kk, vv, s["scale"], n - new)
        at += new
    return [out] + rest
