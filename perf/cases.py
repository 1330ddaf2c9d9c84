"""The work that users of this library have it do, as cases that can be timed and checked.

Decoders are measured by whole calls: one decoding step of every sequence (`Decoder.step`), one prompt (`Decoder.prefill`), one request
served through `Decoder.step_batch`; the calls a host program makes beside them (a linear layer, cached attention, the candidates of
the samplers) by themselves.  Weights are random block codes of realistic spread, made on the GPU; shapes are those of bench.py.
"""
import functools
import importlib
import json
import math
import os
import struct
import tempfile

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

# type -> (id in include/caihip.h, weights per block, bytes per block)
TYPES = {"F16": (1, 1, 2), "Q4_0": (2, 32, 18), "Q4_1": (3, 32, 20), "Q5_0": (6, 32, 22), "Q5_1": (7, 32, 24), "Q8_0": (8, 32, 34), "Q2_K": (10, 256, 84),
         "Q3_K": (11, 256, 110), "Q4_K": (12, 256, 144), "Q5_K": (13, 256, 176), "Q6_K": (14, 256, 210), "I8ROW": (100, 1, 1)}
CACHES = {"f32": (0, 4), "f16": (1, 2), "i8": (2, 1)}
EPS = 1e-6
SPREAD = 0.02    # standard deviation of the weights of a quantised model


@functools.lru_cache(None)
def library():
    """the package, with its GPU chosen"""
    cai = importlib.import_module("neural-api_amd.caihip")
    cai.init(0)
    return cai


def synth():
    return importlib.import_module("neural-api_amd.synth")


# ---------------------------------------------------------------- the cases
def listed():
    """Decoding one sequence and eight; prompts of a short message, a page and a mixture-of-experts model; the single calls; the layered
    bfloat16 decoder both ways."""
    qwen = dict(layers=28, width=3584, heads=28, kv_heads=4, dim=128, ffn=18944, vocab=152064, experts=0, top=0, body="Q4_K", head="Q8_0", mix=False, bias=True,
                tied=False, qk_norm=False, theta=1e6)
    smol = dict(layers=30, width=576, heads=9, kv_heads=3, dim=64, ffn=1536, vocab=49152, experts=0, top=0, body="Q8_0", head="Q8_0", mix=False, bias=False,
                tied=True, qk_norm=False, theta=1e5)
    olmoe = dict(layers=16, width=2048, heads=16, kv_heads=16, dim=128, ffn=1024, vocab=50304, experts=64, top=8, body="Q8_0", head="Q8_0", mix=False, bias=False,
                 tied=False, qk_norm=True, theta=1e4)
    samanex = dict(width=2048, ffn=5632, heads=16, kv_heads=8, dim=128, layers=4, vocab=32768, window=1024)
    return [
        # a small assistant on the desk: the smallest model, one token at a time, where launches are the cost
        dict(smol, name="decode_135m_q8_0", kind="decode", cache="f32", batch=1, context=100),
        # the headline: single-user chat on a 7B model, a page of context behind it
        dict(qwen, name="decode_7b_q4_k", kind="decode", cache="f32", batch=1, context=600),
        # eight users of the same model in the common mixed file (Q6_K beside Q4_K), half-precision cache
        dict(qwen, name="decode_7b_q4_k_m_b8", kind="decode", cache="f16", batch=8, context=200, mix=True, head="Q6_K"),
        # a mixture of experts, one user
        dict(olmoe, name="decode_olmoe_q8_0", kind="decode", cache="f32", batch=1, context=256),
        # a one-line message to the small model
        dict(smol, name="prompt_135m_q8_0_37", kind="prompt", cache="f32", tokens=37),
        # a page read by the 7B model
        dict(qwen, name="prompt_7b_q4_k_511", kind="prompt", cache="f32", tokens=511),
        # half a page read by the mixture of experts
        dict(olmoe, name="prompt_olmoe_q8_0_255", kind="prompt", cache="f32", tokens=255),
        # one linear layer of a host program's own net (the offload boundary), in one of the stored-stream types
        dict(name="linear_q3_k_18944x3584", kind="linear", type="Q3_K", rows=18944, cols=3584, tokens=1, bias=False, act=0),
        # one layer's attention behind a long document, int8 cache
        dict(name="attention_i8_8191", kind="attention", heads=40, kv_heads=8, dim=128, cache="i8", rows=8191, window=0),
        # what a sampled (not greedy) reply asks for after every token
        dict(name="candidates_152064", kind="candidates", vocab=152064, history=512, top=40, temperature=0.8, repetition=1.1, frequency=0.1, presence=0.1),
        # four pages read by the layered decoder
        dict(samanex, name="prompt_samanex_2048", kind="layered", batch=1, tokens=2048, steps=0),
        # four requests of different length served together by the layered decoder: their prompts, then a token of each at a time
        dict(samanex, name="serve_samanex_b4", kind="layered", batch=4, tokens=48, steps=16),
    ]


def log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["decode"] * 4 + ["prompt"] * 4 + ["linear"] * 3 + ["attention", "candidates", "layered", "layered"])
    if kind == "linear":
        t = rng.choice(sorted(TYPES))
        unit = 256 if TYPES[t][1] == 256 else 32
        tokens = rng.choice([1, 1, rng.randint(2, 8), log_int(rng, 9, 2048)])
        rows, cols = log_int(rng, 1000, 40000), unit * log_int(rng, 512 // unit, 18944 // unit)
        most = 3e11 if t in ("Q8_0", "Q4_0", "Q4_K", "Q5_K", "Q6_K") else 2e10
        while rows * cols * tokens > most and tokens > 8:
            tokens = max(8, tokens // 2)
        return dict(kind=kind, type=t, rows=rows, cols=cols, tokens=tokens, bias=rng.random() < 0.5, act=0 if tokens > 8 else rng.choice([0, 0, 1, 2, 3]))
    if kind == "attention":
        kv_heads = rng.choice([1, 2, 4, 8])
        return dict(kind=kind, heads=kv_heads * rng.choice([1, 2, 3, 5, 7, 8]), kv_heads=kv_heads, dim=rng.choice([64, 128]), cache=rng.choice(sorted(CACHES)), rows=log_int(rng, 16, 20000),
                    window=rng.choice([0, 0, 0, 500]))
    if kind == "candidates":
        return dict(kind=kind, vocab=log_int(rng, 1000, 200000), history=log_int(rng, 1, 3000), top=log_int(rng, 1, 1000), temperature=rng.choice([1.0, 0.7, 1.3]),
                    repetition=rng.choice([1.0, 1.1]), frequency=rng.choice([0.0, 0.2]), presence=rng.choice([0.0, 0.1]))
    if kind == "layered":
        pairs = rng.randint(2, 8)
        few = rng.random() < 0.5 and pairs != 7    # (the attention keeps half of them, which has to divide the heads)
        c = dict(kind=kind, width=256 * pairs, ffn=64 * log_int(rng, 16, 100), heads=2 * pairs, kv_heads=pairs if few else 2 * pairs, dim=128, layers=4, vocab=log_int(rng, 2000, 32768), window=rng.choice([64, 300, 1024]))
        return dict(c, batch=1, tokens=log_int(rng, 2, 2048), steps=0) if rng.random() < 0.5 else dict(c, batch=rng.randint(1, 8), tokens=log_int(rng, 4, 100), steps=rng.randint(4, 16))
    body = rng.choice(["Q4_K", "Q4_K", "Q8_0", "Q8_0", "Q6_K", "Q5_K", "Q4_0", "Q2_K", "Q3_K", "Q4_1", "Q5_0", "Q5_1"])
    unit = TYPES[body][1]
    dim, kv_heads = rng.choice([64, 128, 128]), rng.choice([1, 2, 4, 8])
    if unit * 1.0 > dim * kv_heads:
        kv_heads = unit // dim    # (whole blocks in a row of the output projection)
    heads = kv_heads * rng.choice([1, 2, 3, 4])
    experts = rng.choice([0, 0, 0, 8, 32]) if body in ("Q8_0", "Q4_0") else 0
    width = max(unit, 64) * log_int(rng, 512 // max(unit, 64), 4096 // max(unit, 64))
    ffn = unit * (log_int(rng, 1024 // unit, 14336 // unit) if not experts else log_int(rng, 512 // unit, 2048 // unit))
    c = dict(kind=kind, layers=rng.randint(2, 8), width=width, heads=heads, kv_heads=kv_heads, dim=dim, ffn=ffn, vocab=log_int(rng, 2000, 100000), experts=experts,
             top=rng.choice([1, 2, 4]) if experts else 0, body=body, head="Q6_K" if width % 256 == 0 and rng.random() < 0.5 else "Q8_0", mix=body == "Q4_K" and rng.random() < 0.5,
             bias=rng.random() < 0.5, tied=False, qk_norm=bool(experts) and rng.random() < 0.5, theta=1e5, cache=rng.choice(sorted(CACHES)))
    if kind == "decode":
        return dict(c, batch=rng.choice([1, 1, rng.randint(2, 8)]), context=log_int(rng, 2, 1500))
    c["tokens"] = log_int(rng, 2, 2048)
    most = 6e10 if body in ("Q2_K", "Q3_K", "Q4_1", "Q5_0", "Q5_1") else 4e12
    while work(c)["flops"] > most and c["tokens"] > 16:
        c["tokens"] //= 2
    return c


# ---------------------------------------------------------------- weights
def generator(*numbers):
    g = torch.Generator(device="cuda")
    g.manual_seed(hash(tuple(numbers)) % (1 << 62))
    return g


def halves(x):
    return x.to(torch.float16).contiguous().view(torch.uint8).view(*x.shape, 2)


def k_scales(sc, mn):
    """the 12 bytes of eight 6-bit scales and eight 6-bit minima"""
    return torch.cat([(sc[..., :4] & 63) | ((sc[..., 4:] >> 4) << 6), (mn[..., :4] & 63) | ((mn[..., 4:] >> 4) << 6), (sc[..., 4:] & 15) | ((mn[..., 4:] & 15) << 4)], -1)


def blocks(kind, rows, cols, gen):
    """Random blocks in the stored form, uint8 [rows, bytes]: codes of a normal distribution cut at three deviations, scales that differ by
    a third from block to block."""
    _, be, bb = TYPES[kind]
    n = rows * cols // be

    def codes(levels, *shape):
        q = torch.randn(*shape, device="cuda", generator=gen).mul_(levels / 6.0).add_(levels / 2.0)
        return q.round_().clamp_(0, levels - 1).to(torch.uint8)

    def around(x, *shape):
        return x * (1.0 + 0.3 * (2.0 * torch.rand(*shape, device="cuda", generator=gen) - 1.0))

    if kind == "F16":
        return halves(torch.randn(rows, cols, device="cuda", generator=gen) * SPREAD).view(rows, -1)
    if kind in ("Q8_0", "I8ROW"):
        q = (torch.randn(n, be, device="cuda", generator=gen) * 42.0).round_().clamp_(-127, 127).to(torch.int8).view(torch.uint8)
        return q.view(rows, cols) if kind == "I8ROW" else torch.cat([halves(around(SPREAD / 42.0, n)), q], 1).view(rows, -1)
    if be == 32:
        levels = 16 if kind[1] == "4" else 32
        q, unit = codes(levels, n, 32), SPREAD * 6.0 / levels
        d = around(unit, n)
        parts = [halves(d)] + ([halves(-d * levels / 2.0)] if kind[-1] == "1" else [])
        if levels == 32:
            parts.append(((q >> 4).to(torch.int64) << torch.arange(32, device="cuda")).sum(1).to(torch.int32).view(n, 1).view(torch.uint8))
        return torch.cat(parts + [(q[:, :16] & 15) | ((q[:, 16:] & 15) << 4)], 1).view(rows, -1)
    if kind in ("Q4_K", "Q5_K"):
        levels = 16 if kind == "Q4_K" else 32
        q = codes(levels, n, 8, 32)
        sc = torch.randint(24, 64, (n, 8), device="cuda", generator=gen, dtype=torch.uint8)
        d = around(SPREAD * 6.0 / levels / 44.0, n)
        parts = [halves(d), halves(d * levels / 2.0), k_scales(sc, sc)]
        if levels == 32:
            parts.append(sum((q[:, j] >> 4) << j for j in range(8)))
        ql = (q & 15).view(n, 4, 2, 32)
        return torch.cat(parts + [(ql[:, :, 0] | (ql[:, :, 1] << 4)).view(n, 128)], 1).view(rows, -1)
    if kind == "Q6_K":
        q = codes(64, n, 2, 4, 32)
        sc = torch.randint(50, 128, (n, 16), device="cuda", generator=gen, dtype=torch.uint8)
        lo, hi = q & 15, q >> 4
        ql = torch.stack([lo[:, :, 0] | (lo[:, :, 2] << 4), lo[:, :, 1] | (lo[:, :, 3] << 4)], 2).view(n, 128)
        qh = (hi[:, :, 0] | (hi[:, :, 1] << 2) | (hi[:, :, 2] << 4) | (hi[:, :, 3] << 6)).view(n, 64)
        return torch.cat([ql, qh, sc, halves(around(SPREAD * 6.0 / 64 / 88.0, n))], 1).view(rows, -1)
    if kind == "Q2_K":
        q = codes(4, n, 2, 4, 32)
        sc = torch.randint(5, 16, (n, 16), device="cuda", generator=gen, dtype=torch.uint8)
        d = around(SPREAD / 10.0, n)
        qs = (q[:, :, 0] | (q[:, :, 1] << 2) | (q[:, :, 2] << 4) | (q[:, :, 3] << 6)).view(n, 64)
        return torch.cat([sc | (sc << 4), qs, halves(d), halves(d * 1.9)], 1).view(rows, -1)
    q = codes(8, n, 256)
    low = (q & 3).view(n, 2, 4, 32)
    qs = (low[:, :, 0] | (low[:, :, 1] << 2) | (low[:, :, 2] << 4) | (low[:, :, 3] << 6)).view(n, 64)
    mask = sum((q.view(n, 8, 32)[:, j] >> 2) << j for j in range(8))
    sc = torch.randint(44, 64, (n, 16), device="cuda", generator=gen, dtype=torch.uint8)    # 6 bits standing for sc - 32
    packed = torch.cat([(sc[:, :8] & 15) | ((sc[:, 8:] & 15) << 4), (sc[:, 0:4] >> 4) | ((sc[:, 4:8] >> 4) << 2) | ((sc[:, 8:12] >> 4) << 4) | ((sc[:, 12:] >> 4) << 6)], 1)
    return torch.cat([mask, qs, packed, halves(around(SPREAD * 6.0 / 8 / 21.0, n))], 1).view(rows, -1)


def half_at(b, at):
    return b[:, at:at + 2].contiguous().view(torch.float16).to(torch.float64)


def dequantised(kind, raw, cols, scales=None):
    """the same weights in 64 bits, [rows, cols]"""
    _, be, bb = TYPES[kind]
    f = torch.float64
    if kind == "F16":
        return raw.view(torch.float16).to(f)
    if kind == "I8ROW":
        return raw.view(torch.int8).to(f) * scales.to(f)[:, None]
    b = raw.view(-1, bb)
    n = b.shape[0]
    nib = lambda z: torch.cat([z & 15, z >> 4], 1)
    if kind == "Q8_0":
        w = half_at(b, 0) * b[:, 2:].view(torch.int8).to(f)
    elif kind == "Q4_0":
        w = half_at(b, 0) * (nib(b[:, 2:]).to(f) - 8.0)
    elif kind == "Q4_1":
        w = half_at(b, 0) * nib(b[:, 4:]).to(f) + half_at(b, 2)
    elif kind in ("Q5_0", "Q5_1"):
        at = 2 if kind == "Q5_0" else 4
        bit = (b[:, at:at + 4, None] >> torch.arange(8, device=b.device, dtype=torch.uint8)) & 1
        q = (nib(b[:, at + 4:]) | (bit.view(n, 32) << 4)).to(f)
        w = half_at(b, 0) * (q - 16.0) if kind == "Q5_0" else half_at(b, 0) * q + half_at(b, 2)
    elif kind in ("Q4_K", "Q5_K"):
        s = b[:, 4:16]
        sc = torch.cat([s[:, :4] & 63, (s[:, 8:] & 15) | ((s[:, :4] >> 6) << 4)], 1).to(f)
        mn = torch.cat([s[:, 4:8] & 63, (s[:, 8:] >> 4) | ((s[:, 4:8] >> 6) << 4)], 1).to(f)
        z = b[:, -128:].view(n, 4, 32)
        q = torch.stack([z & 15, z >> 4], 2).view(n, 8, 32)
        if kind == "Q5_K":
            q = q | (((b[:, None, 16:48] >> torch.arange(8, device=b.device, dtype=torch.uint8)[None, :, None]) & 1) << 4)
        w = (half_at(b, 0) * sc)[:, :, None] * q.to(f) - (half_at(b, 2) * mn)[:, :, None]
    elif kind == "Q6_K":
        lo, hi = b[:, :128].view(n, 2, 2, 32), b[:, 128:192].view(n, 2, 1, 32)
        q = torch.cat([lo & 15, lo >> 4], 2) | (((hi >> torch.tensor([0, 2, 4, 6], device=b.device, dtype=torch.uint8)[None, None, :, None]) & 3) << 4)
        w = (half_at(b, 208) * b[:, 192:208].view(torch.int8).to(f))[:, :, None] * (q.reshape(n, 16, 16).to(f) - 32.0)
    else:
        shifts = torch.tensor([0, 2, 4, 6], device=b.device, dtype=torch.uint8)[None, None, :, None]
        if kind == "Q2_K":
            q = ((b[:, 16:80].view(n, 2, 1, 32) >> shifts) & 3).reshape(n, 16, 16).to(f)
            w = (half_at(b, 80) * (b[:, :16] & 15).to(f))[:, :, None] * q - (half_at(b, 82) * (b[:, :16] >> 4).to(f))[:, :, None]
        else:
            q = ((b[:, 32:96].view(n, 2, 1, 32) >> shifts) & 3).reshape(n, 256).to(f)
            high = ((b[:, None, :32] >> torch.arange(8, device=b.device, dtype=torch.uint8)[None, :, None]) & 1).reshape(n, 256).to(f)
            s = b[:, 96:108]
            top = (s[:, None, 8:] >> shifts[:, :, :, 0].reshape(1, 4, 1)) & 3
            sc = (torch.cat([s[:, :8] & 15, s[:, :8] >> 4], 1) | (top.reshape(n, 16) << 4)).to(f) - 32.0
            w = (half_at(b, 108) * sc)[:, :, None] * (q + 4.0 * high - 4.0).view(n, 16, 16)
    return w.reshape(-1, cols)


# ---------------------------------------------------------------- decoders of quantised files
def more_bits(i, n):
    """the blocks whose value and down projections a mixed file keeps in Q6_K"""
    return i < n // 8 or i >= 7 * n // 8 or (i - n // 8) % 3 == 2


def tensors(case, seed):
    """(layer, slot, type, rows, cols, blocks, bias) of every matrix, in a fixed order"""
    c, n = case, 0

    def one(layer, slot, kind, rows, cols, bias=False):
        nonlocal n
        n += 1
        g = generator(seed, n)
        raw = blocks(kind, rows, cols, g)
        return layer, slot, kind, rows, cols, raw, torch.randn(rows, device="cuda", generator=g) * 0.1 if bias else None

    d, qw, kw, ffn = c["width"], c["heads"] * c["dim"], c["kv_heads"] * c["dim"], c["ffn"]
    yield one(-1, 0, c["head"], c["vocab"], d)
    if not c["tied"]:
        yield one(-1, 1, c["head"], c["vocab"], d)
    for i in range(c["layers"]):
        high = "Q6_K" if c["mix"] and more_bits(i, c["layers"]) else c["body"]
        yield one(i, 2, c["body"], qw, d, c["bias"])
        yield one(i, 3, c["body"], kw, d, c["bias"])
        yield one(i, 4, high, kw, d, c["bias"])
        yield one(i, 5, c["body"], d, qw)
        many = max(1, c["experts"])
        if c["experts"]:
            yield one(i, 8, c["body"], c["experts"], d)
        yield one(i, 6, c["body"], many * 2 * ffn, d)
        yield one(i, 7, c["body"] if c["experts"] else high, many * d, ffn)


def gains(case, seed):
    """(layer, slot) -> norm gain"""
    g = np.random.default_rng([seed, 1])
    near = lambda n: (1.0 + 0.1 * g.standard_normal(n)).astype(np.float32)
    out = {(-1, 2): near(case["width"])}
    for i in range(case["layers"]):
        out[(i, 0)], out[(i, 1)] = near(case["width"]), near(case["width"])
        if case["qk_norm"]:
            out[(i, 3)], out[(i, 4)] = near(case["heads"] * case["dim"]), near(case["kv_heads"] * case["dim"])
    return out


def texts(case, seed):
    """token ids of every sequence: for a decoding step the cached context (a little shorter from sequence to sequence) and the new token"""
    g = np.random.default_rng([seed, 2])
    if case["kind"] == "prompt":
        return [g.integers(0, case["vocab"], case["tokens"]).astype(np.int32)]
    return [g.integers(0, case["vocab"], max(1, case["context"] - 3 * b) + 1).astype(np.int32) for b in range(case["batch"])]


def prepare_decoder(case, seed):
    cai = library()
    spec = {"tensors": {}, "vecs": gains(case, seed)}
    seqs = texts(case, seed)
    longest = max(len(s) for s in seqs)
    spec["cfg"] = dict(n_layers=case["layers"], d_model=case["width"], n_q_heads=case["heads"], n_kv_heads=case["kv_heads"], head_dim=case["dim"], ffn=case["ffn"], vocab=case["vocab"],
                       max_ctx=-(-(longest + 1) // 256) * 256, eps=EPS, rope_theta=case["theta"], qk_norm_full=int(case["qk_norm"]), n_experts=case["experts"], top_k=case["top"], norm_topk=0)
    for layer, slot, kind, rows, cols, raw, bias in tensors(case, seed):
        bias = None if bias is None else bias.cpu().numpy()
        torch.cuda.synchronize()
        spec["tensors"][(layer, slot)] = dict(qw=cai.QWeight(TYPES[kind][0], rows, cols, raw.data_ptr(), bias))
        del raw
    dec = cai.Decoder(spec, max_batch=len(seqs), kv_dtype=CACHES[case["cache"]][0])
    state = dict(case=case, dec=dec)
    if case["kind"] == "prompt":
        return dict(state, tokens=seqs[0])
    for b, s in enumerate(seqs):
        dec.prefill(s[:-1], 0, b, want_logits=False)
    return dict(state, tokens=np.array([s[-1] for s in seqs], np.int32), places=np.array([len(s) - 1 for s in seqs], np.int32))


def rms(x, gain):
    return x / (x.square().mean(-1, keepdim=True) + float(np.float32(EPS))).sqrt() * torch.as_tensor(gain, device=x.device).to(x.dtype)


def stored(x, cache):
    """rows of keys or values as the cache keeps them"""
    if cache == "f16":
        return x.to(torch.float16).to(x.dtype)
    if cache == "i8":
        s = x.abs().amax(-1, keepdim=True) / 127.0
        return torch.where(s > 0, (x / s).round() * s, x)
    return x


def exact_decoder(case, seed):
    """the same logits in 64 bits: all sequences through the layers together, whole score matrices"""
    f, seqs, g = torch.float64, texts(case, seed), gains(case, seed)
    ids = torch.from_numpy(np.concatenate(seqs)).long().cuda()
    pos = torch.cat([torch.arange(len(s), device="cuda") for s in seqs]).to(f)
    ends = np.cumsum([len(s) for s in seqs])
    h, kvh, dim, ffn, d = case["heads"], case["kv_heads"], case["dim"], case["ffn"], case["width"]
    angle = pos[:, None] * float(np.float32(case["theta"])) ** (-2.0 * torch.arange(dim // 2, device="cuda", dtype=f) / dim)
    cos, sin = angle.cos()[:, None], angle.sin()[:, None]

    def turned(x):
        a, b = x[..., 0::2], x[..., 1::2]
        return torch.stack([cos * a - sin * b, sin * a + cos * b], -1).flatten(-2)

    def times(t, x):
        _, _, kind, _, cols, raw, bias = t
        y = x @ dequantised(kind, raw, cols).T
        return y if bias is None else y + bias.to(f)

    def silu_pair(y):
        return y[:, :ffn] * torch.nn.functional.silu(y[:, ffn:])

    stream = tensors(case, seed)
    embed = next(stream)
    head = embed if case["tied"] else next(stream)
    x = dequantised(embed[2], embed[5][ids].contiguous(), d)
    for i in range(case["layers"]):
        u = rms(x, g[(i, 0)])
        q, k, v = (times(next(stream), u) for _ in range(3))
        if case["qk_norm"]:
            q, k = rms(q, g[(i, 3)]), rms(k, g[(i, 4)])
        q, k, v = turned(q.view(-1, h, dim)), stored(turned(k.view(-1, kvh, dim)), case["cache"]), stored(v.view(-1, kvh, dim), case["cache"])
        out = []
        for lo, hi in zip([0, *ends[:-1]], ends):
            seen = torch.ones(hi - lo, hi - lo, device="cuda", dtype=torch.bool).tril()
            for j in range(h):
                s = q[lo:hi, j] @ k[lo:hi, j * kvh // h].T / math.sqrt(dim)
                out.append(s.masked_fill(~seen, -math.inf).softmax(-1) @ v[lo:hi, j * kvh // h])
        out = torch.cat([torch.stack(out[b * h:(b + 1) * h], 1) for b in range(len(seqs))]).flatten(1)
        x = x + times(next(stream), out)
        u = rms(x, g[(i, 1)])
        if not case["experts"]:
            mid = silu_pair(times(next(stream), u))
            x = x + times(next(stream), mid)
            continue
        weight, chosen = times(next(stream), u).softmax(-1).topk(case["top"], -1)
        up, down = (next(stream) for _ in range(2))
        for e in range(case["experts"]):
            row, rank = (chosen == e).nonzero(as_tuple=True)
            if len(row):
                a = silu_pair(u[row] @ dequantised(up[2], up[5][e * 2 * ffn:(e + 1) * 2 * ffn], d).T)
                x.index_add_(0, row, weight[row, rank][:, None] * (a @ dequantised(down[2], down[5][e * d:(e + 1) * d], ffn).T))
    y = rms(x[torch.as_tensor(ends - 1, device="cuda")], g[(-1, 2)])
    return times(head, y)


# ---------------------------------------------------------------- the layered decoder
def layered_config(case):
    return synth().layered_config(width=case["width"], ff=case["ffn"], heads=case["heads"], kv_heads=case["kv_heads"], dim=case["dim"], n_layers=case["layers"], vocab=case["vocab"], window=case["window"])


def layered_weights(case, seed):
    """name -> bfloat16 tensor"""
    out = {}
    for n, (name, (shape, std, mean)) in enumerate(synth().layered_shapes(layered_config(case)).items()):
        out[name] = (torch.randn(shape, device="cuda", generator=generator(seed, 1000 + n)) * std + mean).to(torch.bfloat16)
    return out


def layered_texts(case, seed):
    """(the prompts, the tokens fed afterwards [steps][batch])"""
    g = np.random.default_rng([seed, 3])
    prompts = [g.integers(0, case["vocab"], max(1, case["tokens"] - 5 * b)).astype(np.int32) for b in range(case["batch"])]
    return prompts, g.integers(0, case["vocab"], (case["steps"], case["batch"])).astype(np.int32)


def prepare_layered(case, seed):
    cai = library()
    weights, head, at = layered_weights(case, seed), {}, 0
    for name, w in weights.items():
        head[name] = dict(dtype="BF16", shape=list(w.shape), data_offsets=[at, at + 2 * w.numel()])
        at += 2 * w.numel()
    text = json.dumps(head).encode()
    text += b" " * (-len(text) % 8)
    with tempfile.TemporaryDirectory() as folder:
        with open(os.path.join(folder, "config.json"), "w") as f:
            json.dump(layered_config(case), f)
        with open(os.path.join(folder, "model.safetensors"), "wb") as f:
            f.write(struct.pack("<Q", len(text)) + text)
            for w in weights.values():
                f.write(w.reshape(-1).view(torch.uint8).cpu().numpy())
        dec = cai.Decoder.load(folder, case["batch"] * (-(-(case["tokens"] + case["steps"]) // 64) + 1) * 64, case["batch"], cai.DTYPE_BF16)
    prompts, later = layered_texts(case, seed)
    return dict(case=case, dec=dec, prompts=prompts, later=later)


def run_layered(state):
    """reset, the prompts as one engine step, then a step per token; the logits of every sequence's newest token each time (their arg-max is
    left out: sixteen-bit activations decide ties of a random model differently in every correct implementation)"""
    dec, out = state["dec"], []
    for b in range(len(state["prompts"])):
        dec.reset(b)
    out.append(dec.step_batch([(b, p, [len(p) - 1]) for b, p in enumerate(state["prompts"])])[1])
    for tokens in state["later"]:
        out.append(dec.step_batch([(b, tokens[b:b + 1], [0]) for b in range(len(tokens))])[1])
    return out


def exact_layered(case, seed):
    f = torch.float64
    cfg = layered_config(case)
    w = {n: t.to(f) for n, t in layered_weights(case, seed).items()}
    eps = cfg["norm"]["eps"]
    silu, sigmoid = torch.nn.functional.silu, torch.sigmoid

    def squashed(name, x):
        return torch.tanh(w[name + ".alpha"] * x) * w[name] + w[name + ".b"]

    def normed(x):
        return x / (x.square().mean(-1, keepdim=True) + eps).sqrt()

    def unit(x):
        return x / (x.square().sum(-1, keepdim=True) + 1e-6).sqrt()

    def conv(x, taps):
        n = taps.shape[1]
        padded = torch.cat([x.new_zeros(n - 1, x.shape[1]), x])
        return sum(padded[k:k + x.shape[0]] * taps[:, k] for k in range(n))

    def delta(p, c, u, per_channel):
        t, h, g, d, dv = u.shape[0], c["heads"], c["kv_heads"], c["dim"], c["vdim"]
        q, k, v = (silu(conv(u @ w[p + n].T, w[p + n + ".conv"])) for n in "qkv")
        q, k = (unit(z.view(t, g, d)).repeat_interleave(h // g, 1) for z in (q, k))
        q, v, beta, rate = q * d ** -0.5, v.view(t, h, dv), sigmoid(u @ w[p + "b"].T), w[p + "A_log"].exp()
        if per_channel:
            z = u @ w[p + "a1"].T @ w[p + "a2"].T + w[p + "dt_bias"].view(-1)
            decay = (-rate[:, None] * torch.nn.functional.softplus(z, threshold=700).view(t, h, d)).exp()
            gate = sigmoid(u @ w[p + "g1"].T @ w[p + "g2"].T)
        else:
            decay = (-rate * torch.nn.functional.softplus(u @ w[p + "a"].T + w[p + "dt_bias"], threshold=700)).exp()[:, :, None].expand(t, h, d)
            gate = silu(u @ w[p + "g"].T)
        s, out = u.new_zeros(h, d, dv), []
        for i in range(t):
            s = s * decay[i][:, :, None]
            s = s + k[i][:, :, None] * (beta[i][:, None] * (v[i] - (k[i][:, None] @ s)[:, 0]))[:, None]
            out.append((q[i][:, None] @ s)[:, 0])
        o = normed(torch.stack(out)) * w[p + "norm"] * gate.view(t, h, dv)
        return o.flatten(1) @ w[p + "o"].T

    def window(p, c, u):
        t, h, g, d = u.shape[0], c["heads"], c["kv_heads"], c["dim"]
        q = normed((u @ w[p + "q"].T).view(t, h, d)) * w[p + "q.norm"]
        k = normed((u @ w[p + "k"].T).view(t, g, d)) * w[p + "k.norm"]
        v = (u @ w[p + "v"].T).view(t, g, -1)
        i = torch.arange(t, device="cuda")
        seen = (i[None] <= i[:, None]) & (i[:, None] - i[None] < c["mask"]["size"])
        o = [(q[:, j] @ k[:, j * g // h].T * c["scale"]).masked_fill(~seen, -math.inf).softmax(-1) @ v[:, j * g // h] for j in range(h)]
        return torch.cat(o, 1) @ w[p + "o"].T

    def forward(tokens):
        x = w["embed"][torch.from_numpy(tokens).long().cuda()]
        for i, layer in enumerate(cfg["layers"]):
            p, m = "l%d." % i, layer["mixer"]
            u = squashed(p + "norm1", x)
            if layer["type"] == "delta":
                y = delta(p + "mix.", m, u, False)
            else:
                y = 0.5 * (normed(window(p + "mix.left.", m["left"], u)) * w[p + "mix.left.out"] + normed(delta(p + "mix.right.", m["right"], u, True)) * w[p + "mix.right.out"])
            x = x + squashed(p + "norm1b", y)
            u = squashed(p + "norm2", x)
            x = x + squashed(p + "norm2b", ((u @ w[p + "mlp.gate"].T).relu() * (u @ w[p + "mlp.up"].T)) @ w[p + "mlp.down"].T)
        return x

    prompts, later = layered_texts(case, seed)
    rows = [forward(np.concatenate([t, later[:, b]]))[len(t) - 1:] for b, t in enumerate(prompts)]
    return [squashed("final.norm", torch.stack([r[s] for r in rows])) @ w["head"].T for s in range(1 + len(later))]


# ---------------------------------------------------------------- single calls
def linear_inputs(case, seed):
    g = generator(seed, 1)
    raw = blocks(case["type"], case["rows"], case["cols"], g)
    scales = SPREAD / 42.0 * (0.7 + 0.6 * torch.rand(case["rows"], device="cuda", generator=g)) if case["type"] == "I8ROW" else None
    bias = torch.randn(case["rows"], device="cuda", generator=g) * 0.1 if case["bias"] else None
    return raw, scales, bias, torch.randn(case["tokens"], case["cols"], device="cuda", generator=g)


def attention_inputs(case, seed):
    """keys and values of the cached rows [kv_heads, rows, dim] with the scales of an int8 cache, and the new q | k | v"""
    g = generator(seed, 1)
    shape = (case["kv_heads"], case["rows"], case["dim"])
    k, v = torch.randn(shape, device="cuda", generator=g), torch.randn(shape, device="cuda", generator=g)
    new = torch.randn((case["heads"] + 2 * case["kv_heads"]) * case["dim"], device="cuda", generator=g)
    if case["cache"] == "f16":
        return k.half(), v.half(), None, None, new
    if case["cache"] == "f32":
        return k, v, None, None, new
    ks, vs = k.abs().amax(-1) / 127.0, v.abs().amax(-1) / 127.0
    return (k / ks[..., None]).round().to(torch.int8), (v / vs[..., None]).round().to(torch.int8), ks, vs, new


def candidates_inputs(case, seed):
    g, r = generator(seed, 1), np.random.default_rng([seed, 4])
    logits = torch.randn(case["vocab"], device="cuda", generator=g) * 2.5
    ids, counts = np.unique(r.integers(0, case["vocab"], case["history"]).astype(np.int32), return_counts=True)
    return logits, ids.astype(np.int32), counts.astype(np.int32)


def prepare_single(case, seed):
    cai = library()
    state = dict(case=case, lib=cai.load(), check=cai.check)
    if case["kind"] == "linear":
        raw, scales, bias, x = linear_inputs(case, seed)
        torch.cuda.synchronize()
        w = cai.QWeight(TYPES[case["type"]][0], case["rows"], case["cols"], raw.data_ptr(), None if bias is None else bias.cpu().numpy(), None if scales is None else scales.data_ptr())
        return dict(state, w=w, x=x, y=torch.empty(case["tokens"], case["rows"], device="cuda"))
    if case["kind"] == "attention":
        k, v, ks, vs, new = attention_inputs(case, seed)
        kv = cai.KVCache(1, case["kv_heads"], case["dim"], -(-(case["rows"] + 1) // 256) * 256, CACHES[case["cache"]][0])
        kv.import_layer(0, k.cpu().numpy(), v.cpu().numpy(), None if ks is None else ks.cpu().numpy(), None if vs is None else vs.cpu().numpy())
        torch.cuda.synchronize()
        return dict(state, kv=kv, new=new, y=torch.empty(case["heads"] * case["dim"], device="cuda"))
    logits, ids, counts = candidates_inputs(case, seed)
    torch.cuda.synchronize()
    n = min(case["top"], case["vocab"])
    return dict(state, logits=logits, ids=ids, counts=counts, tokens=np.zeros(n, np.int32), probs=np.zeros(n, np.float32))


DEVICE = 3    # CAI_X_DEVICE | CAI_Y_DEVICE


def run_single(state):
    case, lib, check = state["case"], state["lib"], state["check"]
    if case["kind"] == "linear":
        x, y, h = state["x"].data_ptr(), state["y"].data_ptr(), state["w"].h
        check(lib.cai_qgemv(h, x, case["tokens"], y, case["act"], DEVICE) if case["tokens"] <= 8 else lib.cai_qgemm(h, x, case["tokens"], y, DEVICE))
        return state["y"]
    if case["kind"] == "attention":
        check(lib.cai_attn_decode(state["kv"].h, 0, state["new"].data_ptr(), case["heads"], case["window"], 0.0, state["y"].data_ptr(), DEVICE))
        state["kv"].truncate(case["rows"])
        return state["y"]
    import ctypes
    found = ctypes.c_int()
    check(lib.cai_sample_candidates(state["logits"].data_ptr(), case["vocab"], state["ids"].ctypes.data, state["counts"].ctypes.data, len(state["ids"]), case["repetition"], case["frequency"],
                                    case["presence"], case["temperature"], len(state["tokens"]), state["tokens"].ctypes.data, state["probs"].ctypes.data, ctypes.byref(found), 1))
    return state["tokens"], state["probs"]


def exact_single(case, seed):
    f = torch.float64
    if case["kind"] == "linear":
        raw, scales, bias, x = linear_inputs(case, seed)
        y = x.to(f) @ dequantised(case["type"], raw, case["cols"], scales).T
        y = y if bias is None else y + bias.to(f)
        return (lambda z: z, torch.relu, torch.sigmoid, torch.tanh)[case["act"]](y)
    if case["kind"] == "attention":
        k, v, ks, vs, new = attention_inputs(case, seed)
        h, g, dim = case["heads"], case["kv_heads"], case["dim"]
        q, nk, nv = new.to(f).split([h * dim, g * dim, g * dim])
        k, v = k.to(f), v.to(f)
        if ks is not None:
            k, v = k * ks.to(f)[..., None], v * vs.to(f)[..., None]
        k, v = torch.cat([k, stored(nk.view(g, 1, dim), case["cache"])], 1), torch.cat([v, stored(nv.view(g, 1, dim), case["cache"])], 1)
        if case["window"]:
            k, v = k[:, -case["window"]:], v[:, -case["window"]:]
        s = q.view(g, h // g, dim) @ k.transpose(1, 2) / math.sqrt(dim)
        return (s.softmax(-1) @ v).reshape(-1)
    logits, ids, counts = candidates_inputs(case, seed)
    p = logits.to(f).softmax(-1)
    at, times = torch.from_numpy(ids).long().cuda(), torch.from_numpy(counts).cuda().to(f)
    p[at] = p[at] ** float(np.float32(case["repetition"])) * (-(float(np.float32(case["frequency"])) * times + float(np.float32(case["presence"])))).exp()
    p = p / p.sum()
    p = p ** (1.0 / float(np.float32(case["temperature"])))
    best, token = (p / p.sum()).sort(descending=True, stable=True)
    n = min(case["top"], case["vocab"])
    return token[:n].to(torch.int32), best[:n]


# ---------------------------------------------------------------- what a measurement asks for
def prepare(case, seed):
    if case["kind"] in ("decode", "prompt"):
        return prepare_decoder(case, seed)
    return prepare_layered(case, seed) if case["kind"] == "layered" else prepare_single(case, seed)


def run(state):
    case = state["case"]
    if case["kind"] == "decode":
        dec, places = state["dec"], state["places"]
        token, logits = dec.step(state["tokens"], places)
        for b, n in enumerate(places):
            dec.truncate(int(n), b)
        return token, logits
    if case["kind"] == "prompt":
        state["dec"].reset()
        token, logits = state["dec"].prefill(state["tokens"])
        return np.array([token], np.int32), logits
    return run_layered(state) if case["kind"] == "layered" else run_single(state)


def exact(case, seed):
    if case["kind"] in ("decode", "prompt"):
        y = exact_decoder(case, seed)
        return y.argmax(-1).to(torch.int32), y if case["kind"] == "decode" else y[0]
    return exact_layered(case, seed) if case["kind"] == "layered" else exact_single(case, seed)


def decoder_parts(case):
    """(bytes of one block's attention matrices, weights in them, the same of one expert or the feed-forward, bytes of a vocabulary row)"""
    kind, be, bb = TYPES[case["body"]]
    d, qw, kw = case["width"], case["heads"] * case["dim"], case["kv_heads"] * case["dim"]
    a, e = 2 * qw * d + 2 * kw * d + (case["experts"] or 0) * d, 3 * d * case["ffn"]
    return a * bb / be, a, e * bb / be, e, d * TYPES[case["head"]][2] / TYPES[case["head"]][1]


def work(case):
    kind = case["kind"]
    if kind == "linear":
        _, be, bb = TYPES[case["type"]]
        r, c, t = case["rows"], case["cols"], case["tokens"]
        return {"bytes": r * c * bb / be + 4 * t * (r + c), "flops": 2.0 * r * c * t}
    if kind == "attention":
        rows = min(case["rows"] + 1, case["window"] or 1 << 30)
        size = CACHES[case["cache"]][1] * case["dim"] + (4 if case["cache"] == "i8" else 0)
        return {"bytes": 2.0 * rows * case["kv_heads"] * size + 8.0 * case["heads"] * case["dim"], "flops": 4.0 * rows * case["heads"] * case["dim"]}
    if kind == "candidates":
        return {"bytes": 4.0 * case["vocab"] + 8.0 * (case["history"] + case["top"]), "flops": 8.0 * case["vocab"]}
    if kind == "layered":
        n = synth().layered_active_weights(layered_config(case))
        rows = sum(len(p) for p in layered_texts(case, 0)[0])
        fed, passes = rows + case["steps"] * case["batch"], 1 + case["steps"]
        wanted = passes * case["batch"]
        return {"bytes": passes * 2.0 * (n + case["vocab"] * case["width"]) + 4.0 * wanted * case["vocab"], "flops": 2.0 * n * fed + 2.0 * wanted * case["vocab"] * case["width"]}
    ab, a, eb, e, vb = decoder_parts(case)
    new = [1] * case["batch"] if kind == "decode" else [case["tokens"]]
    old = [max(1, case["context"] - 3 * b) for b in range(case["batch"])] if kind == "decode" else [0]
    rows = sum(new)
    experts = min(case["experts"], rows * case["top"]) if case["experts"] else 1
    cache = 2.0 * case["kv_heads"] * (CACHES[case["cache"]][1] * case["dim"] + (4 if case["cache"] == "i8" else 0))
    size = case["layers"] * (ab + experts * eb + cache * sum(o + n for o, n in zip(old, new))) + vb * (case["vocab"] + rows) + 4.0 * len(new) * case["vocab"]
    pairs = sum(n * o + n * (n + 1) / 2 for o, n in zip(old, new))
    flops = case["layers"] * (2.0 * rows * (a + max(1, case["top"]) * e) + 4.0 * pairs * case["heads"] * case["dim"]) + 2.0 * len(new) * case["vocab"] * case["width"]
    return {"bytes": size, "flops": flops}


def tolerance(case):
    """about four times the distance between the library and 64 bits over these ranges"""
    kind = case["kind"]
    if kind == "layered":
        return {"rel": 0.011, "max": 0.11}                    # bfloat16 activations through every layer: 0.0027
    if kind in ("linear", "attention"):
        return {"rel": 2e-6, "max": 4e-5}                     # 32-bit sums, activations of 22 bits and more: 4e-7
    if kind == "candidates":
        return {"rel": 2e-6, "max": 4e-5, "differ": 0.005}    # neighbours a rounding apart may trade places
    if case["cache"] == "i8":
        return {"rel": 7e-3, "max": 7e-2}                     # a cached element on the edge between two codes moves by a whole code: 0.0017
    if case["cache"] == "f16":
        return {"rel": 1.5e-3, "max": 1.5e-2}                 # the same with half-precision rows: 0.0003
    if case["experts"]:
        return {"rel": 1e-3, "max": 1e-2}                     # two experts whose scores are a rounding apart may trade places for an earlier token
    return {"rel": 1e-4, "max": 4e-3}                         # 32-bit angles of the rotation: 2.5e-5
