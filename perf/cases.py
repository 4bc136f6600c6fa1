"""The work that a user of this library has it do, as cases that can be timed and checked.

Four kinds, each through the Python binding's public entry points (flint-mac_amd/flint_attn.py):

  decode   one token for each of n_seq sequences through one attention layer (KVLayer.decode): a
           chat reply being written, alone or batched over conversations;
  prefill  T prompt tokens through one attention layer at position p0 (KVLayer.prefill): a first
           prompt (p0 = 0) or a follow-up message over a cached conversation;
  proj     T tokens through a layer's q/k/v and o projections in a GGUF weight format (qkv_proj,
           o_proj and their *_rows forms): one decoded token, a few batched ones, a prompt;
  step /   a whole session over Flint's 49 attention blocks (Model.step, Model.prefill): the next
  prompt   token at position pos, and T tokens at position p0.

Shapes are Flint's (32 query heads, 4 KV heads, head dimension 128, hidden size 2048, SWA window
513 over a 1024-slot ring); inputs follow the library's tests and benchmark: raw q|k|v, cached V
and hidden rows ~ N(0, 1), gains ~ U(0.5, 1.5), sinks ~ N(0, 1), weight rows of unit gain.

exact() restates the maths in 64 bits with torch alone. Three things are taken as the path defines
them: K and V are rounded to the cache's type, a RoPE angle is the float product of the position
and a float frequency, and a weight is its GGUF block's value.
"""
import math
import os
import random
import sys
import tempfile

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "flint-mac_amd"))
import flint_attn as fa  # noqa: E402
import gguf_writer as gw  # noqa: E402

HEADS, KV_HEADS, DIM, EMBD, QKV = 32, 4, 128, 2048, 5120
GROUP, Q_DIM, KV_DIM = HEADS // KV_HEADS, HEADS * DIM, KV_HEADS * DIM
WINDOW, RING, THETA, EPS = 513, 1024, 1.0e4, 1e-6
# Flint's 49 layers: full attention at 0, 1, 5, ..., 45, 48, sliding window with RoPE elsewhere
FULL = [il in (0, 48) or il % 4 == 1 for il in range(49)]
VOCAB = 1024
KV = {"f16": torch.float16, "bf16": torch.bfloat16}
# bits of a weight: q8_0 34 bytes per 32, the k-quants and iq4_xs per 256
W_BITS = {"q8_0": 8.5, "q5_K": 5.5, "q6_K": 6.5625, "iq4_xs": 4.25, "f16": 16, "bf16": 16}


def listed():
    return [
        # the smallest call: one token of one conversation through a sliding-window layer
        dict(name="decode_swa", kind="decode", layer="swa", kv="f16", n_seq=1, ctx_lo=901, ctx_hi=901),
        # one long conversation through a full layer
        dict(name="decode_full_32k", kind="decode", layer="full", kv="f16", n_seq=1, ctx_lo=32768, ctx_hi=32768),
        # 16 conversations of 4k to 65k positions decoded together
        dict(name="decode_batch16", kind="decode", layer="full", kv="bf16", n_seq=16, ctx_lo=4096, ctx_hi=65536),
        # a long first prompt through a full layer and through a sliding-window one
        dict(name="prefill_full_4000", kind="prefill", layer="full", kv="bf16", T=4000, p0=0),
        dict(name="prefill_swa_4000", kind="prefill", layer="swa", kv="bf16", T=4000, p0=0),
        # a short follow-up message over a long cached conversation
        dict(name="prefill_turn", kind="prefill", layer="full", kv="f16", T=187, p0=20011),
        # one decoded token's projections
        dict(name="proj_token", kind="proj", T=1, w="q8_0", wv="q8_0"),
        # a batch of decoded tokens' projections, in the mixed formats of a 5-bit model file
        dict(name="proj_batch9", kind="proj", T=9, w="q5_K", wv="q6_K"),
        # a message's projections, and a long prompt's
        dict(name="proj_message", kind="proj", T=121, w="iq4_xs", wv="q8_0"),
        dict(name="proj_prompt", kind="proj", T=4000, w="q8_0", wv="q8_0"),
        # a session: the next token at 6001 cached positions; a 1000-token first prompt
        dict(name="model_step", kind="step", w="q8_0", pos=6001),
        dict(name="model_prompt", kind="prompt", w="q8_0", T=1000, p0=0),
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["decode"] * 3 + ["prefill"] * 3 + ["proj"] * 4 + ["step", "prompt"])
    if kind == "decode":
        n_seq = 1 if rng.random() < 0.4 else _log(rng, 2, 32)
        hi = _log(rng, 16, min(65536, 500000 // n_seq))
        lo = hi if n_seq == 1 else max(1, hi // rng.choice([1, 2, 4, 16]))
        return dict(kind=kind, layer=rng.choice(["full", "swa"]), kv=rng.choice(["f16", "bf16"]), n_seq=n_seq,
                    ctx_lo=lo, ctx_hi=hi)
    if kind == "prefill":
        layer, T = rng.choice(["full", "swa"]), _log(rng, 1, 4000)
        p0 = 0 if rng.random() < 0.4 else _log(rng, 16, 32768)
        if p0 and layer == "swa":  # a pass must not overwrite ring slots that its window reads
            T = min(T, RING - WINDOW)
        while T * (p0 + T / 2) > 4000 * 2000:
            p0 //= 2
        return dict(kind=kind, layer=layer, kv=rng.choice(["f16", "bf16"]), T=T, p0=p0)
    w = rng.choice(["q8_0", "q5_K", "q6_K", "iq4_xs"])
    if kind == "proj":
        T = 1 if rng.random() < 0.25 else _log(rng, 2, 4000)
        w = rng.choice([w, w, w, "f16", "bf16"])
        return dict(kind=kind, T=T, w=w, wv=rng.choice([w, "q8_0", "q6_K"]))
    if kind == "step":
        return dict(kind=kind, w=w, pos=_log(rng, 16, 8000))
    T = _log(rng, 2, 1000)
    return dict(kind=kind, w=w, T=T, p0=_log(rng, 16, 4000) if T <= RING - WINDOW and rng.random() < 0.5 else 0)


# ---- weights in the GGUF block layouts -------------------------------------------------------


def _half_bytes(h):
    return h.to(torch.float16).contiguous().view(torch.uint8).reshape(*h.shape, 2)


def _weights(w, n, k, g, dev):
    """n rows of k elements of format w, rows of unit gain, as uint8 [n][row bytes]: random quants
    and sub-block scales under super-block scales that give the elements a deviation of 1/sqrt(k)."""
    r = lambda lo, hi, *s: torch.randint(lo, hi, s, generator=g, device=dev, dtype=torch.int32)  # noqa: E731
    norm = lambda *s: torch.randn(s, generator=g, device=dev)  # noqa: E731
    std = 1 / math.sqrt(k)
    if w in KV:
        return (norm(n, k) * std).to(KV[w]).view(torch.uint8).reshape(n, 2 * k)
    if w == "q8_0":
        q = (norm(n, k // 32, 32) * 40).round().clamp(-127, 127).to(torch.int8).view(torch.uint8)
        d = (0.75 + 0.5 * torch.rand((n, k // 32), generator=g, device=dev)) * (std / 40)
        return torch.cat([_half_bytes(d), q], 2).reshape(n, -1)
    nb = k // 256
    u = 0.75 + 0.5 * torch.rand((n, nb), generator=g, device=dev)
    byte = lambda x: x.to(torch.uint8)  # noqa: E731
    if w == "q5_K":  # d * sc * q - dmin * m with m = sc and dmin = 15.5 d: elements centred on 0
        d = u * (std / (9.2 * 42))
        sc = r(20, 64, n, nb, 8)
        lo, hi = sc[..., :4], sc[..., 4:]
        s = torch.cat([lo | (hi >> 4 << 6), lo | (hi >> 4 << 6), (hi & 15) | ((hi & 15) << 4)], 2)
        return torch.cat([_half_bytes(d), _half_bytes(15.5 * d), byte(s), byte(r(0, 256, n, nb, 160))], 2).reshape(n, -1)
    if w == "q6_K":
        return torch.cat([byte(r(0, 256, n, nb, 192)), byte(r(32, 96, n, nb, 16)), _half_bytes(u * (std / (18.5 * 64)))],
                         2).reshape(n, -1)
    assert w == "iq4_xs"
    return torch.cat([_half_bytes(u * (std / (67 * 18.5))), byte(r(0, 256, n, nb, 134))], 2).reshape(n, -1)


def _elements(w, rows):
    """The rows' elements in 64 bits."""
    n = rows.shape[0]
    f64 = lambda b: b.contiguous().view(torch.float16).reshape(b.shape[:-1]).double()  # noqa: E731
    if w in KV:
        return rows.view(KV[w]).double()
    if w == "q8_0":
        b = rows.reshape(n, -1, 34)
        return (f64(b[..., :2])[..., None] * b[..., 2:].contiguous().view(torch.int8).double()).reshape(n, -1)
    b = rows.reshape(n, -1, {"q5_K": 176, "q6_K": 210, "iq4_xs": 136}[w])
    nb = b.shape[1]
    i = b.int()
    if w == "q5_K":
        s = i[..., 4:16]
        sc = torch.cat([s[..., :4] & 63, (s[..., 8:] & 15) | (s[..., :4] >> 6 << 4)], 2)
        mn = torch.cat([s[..., 4:8] & 63, (s[..., 8:] >> 4) | (s[..., 4:8] >> 6 << 4)], 2)
        ql, qh = i[..., 48:].reshape(n, nb, 4, 1, 32), i[..., 16:48].reshape(n, nb, 1, 1, 32)
        j = torch.arange(8, device=rows.device).reshape(1, 1, 4, 2, 1)
        q = ((ql >> 4 * (j & 1)) & 15) + (((qh >> j) & 1) << 4)
        d1 = f64(b[..., :2])[..., None] * sc
        m1 = f64(b[..., 2:4])[..., None] * mn
        return (d1[..., None] * q.reshape(n, nb, 8, 32) - m1[..., None]).reshape(n, -1)
    if w == "q6_K":  # halves of 128: quarter t of a half is ql[64 h + 32 (t & 1)] >> 4 (t >> 1), qh >> 2 t
        ql, qh = i[..., :128].reshape(n, nb, 2, 2, 32), i[..., 128:192].reshape(n, nb, 2, 1, 32)
        ql = torch.cat([ql & 15, ql >> 4], 3)
        t = torch.arange(4, device=rows.device).reshape(1, 1, 1, 4, 1)
        q = (ql | (((qh >> 2 * t) & 3) << 4)) - 32
        sc = b[..., 192:208].contiguous().view(torch.int8).double() * f64(b[..., 208:])[..., None]
        return (sc[..., None] * q.reshape(n, nb, 16, 16)).reshape(n, -1)
    assert w == "iq4_xs"
    table = torch.tensor([-127, -104, -83, -65, -49, -35, -22, -10, 1, 13, 25, 38, 53, 69, 89, 113], device=rows.device,
                         dtype=torch.float64)
    j = torch.arange(8, device=rows.device).reshape(1, 1, 8)
    low = (i[..., 4:8].repeat_interleave(2, dim=2) >> 4 * (j & 1)) & 15
    high = ((i[..., 2:3] | (i[..., 3:4] << 8)) >> 2 * j) & 3
    dl = f64(b[..., :2])[..., None] * ((low | (high << 4)) - 32)
    q = i[..., 8:].reshape(n, nb, 8, 16)
    return (dl[..., None] * table[torch.cat([q & 15, q >> 4], 3).long()]).reshape(n, -1)


# ---- inputs ----------------------------------------------------------------------------------


def _gen(seed, dev="cuda"):
    g = torch.Generator(device=dev)
    g.manual_seed(int(seed) & 0x7fffffffffff)
    return g


def _positions(case):
    """The sequences' positions: part of the case, the same for every seed."""
    r = random.Random("%(n_seq)d %(ctx_lo)d %(ctx_hi)d" % case)
    return [r.randint(case["ctx_lo"], case["ctx_hi"]) for _ in range(case["n_seq"])]


def _attention_inputs(case, seed):
    """Plain tensors of a decode or prefill case: the layer's weights, its cache and the raw q|k|v rows."""
    g, dev, dt = _gen(seed), "cuda", KV[case["kv"]]
    decode = case["kind"] == "decode"
    n_seq = case["n_seq"] if decode else 1
    top = max(_positions(case)) + 1 if decode else case["p0"] + case["T"]
    slots = RING if case["layer"] == "swa" else (top + 31) // 32 * 32
    u = lambda n: 0.5 + torch.rand(n, generator=g, device=dev)  # noqa: E731
    s = dict(q_norm=u(DIM), k_norm=u(DIM), sinks=torch.randn(HEADS, generator=g, device=dev), slots=slots, n_seq=n_seq,
             qkv=torch.randn((n_seq if decode else case["T"], QKV), generator=g, device=dev))
    for name in ("k", "v"):
        s[name] = torch.randn((n_seq, KV_HEADS, slots // 32, 32 * DIM), generator=g, device=dev, dtype=dt)
    return s


def _proj_inputs(case, seed):
    g, dev, T = _gen(seed), "cuda", case["T"]
    w, wv = case["w"], case["wv"]
    s = dict(wq=(_weights(w, Q_DIM, EMBD, g, dev), w), wk=(_weights(w, KV_DIM, EMBD, g, dev), w),
             wv=(_weights(wv, KV_DIM, EMBD, g, dev), wv), wo=(_weights(w, EMBD, Q_DIM, g, dev), w),
             norm=0.5 + torch.rand(EMBD, generator=g, device=dev))
    s["x"] = torch.randn((T, EMBD), generator=g, device=dev)
    s["att"] = torch.randn((T, Q_DIM), generator=g, device=dev)
    return s


def _model_tensors(w, dev):
    """The session's model: weights that belong to the format alone (a user has one model file)."""
    g = _gen(1000 + sorted(W_BITS).index(w), dev)
    u = lambda n: 0.5 + torch.rand(n, generator=g, device=dev)  # noqa: E731
    m = dict(embd=torch.randn((VOCAB, EMBD), generator=g, device=dev).half(), layers=[])
    for _ in FULL:
        m["layers"].append(dict(
            norm=u(EMBD), q_norm=u(DIM), k_norm=u(DIM), sinks=torch.randn(HEADS, generator=g, device=dev),
            q=_weights(w, Q_DIM, EMBD, g, dev), k=_weights(w, KV_DIM, EMBD, g, dev), v=_weights(w, KV_DIM, EMBD, g, dev),
            o=_weights(w, EMBD, Q_DIM, g, dev)))
    return m


_files = {}


def _model_file(w):
    """The model as a GGUF file, written once a process."""
    if w not in _files:
        m = _model_tensors(w, "cuda")
        f32 = lambda t: t.float().cpu().numpy()  # noqa: E731
        tensors = [("token_embd.weight", m["embd"].cpu().numpy(), gw.T_F16),
                   ("output_norm.weight", np.ones(EMBD, np.float32), gw.T_F32),
                   ("output.weight", np.zeros((1, EMBD), np.float32), gw.T_F16)]
        for il, L in enumerate(m["layers"]):
            b = "blk.%d." % il
            tensors.append((b + "attn_norm.weight", f32(L["norm"]), gw.T_F32))
            for name, key, k, n in (("attn_q", "q", EMBD, Q_DIM), ("attn_k", "k", EMBD, KV_DIM),
                                    ("attn_v", "v", EMBD, KV_DIM), ("attn_output", "o", Q_DIM, EMBD)):
                tensors.append((b + name + ".weight", L[key].cpu().numpy(), fa.W_TYPES[w], (k, n)))
            tensors += [(b + "attn_q_norm.weight", f32(L["q_norm"]), gw.T_F32),
                        (b + "attn_k_norm.weight", f32(L["k_norm"]), gw.T_F32),
                        (b + "attn_sinks.weight", f32(L["sinks"]), gw.T_F32)] + gw.flint_zero_ffn(il)
        swa = [not f for f in FULL]
        folder = tempfile.TemporaryDirectory()
        path = os.path.join(folder.name, "model.gguf")
        gw.write_gguf(path, gw.flint_meta(swa, swa, WINDOW, THETA, EPS, EMBD), tensors)
        _files[w] = (folder, path)
    return _files[w][1]


def _tokens(case, seed):
    n = case["pos"] + 1 if case["kind"] == "step" else case["p0"] + case["T"]
    r = random.Random(int(seed))
    return [r.randrange(VOCAB) for _ in range(n)]


def prepare(case, seed):
    if case["kind"] in ("decode", "prefill"):
        s = _attention_inputs(case, seed)
        swa = case["layer"] == "swa"
        kv = fa.KVLayer(is_swa=swa, has_rope=swa, n_slots=s["slots"], kv_dtype=case["kv"], rope_theta=THETA, window=WINDOW,
                        q_norm=s["q_norm"], k_norm=s["k_norm"], sinks=s["sinks"], n_seq=s["n_seq"], rms_eps=EPS)
        kv.k.copy_(s["k"].view_as(kv.k))
        kv.v.copy_(s["v"].view_as(kv.v))
        st = dict(case=case, kv=kv, qkv=s["qkv"], att=torch.empty((s["qkv"].shape[0], Q_DIM), device="cuda"))
        if case["kind"] == "decode":
            pos = _positions(case)
            st["pos"] = pos[0] if len(pos) == 1 else pos
        return st
    if case["kind"] == "proj":
        s = _proj_inputs(case, seed)
        s.update(case=case, qkv=torch.empty((case["T"], QKV), device="cuda"))
        return s
    # a session that has processed the tokens before the pass
    tokens = _tokens(case, seed)
    before = tokens[:case["pos"] if case["kind"] == "step" else case["p0"]]
    model = fa.Model(_model_file(case["w"]), n_ctx=(len(tokens) + 31) // 32 * 32)
    if before:
        model.prefill(before, torch.empty((len(before), EMBD), device="cuda"))
    n = len(tokens) - len(before)
    return dict(case=case, model=model, tokens=tokens[len(before):], pos=len(before), x=torch.empty((n, EMBD), device="cuda"))


def run(state):
    case, s = state["case"], state
    if case["kind"] == "decode":
        s["kv"].decode(s["qkv"], s["att"], s["pos"])
        return dict(att=s["att"], k=s["kv"].k, v=s["kv"].v)
    if case["kind"] == "prefill":
        s["kv"].prefill(s["qkv"], s["att"], case["p0"])
        return dict(att=s["att"], k=s["kv"].k, v=s["kv"].v)
    if case["kind"] == "proj":
        if case["T"] == 1:
            fa.qkv_proj(s["wq"], s["wk"], s["wv"], s["x"], s["norm"], s["qkv"], rms_eps=EPS)
            fa.o_proj(s["wo"], s["att"], s["x"])
        else:
            fa.qkv_proj_rows(s["wq"], s["wk"], s["wv"], s["x"], s["norm"], s["qkv"], rms_eps=EPS)
            fa.o_proj_rows(s["wo"], s["att"], s["x"])
        return dict(qkv=s["qkv"], x=s["x"])
    m = s["model"]
    if case["kind"] == "step":
        m.step(s["tokens"][0], s["x"][0])
    else:
        m.prefill(s["tokens"], s["x"])
    m.truncate(s["pos"])  # the next pass is the same position's
    return dict(x=s["x"])


# ---- what a pass cannot do without -----------------------------------------------------------


def _attended(layer, p0, T):
    """Key positions that the queries at p0 .. p0 + T - 1 attend to, summed; and the cached ones among them, each once."""
    if layer == "full":
        return T * p0 + T * (T + 1) // 2, p0
    return sum(min(p + 1, WINDOW) for p in range(p0, p0 + T)), min(p0, WINDOW - 1)


def _attention_work(layer, p0, T):
    pairs, cached = _attended(layer, p0, T)
    kept = T if layer == "full" else min(T, RING)
    return 4 * (T * (QKV + Q_DIM)) + 4 * KV_DIM * (cached + kept), 4 * Q_DIM * pairs


def _proj_work(w, wv, T):
    weights = (Q_DIM + KV_DIM) * EMBD * W_BITS[w] / 8 + KV_DIM * EMBD * W_BITS[wv] / 8 + EMBD * Q_DIM * W_BITS[w] / 8
    return weights + 4 * T * (EMBD + QKV + Q_DIM + EMBD), 2 * T * EMBD * (QKV + Q_DIM)


def work(case):
    kind = case["kind"]
    if kind == "decode":
        parts = [_attention_work(case["layer"], p, 1) for p in _positions(case)]
    elif kind == "prefill":
        parts = [_attention_work(case["layer"], case["p0"], case["T"])]
    elif kind == "proj":
        parts = [_proj_work(case["w"], case["wv"], case["T"])]
    else:
        # a session's pass: every layer's weights and the cached keys in, the tokens' K and V and the last hidden
        # rows out; what passes between the stages is not counted
        T, p0 = (1, case["pos"]) if kind == "step" else (case["T"], case["p0"])
        parts = [(4 * T * EMBD, 0)]
        for full in FULL:
            (ab, af), (pb, pf) = _attention_work("full" if full else "swa", p0, T), _proj_work(case["w"], case["w"], T)
            parts.append((ab - 4 * T * (QKV + Q_DIM) + pb - 4 * T * (2 * EMBD + QKV + Q_DIM), af + pf))
    return dict(bytes=sum(b for b, _ in parts), flops=sum(f for _, f in parts))


# ---- the same in 64 bits ---------------------------------------------------------------------


def _k_order():
    """Where (slot of a tile, dim) of K lies in its 4096-element tile (include/flint_attn.h)."""
    r, d = torch.arange(32, device="cuda")[:, None], torch.arange(DIM, device="cuda")[None, :]
    return (8 * (((r >> 2) & 1) * 256 + (d >> 5) * 64 + ((d >> 3) & 3) * 16 + ((r >> 3 << 2) | (r & 3))) + (d & 7)).reshape(-1)


def _slots_k(k):  # [KV_HEADS][tiles][4096] -> [KV_HEADS][slots][DIM]
    return k[..., _k_order()].reshape(KV_HEADS, -1, DIM)


def _slots_v(v):
    return v.reshape(KV_HEADS, -1, DIM, 32).transpose(2, 3).reshape(KV_HEADS, -1, DIM)


def _norm_rope(x, gain, pos, rope):
    """RMSNorm over the head dimension (+ NEOX RoPE) of x [T][heads][DIM] at positions pos [T]."""
    x = x.double()
    x = x / torch.sqrt(x.square().mean(-1, keepdim=True) + float(np.float32(EPS))) * gain.double()
    if not rope:
        return x
    freq = torch.tensor([float(np.float32(THETA ** (-2 * i / DIM))) for i in range(DIM // 2)], device=x.device).float()
    a = (pos.float()[:, None] * freq[None, :]).double()[:, None, :]
    x0, x1 = x[..., :DIM // 2], x[..., DIM // 2:]
    return torch.cat([x0 * a.cos() - x1 * a.sin(), x0 * a.sin() + x1 * a.cos()], -1)


def _attend(q, k, v, sinks, p0, base, swa):
    """Queries q [T][HEADS][DIM] at p0 .. over keys k, v [KV_HEADS][n][DIM] at positions base ..; out [T][Q_DIM]."""
    T, out = q.shape[0], torch.empty((q.shape[0], HEADS, DIM), device=q.device, dtype=torch.float64)
    for t0 in range(0, T, 512):
        t1 = min(T, t0 + 512)
        lo = max(0, p0 + t0 - (WINDOW - 1) - base) if swa else 0
        hi = p0 + t1 - base
        qp = torch.arange(p0 + t0, p0 + t1, device=q.device)[:, None]
        kp = torch.arange(base + lo, base + hi, device=q.device)[None, :]
        hidden = (kp > qp) | (qp - kp >= WINDOW if swa else kp < 0)
        for h in range(KV_HEADS):
            qh = q[t0:t1, h * GROUP:(h + 1) * GROUP].transpose(0, 1).reshape(-1, DIM)
            s = (qh @ k[h, lo:hi].T).reshape(GROUP, t1 - t0, hi - lo) / math.sqrt(DIM)
            s.masked_fill_(hidden, -math.inf)
            sink = sinks[h * GROUP:(h + 1) * GROUP].double()[:, None, None]
            top = torch.maximum(s.amax(-1, keepdim=True), sink)
            e = (s - top).exp()
            e /= e.sum(-1, keepdim=True) + (sink - top).exp()
            out[t0:t1, h * GROUP:(h + 1) * GROUP] = (e.reshape(-1, hi - lo) @ v[h, lo:hi]).reshape(GROUP, -1, DIM).transpose(0, 1)
    return out.reshape(T, Q_DIM)


def _attention(qkv, p0, old_k, old_v, q_norm, k_norm, sinks, swa, dt):
    """New rows qkv [T][QKV] at p0 over the cached old_k, old_v [KV_HEADS][n][DIM] that end at p0: the output, and the new
    K and V [T][KV_HEADS][DIM] as the cache (type dt) holds them."""
    T = qkv.shape[0]
    pos = torch.arange(p0, p0 + T, device=qkv.device)
    q = _norm_rope(qkv[:, :Q_DIM].reshape(T, HEADS, DIM), q_norm, pos, swa)
    k = _norm_rope(qkv[:, Q_DIM:Q_DIM + KV_DIM].reshape(T, KV_HEADS, DIM), k_norm, pos, swa).to(dt)
    v = qkv[:, Q_DIM + KV_DIM:].reshape(T, KV_HEADS, DIM).to(dt)
    ks = torch.cat([old_k.double(), k.transpose(0, 1).double()], 1)
    vs = torch.cat([old_v.double(), v.transpose(0, 1).double()], 1)
    return _attend(q, ks, vs, sinks, p0, p0 - old_k.shape[1], swa), k, v


def _exact_attention(case, seed):
    s = _attention_inputs(case, seed)
    swa, slots, dt = case["layer"] == "swa", s["slots"], KV[case["kv"]]
    out, order, d = [], _k_order().reshape(32, DIM), torch.arange(DIM, device="cuda")
    starts = _positions(case) if case["kind"] == "decode" else [case["p0"]]
    for i, p0 in enumerate(starts):
        qkv = s["qkv"][i:i + 1] if case["kind"] == "decode" else s["qkv"]
        first = max(0, p0 - (WINDOW - 1)) if swa else 0
        at = torch.arange(first, p0, device="cuda") % slots
        att, k, v = _attention(qkv, p0, _slots_k(s["k"][i])[:, at], _slots_v(s["v"][i])[:, at], s["q_norm"], s["k_norm"],
                               s["sinks"], swa, dt)
        out.append(att)
        keep = min(qkv.shape[0], slots)
        pos = torch.arange(p0 + qkv.shape[0] - keep, p0 + qkv.shape[0], device="cuda")
        tile, r = (pos % slots) // 32, pos % 32
        s["k"][i][:, tile[:, None], order[r]] = k[-keep:].transpose(0, 1)
        s["v"][i].view(KV_HEADS, -1, DIM, 32)[:, tile[:, None], d[None, :], r[:, None]] = v[-keep:].transpose(0, 1)
    return dict(att=torch.cat(out), k=s["k"], v=s["v"].reshape(s["n_seq"], KV_HEADS, slots // 32, DIM, 32))


def _normed(x, gain):
    return x / torch.sqrt(x.square().mean(-1, keepdim=True) + float(np.float32(EPS))) * gain.double()


def exact(case, seed):
    if case["kind"] in ("decode", "prefill"):
        return _exact_attention(case, seed)
    if case["kind"] == "proj":
        s = _proj_inputs(case, seed)
        x = s["x"].double()
        xn = _normed(x, s["norm"])
        qkv = torch.cat([xn @ _elements(t, w).T for w, t in (s["wq"], s["wk"], s["wv"])], 1)
        return dict(qkv=qkv, x=x + s["att"].double() @ _elements(s["wo"][1], s["wo"][0]).T)
    m, w = _model_tensors(case["w"], "cuda"), case["w"]
    tokens = torch.tensor(_tokens(case, seed), device="cuda")
    x = m["embd"][tokens].double()
    none = torch.empty((KV_HEADS, 0, DIM), device="cuda")
    for full, L in zip(FULL, m["layers"]):
        xn = _normed(x, L["norm"])
        qkv = torch.cat([xn @ _elements(w, L[key]).T for key in "qkv"], 1)
        att, _, _ = _attention(qkv, 0, none, none, L["q_norm"], L["k_norm"], L["sinks"], not full, torch.float16)
        x = x + att @ _elements(w, L["o"]).T
    return dict(x=x[-1:] if case["kind"] == "step" else x[case["p0"]:])


def tolerance(case):
    # about four times what exact() shows; "max" leaves room for a cached K or V one unit in the last place away
    if case["kind"] == "decode":  # fp32-accurate scores; the probabilities in two halves of the cache's type
        return {"rel": 4e-6 if case["kv"] == "f16" else 4e-5, "max": 0.01}
    if case["kind"] == "prefill":  # q and the probabilities enter the products in f16
        return {"rel": 1.2e-3, "max": 0.05}
    if case["kind"] == "proj":  # fp32 sums
        return {"rel": 1e-6, "max": 1e-4}
    return {"rel": 1.2e-3, "max": 0.05}  # 49 layers whose prompts pass q and the probabilities through f16
