"""The work a program has this engine do, as timed cases: single calls of the
public class over the sizes, cache types and options in use, on a two-layer
backbone (one call then is a few kernels of each kind) and on the full
26-layer model.  Weights are random f16 (N(0, 0.02), gains around 1) loaded
through load_tensor; an engine is made once per shape and kept, as a serving
program keeps it, while every state has inputs of its own.
`exact` restates each path in 64-bit torch on the same weights and inputs."""
import math
import os
import sys
import zlib

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "webgpu-voxtral_amd"))

import voxtral_amd as V  # noqa: E402

DIM, HD, NH, NKV, HID = 3072, 128, 32, 8, 9216
QD, KVD = NH * HD, NKV * HD
VOCAB, AUDIO_VOCAB, SEMV, NAC, LEVELS = 131072, 9088, 8320, 36, 21
NFE, ALPHA, FM_LAYERS = 8, 1.2, 3
CD, CHID, CSEMD, CIN = 1024, 4096, 256, 292
MAX_SEQ = 4096
VOICE_AT = 2           # where buildTTSPrompt's voice rows start
AUDIO_TOKEN = 24       # the token that starts the frame loop
LAYER_PARAMS = (QD + 2 * KVD) * DIM + DIM * QD + 3 * HID * DIM
FM_HEAD = (SEMV + DIM) * DIM
EPS, FM_EPS, CODEC_EPS, QK_EPS, THETA = 1e-5, 1e-5, 0.01, 1e-6, 1e6
WINDOWS = (2, 4, 8, 16)


# ------------------------------------------------------------------ cases
def listed():
    return [
        # one sampled semantic code: the smallest call, a serving loop that
        # samples outside generate() makes one per frame
        {"name": "sample_top_p", "kind": "sample", "n": SEMV, "valid": 8194, "top_p": 0.9, "temp": 0.8},
        # a next-token step early in a context, with the tied LM head
        {"name": "step_lm_head", "kind": "step", "layers": 2, "ctx": 40, "kv16": 0, "lm": 1},
        # a step at the end of a long context, f16 cache
        {"name": "step_ctx3900_kv16", "kind": "step", "layers": 2, "ctx": 3900, "kv16": 1, "lm": 0},
        # the headline: one decode step of the full model at context 512
        {"name": "step_26_ctx512", "kind": "step", "layers": 26, "ctx": 512, "kv16": 0, "lm": 0},
        # one frame's flow-matching loop, hidden state to acoustic values
        {"name": "fm_frame", "kind": "fm"},
        # a few tokens (a short continuation), then the step that follows
        {"name": "prompt_9", "kind": "prompt", "layers": 2, "n": 9, "voice": 0, "kv16": 0, "at": 0},
        # a TTS prompt: 64 voice rows and an odd number of tokens
        {"name": "prompt_253_voice", "kind": "prompt", "layers": 2, "n": 253, "voice": 64, "kv16": 0, "at": 0},
        # a long text behind an earlier context, in two chunks, f16 cache
        {"name": "prompt_1300_kv16", "kind": "prompt", "layers": 2, "n": 1300, "voice": 64, "kv16": 1, "at": 500},
        # the 256-token prompt on the full model: time to the first frame
        {"name": "prompt_26_256", "kind": "prompt", "layers": 26, "n": 256, "voice": 64, "kv16": 0, "at": 0},
        # one second of audio, as a streaming caller decodes it
        {"name": "codec_13", "kind": "codec", "frames": 13},
        # a whole utterance: 20 seconds of audio
        {"name": "codec_250", "kind": "codec", "frames": 250},
        # an utterance end to end: prompt, frames on the device, audio
        {"name": "generate_16", "kind": "generate", "layers": 2, "n": 197, "voice": 64, "frames": 16, "sampling": "top_p"},
    ]


def _log_int(rng, lo, hi):
    return min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.49))))))


def draw(rng):
    kind = rng.choice(["sample", "step", "step", "fm", "prompt", "prompt", "prompt", "prompt_26", "codec", "codec",
                       "generate"])
    if kind == "sample":
        n = rng.randint(2000, SEMV)
        return {"kind": "sample", "n": n, "valid": rng.randint(n // 2, n), "top_p": round(rng.uniform(0.3, 1.0), 3),
                "temp": round(rng.uniform(0.4, 1.5), 3)}
    if kind == "step":
        return {"kind": "step", "layers": 2, "ctx": _log_int(rng, 1, MAX_SEQ - 1), "kv16": rng.randint(0, 1),
                "lm": rng.randint(0, 1)}
    if kind == "fm":
        return {"kind": "fm", "scale": round(rng.uniform(0.3, 3.0), 3)}
    if kind == "prompt":
        n = _log_int(rng, 1, 1300)
        return {"kind": "prompt", "layers": 2, "n": n, "voice": rng.choice([0, min(64, max(0, n - 5))]),
                "kv16": rng.randint(0, 1), "at": rng.choice([0, 0, rng.randint(1, 1000)])}
    if kind == "prompt_26":
        n = rng.randint(64, 256)
        return {"kind": "prompt", "layers": 26, "n": n, "voice": rng.randint(0, n - 5) // 2, "kv16": 0, "at": 0}
    if kind == "codec":
        return {"kind": "codec", "frames": _log_int(rng, 1, 250)}
    return {"kind": "generate", "layers": 2, "n": rng.randint(70, 197), "voice": rng.randint(16, 64),
            "frames": rng.randint(4, 16), "sampling": rng.choice(["top_p", "greedy"])}


# ---------------------------------------------------------------- weights
def _gen(name):
    return torch.Generator("cuda").manual_seed(zlib.crc32(name.encode()))


def _weight(name, shape, gain=False, std=0.02):
    w = torch.empty(shape, dtype=torch.float32, device="cuda").normal_(0.0, std, generator=_gen(name))
    return (w + 1.0 if gain else w).to(torch.float16)


def _layer_tensors(p):
    return {
        p + ".attention_norm.weight": ((DIM,), True), p + ".attention.wq.weight": ((QD, DIM), False),
        p + ".attention.wk.weight": ((KVD, DIM), False), p + ".attention.wv.weight": ((KVD, DIM), False),
        p + ".attention.wo.weight": ((DIM, QD), False), p + ".ffn_norm.weight": ((DIM,), True),
        p + ".feed_forward.w1.weight": ((HID, DIM), False), p + ".feed_forward.w2.weight": ((DIM, HID), False),
        p + ".feed_forward.w3.weight": ((HID, DIM), False)}


A = "acoustic_transformer."
C = "audio_tokenizer."
EMB = "mm_audio_embeddings.tok_embeddings.weight"


def _tensors(layers, codec):
    t = {EMB: ((VOCAB, DIM), False),
         "mm_audio_embeddings.audio_codebook_embeddings.embeddings.weight": ((AUDIO_VOCAB, DIM), False),
         "norm.weight": ((DIM,), True)}
    for i in range(layers):
        t.update(_layer_tensors("layers.%d" % i))
    for i in range(FM_LAYERS):
        t.update(_layer_tensors(A + "layers.%d" % i))
    t.update({A + "input_projection.weight": ((DIM, NAC), False), A + "llm_projection.weight": ((DIM, DIM), False),
              A + "time_projection.weight": ((DIM, DIM), False), A + "norm.weight": ((DIM,), True),
              A + "semantic_codebook_output.weight": ((SEMV, DIM), False),
              A + "acoustic_codebook_output.weight": ((NAC, DIM), False)})
    if not codec:
        return t
    conv = ".conv.parametrizations.weight.original"
    t.update({C + "decoder_blocks.0" + conv + "1": ((CD, CIN, 3), False), C + "decoder_blocks.0" + conv + "0": ((CD, 1, 1), True),
              C + "output_proj" + conv + "1": ((240, CD, 7), False), C + "output_proj" + conv + "0": ((240, 1, 1), True),
              C + "quantizer.semantic_codebook.embedding_sum": ((8192, CSEMD), False),
              C + "quantizer.semantic_codebook.cluster_usage": ((8192,), True)})
    for s in range(4):
        for l in range(2):
            p = C + "decoder_blocks.%d.layers.%d." % (1 + 2 * s, l)
            t.update({p + n: ((CD,), True) for n in ("attention_norm.weight", "attention.q_norm.weight", "attention.k_norm.weight",
                                                     "attention_scale", "ffn_norm.weight", "ffn_scale")})
            t.update({p + "attention.w%s.weight" % n: ((CD, CD), False) for n in "qkvo"})
            t.update({p + "feed_forward.w1.weight": ((CHID, CD), False), p + "feed_forward.w3.weight": ((CHID, CD), False),
                      p + "feed_forward.w2.weight": ((CD, CHID), False)})
        if s < 3:
            b = C + "decoder_blocks.%d" % (2 + 2 * s) + conv
            t.update({b + "1": ((CD, CD, 4), False), b + "0": ((CD, 1, 1), True)})
    return t


_engines = {}
_holds = {}  # engine -> positions its cache was last filled to


def _engine(layers, kv16, codec):
    key = (layers, kv16, codec)
    if key not in _engines:
        e = V.VoxtralEngine(V.default_config(n_layers=layers, kv_f16=kv16, codec=codec), max_seq_len=MAX_SEQ).init()
        for name, (shape, gain) in _tensors(layers, codec).items():
            e.load_tensor(name, _weight(name, shape, gain).cpu().numpy())
        _engines[key] = e
    return _engines[key]


def _kv_rows(layer, which, n):
    """Cached K or V rows [n][1024] of the context a step or prompt follows, exact in f16."""
    r = torch.empty((MAX_SEQ, KVD), dtype=torch.float32, device="cuda").normal_(0.0, 1.0, generator=_gen("kv.%d.%d" % (layer, which)))
    return r[:n].to(torch.float16).to(torch.float32)


def _context(e, layers, n):
    if _holds.get(id(e)) != n:
        for l in range(layers):
            for which in (0, 1):
                if n:
                    e.write_kv(l, which, 0, _kv_rows(l, which, n).cpu().numpy())
        _holds[id(e)] = n


# ----------------------------------------------------------------- inputs
def _inputs(case, seed):
    g = np.random.default_rng([seed, zlib.crc32(case["kind"].encode())])
    k = case["kind"]
    if k == "sample":
        x = (g.standard_normal(case["n"]) * 2.0).astype(np.float32)
        x[g.integers(1, case["valid"], 8)] += 6.0  # the few codes a trained head favours
        return {"logits": x, "state": int(g.integers(0, 2**62))}
    if k == "step":
        return {"x": g.standard_normal(DIM).astype(np.float32)}
    if k == "fm":
        return {"h": (g.standard_normal(DIM) * case.get("scale", 1.0)).astype(np.float32), "noise": g.standard_normal(NAC).astype(np.float32)}
    if k in ("prompt", "generate"):
        toks = g.integers(1000, VOCAB, case["n"]).astype(np.int32)
        voice = g.standard_normal((case["voice"], DIM)).astype(np.float32) if case["voice"] else None
        if voice is not None:
            toks[VOICE_AT:VOICE_AT + case["voice"]] = AUDIO_TOKEN
        return {"toks": toks, "voice": voice, "seed": int(g.integers(0, 2**31))}
    return {"sem": g.integers(2, 8192, case["frames"]).astype(np.uint32),
            "ac": g.integers(2, 2 + LEVELS, (case["frames"], NAC)).astype(np.uint32)}


def prepare(case, seed):
    k = case["kind"]
    s = _inputs(case, seed)
    layers, kv16 = case.get("layers", 2), case.get("kv16", 0)
    s["e"], s["case"] = _engine(layers, kv16, 0 if kv16 else 1), case
    if k == "step":
        _context(s["e"], layers, case["ctx"])
    elif k == "prompt":
        _context(s["e"], layers, case["at"])
    elif k == "generate":
        _holds.pop(id(s["e"]), None)  # the prompt overwrites the cache
    return s


def run(s):
    e, c = s["e"], s["case"]
    k = c["kind"]
    if k == "sample":
        code, state = e.sample_top_p(s["logits"], c["valid"], c["top_p"], c["temp"], s["state"])
        return [code, state >> 32, state & 0xFFFFFFFF]
    if k == "step":
        e.position = c["ctx"]
        top, normed = e.backbone_step(precomputed=s["x"], lm_head=bool(c["lm"]))
        return [normed, e.debug_read("logits", VOCAB), top] if c["lm"] else [normed]
    if k == "fm":
        e.debug_write("normed", s["h"])
        r = e.debug_fm_step(s["noise"])
        return [r["semantic_logits"], r["x_final"]]
    if k == "prompt":
        # the prompt, its last hidden state, and the step that starts the
        # frame loop: it reads every K/V row that the prompt wrote
        e.position = c["at"]
        e.prefill(s["toks"], VOICE_AT, c["voice"], s["voice"])
        last = e.debug_read("normed", DIM)
        return [last, e.backbone_step(AUDIO_TOKEN)[1]]
    if k == "codec":
        return [e.codec_decode(s["sem"], s["ac"])]
    r = e.generate(s["toks"], VOICE_AT, c["voice"], s["voice"], max_frames=c["frames"], sampling=c["sampling"],
                   seed=s["seed"], ignore_eos=True)
    return [np.array(r["semanticCodes"]), np.array(r["acousticCodes"]), r["audio"], e.debug_read("semantic_logits", SEMV)]


# ------------------------------------------------------------------- work
def _codec_work(T):
    flops, params, tt = 2 * T * CD * CIN * 3, CD * CIN * 3 + 240 * CD * 7 + 3 * CD * CD * 4, T
    for s, w in enumerate(WINDOWS):
        layer = 4 * CD * CD + 3 * CHID * CD
        params += 2 * layer
        flops += 2 * tt * (2 * layer + 2 * 2 * CD * w)
        if s < 3:
            tt *= 2
            flops += 2 * tt * CD * 2 * CD
    return 2 * params + T * (4 + 4 * NAC + 2 * CSEMD + 4 * 1920), flops + 2 * tt * 240 * CD * 7


def _step_work(layers, keys, kv_bytes):
    return (layers * (2 * LAYER_PARAMS + 2 * KVD * kv_bytes * (keys + 1)) + 8 * DIM,
            layers * (2 * LAYER_PARAMS + 4 * QD * keys))


def _prompt_work(layers, n, at, kv_bytes):
    keys = at + n
    return (layers * (2 * LAYER_PARAMS + 2 * KVD * kv_bytes * (keys + n)) + 2 * DIM * n,
            layers * (2 * LAYER_PARAMS * n + 4 * QD * (n * at + n * (n + 1) // 2)))


_FM_BYTES = (NFE - 1) * 2 * (FM_LAYERS * LAYER_PARAMS + 2 * DIM * NAC) + 2 * FM_HEAD
_FM_FLOPS = 6 * (NFE - 1) * 2 * FM_LAYERS * LAYER_PARAMS + 2 * FM_HEAD


def work(case):
    k = case["kind"]
    if k == "sample":
        return {"bytes": 4 * case["n"], "flops": 20 * case["n"]}
    kvb = 2 if case.get("kv16") else 4
    if k == "step":
        b, f = _step_work(case["layers"], case["ctx"] + 1, kvb)
        if case["lm"]:
            b, f = b + 2 * VOCAB * DIM + 4 * VOCAB, f + 2 * VOCAB * DIM
    elif k == "fm":
        # the weights cross HBM once per Euler step: 0.7 GB of them stay nowhere on the chip
        b, f = _FM_BYTES, _FM_FLOPS
    elif k == "codec":
        b, f = _codec_work(case["frames"])
    elif k == "prompt":
        b, f = _prompt_work(case["layers"], case["n"], case["at"], kvb)
        b2, f2 = _step_work(case["layers"], case["at"] + case["n"] + 1, kvb)
        b, f = b + b2, f + f2
    else:
        n, F = case["n"], case["frames"]
        b, f = _prompt_work(case["layers"], n, 0, kvb)
        bc, fc = _codec_work(F)
        b, f = b + bc + F * _FM_BYTES, f + fc + F * _FM_FLOPS
        for i in range(F):
            b1, f1 = _step_work(case["layers"], n + 1 + i, kvb)
            b, f = b + b1, f + f1
    return {"bytes": b, "flops": f}


def tolerance(case):
    """About four times what the path's f32 sums (and, with an f16 cache, the rounding of K and V
    values that lie near a tie) differ by from `exact`: seen are, as relative errors, 3e-6 for a
    step, 7e-7 for a frame, 4e-6 for a two-layer prompt (9e-5 behind an f16 cache), 1.2e-5 through
    26 layers and 2e-6 for audio; the worst single value was off by five times that."""
    k, kv16 = case["kind"], case.get("kv16")
    if k == "sample":
        return "exact"
    if k == "prompt":
        rel = 3.5e-4 if kv16 else 5e-5 if case["layers"] > 2 else 2e-5
    else:
        rel = {"step": 4e-5 if kv16 else 1.5e-5, "fm": 4e-6, "codec": 8e-6, "generate": 2e-5}[k]
    return {"rel": rel, "max": 5 * rel}


# ------------------------------------------------------------- 64 bits
def _w64(name, shape, gain=False):
    return _weight(name, shape, gain).to(torch.float64)


def _t64(a):
    return torch.from_numpy(np.ascontiguousarray(a)).to("cuda", torch.float64)


def _rms(x, g, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps) * g


def _rope(x, pos):
    """x [n][heads * 128], interleaved pairs; pos [n]"""
    n = x.shape[0]
    ang = pos[:, None] * THETA ** (-torch.arange(0, HD, 2, dtype=torch.float64, device="cuda") / HD)
    c, s = torch.cos(ang)[:, None], torch.sin(ang)[:, None]
    v = x.reshape(n, -1, HD // 2, 2)
    return torch.stack([v[..., 0] * c - v[..., 1] * s, v[..., 0] * s + v[..., 1] * c], -1).reshape(n, -1)


def _attend(q, k, v, at, causal=True):
    """q [n][4096], k and v [at + n][1024]; query i sees keys up to at + i"""
    out = torch.empty_like(q)
    n, m = q.shape[0], k.shape[0]
    hide = torch.ones((n, m), dtype=torch.bool, device="cuda").tril(at).logical_not()
    for h in range(NH):
        a, b = h * HD, (h * NKV // NH) * HD
        s = q[:, a:a + HD] @ k[:, b:b + HD].t() / math.sqrt(HD)
        if causal:
            s = s.masked_fill(hide, -math.inf)
        out[:, a:a + HD] = torch.softmax(s, -1) @ v[:, b:b + HD]
    return out


def _block(p, x, attend, eps):
    w = {n[len(p) + 1:]: _w64(n, sh, g) for n, (sh, g) in _layer_tensors(p).items()}
    h = _rms(x, w["attention_norm.weight"], eps)
    a = attend(*(h @ w["attention.w%s.weight" % c].t() for c in "qkv"))
    x = x + a @ w["attention.wo.weight"].t()
    h = _rms(x, w["ffn_norm.weight"], eps)
    return x + (torch.nn.functional.silu(h @ w["feed_forward.w1.weight"].t()) * (h @ w["feed_forward.w3.weight"].t())) @ w["feed_forward.w2.weight"].t()


def _backbone(x, layers, at, kv16):
    """Final-norm rows of x [n][3072] at positions at .. behind the prepared context."""
    n = x.shape[0]
    pos = torch.arange(at, at + n, dtype=torch.float64, device="cuda")

    def held(v):  # as the cache holds it
        return v.to(torch.float16).to(torch.float64) if kv16 else v

    for l in range(layers):
        def attend(q, k, v):
            old = [_kv_rows(l, w, at).to(torch.float64) for w in (0, 1)]
            return _attend(_rope(q, pos), torch.cat([old[0], held(_rope(k, pos))]), torch.cat([old[1], held(v)]), at)
        x = _block("layers.%d" % l, x, attend, EPS)
    return _rms(x, _w64("norm.weight", (DIM,), True), EPS)


def _fm(h, noise):
    t = {n[len(A):]: _w64(n, sh, g) for n, (sh, g) in _tensors(0, 0).items() if n.startswith(A) and ".layers." not in n}
    sem, llm = t["semantic_codebook_output.weight"] @ h, t["llm_projection.weight"] @ h
    x, half, dt = noise, DIM // 2, 1.0 / (NFE - 1)
    freq = torch.exp(-math.log(1e4) * torch.arange(half, dtype=torch.float64, device="cuda") / half)

    def attend(q, k, v):
        return torch.cat([_attend(q[i:i + 3], k[i:i + 3], v[i:i + 3], 0, causal=False) for i in (0, 3)])

    for step in range(NFE - 1):
        tp = t["time_projection.weight"] @ torch.cat([torch.cos(step * dt * freq), torch.sin(step * dt * freq)])
        xp = t["input_projection.weight"] @ x
        seq = torch.stack([xp, tp, llm, xp, tp, torch.zeros_like(llm)])
        for i in range(FM_LAYERS):
            seq = _block(A + "layers.%d" % i, seq, attend, FM_EPS)
        v = _rms(seq[[0, 3]], t["norm.weight"], FM_EPS) @ t["acoustic_codebook_output.weight"].t()
        x = x + (ALPHA * v[0] + (1 - ALPHA) * v[1]) * dt
    return [sem, x]


def _codec(sem, ac):
    w = {n[len(C):]: _w64(n, sh, g) for n, (sh, g) in _tensors(0, 1).items() if n.startswith(C)}
    T = sem.shape[0]
    dev = torch.device("cuda")
    cb = w["quantizer.semantic_codebook.embedding_sum"] / w["quantizer.semantic_codebook.cluster_usage"].clamp(min=1e-5)[:, None]
    cb = cb.to(torch.float16).to(torch.float64)
    x = torch.cat([cb[torch.from_numpy(sem.astype(np.int64)).to(dev)], (_t64(ac) - 2.0) * 2.0 / (LEVELS - 1) - 1.0], 1)

    def conv(x, v, g):  # causal, weight-normed: v [out][in][k]
        k = v.shape[2]
        v = v * (g.reshape(-1) / v.flatten(1).norm(dim=1))[:, None, None]
        p = torch.cat([x.new_zeros(k - 1, x.shape[1]), x])
        return sum(p[j:j + x.shape[0]] @ v[:, :, j].t() for j in range(k))

    def up(x, v, g):  # stride 2, kernel 4: v [in][out][4]
        v = v * (g.reshape(-1) / v.flatten(1).norm(dim=1))[:, None, None]
        q = torch.cat([x.new_zeros(1, x.shape[1]), x[:-1]])
        return torch.stack([x @ v[:, :, r] + q @ v[:, :, r + 2] for r in (0, 1)], 1).reshape(2 * x.shape[0], -1)

    n = ".conv.parametrizations.weight.original"
    x = conv(x, w["decoder_blocks.0" + n + "1"], w["decoder_blocks.0" + n + "0"])
    slope = 2.0 ** -torch.arange(1, 9, dtype=torch.float64, device=dev)
    for s in range(4):
        T = x.shape[0]
        for l in range(2):
            def p(name):
                return w["decoder_blocks.%d.layers.%d.%s" % (1 + 2 * s, l, name)]
            h = _rms(x, p("attention_norm.weight"), CODEC_EPS)
            q, k, v = ((h @ p("attention.w%s.weight" % c).t()).reshape(T, 8, HD) for c in "qkv")
            q, k = _rms(q, p("attention.q_norm.weight").reshape(8, HD), QK_EPS), _rms(k, p("attention.k_norm.weight").reshape(8, HD), QK_EPS)
            W = WINDOWS[s]
            pad = x.new_zeros(W - 1, 8, HD)
            ks, vs = (torch.cat([pad, z]).unfold(0, W, 1) for z in (k, v))  # [T][8][128][W]
            back = torch.arange(W - 1, -1, -1, device=dev)
            sc = (q[..., None] * ks).sum(2) / math.sqrt(HD) - slope[:, None] * back
            sc = sc.masked_fill((torch.arange(T, device=dev)[:, None] < back)[:, None], -math.inf)
            a = (torch.softmax(sc, -1)[:, :, None] * vs).sum(-1).reshape(T, CD)
            x = x + (a @ p("attention.wo.weight").t()) * p("attention_scale")
            h = _rms(x, p("ffn_norm.weight"), CODEC_EPS)
            f = torch.nn.functional.silu(h @ p("feed_forward.w1.weight").t()) * (h @ p("feed_forward.w3.weight").t())
            x = x + (f @ p("feed_forward.w2.weight").t()) * p("ffn_scale")
        if s < 3:
            b = "decoder_blocks.%d" % (2 + 2 * s) + n
            x = up(x, w[b + "1"], w[b + "0"])
    return conv(x, w["output_proj" + n + "1"], w["output_proj" + n + "0"]).reshape(-1)


def _sample(case, i):
    s = (i["logits"].astype(np.float64) / case["temp"]).astype(np.float32)
    s[0] = s[case["valid"]:] = -np.inf
    p = np.exp(s.astype(np.float64) - float(s.max())).astype(np.float32)
    p = (p.astype(np.float64) / p.sum(dtype=np.float64)).astype(np.float32)
    order = np.argsort(-p, kind="stable")
    cum = np.cumsum(p[order], dtype=np.float64)
    cut = min(int(np.searchsorted(cum, case["top_p"])) + 1, len(cum))
    m = (1 << 64) - 1
    state = z = (i["state"] + 0x9E3779B97F4A7C15) & m
    z = ((z ^ (z >> 30)) * 0xBF58476D1CE4E5B9) & m
    z = ((z ^ (z >> 27)) * 0x94D049BB133111EB) & m
    r = float((z ^ (z >> 31)) >> 11) * 2.0**-53 * cum[cut - 1]
    return [int(order[int(np.searchsorted(cum[:cut], r))]), state >> 32, state & 0xFFFFFFFF]


def exact(case, seed):
    k = case["kind"]
    i = _inputs(case, seed)
    if k == "sample":
        return _sample(case, i)
    if k == "step":
        h = _backbone(_t64(i["x"])[None], case["layers"], case["ctx"], case["kv16"])[0]
        if not case["lm"]:
            return [h]
        emb = _weight(EMB, (VOCAB, DIM))
        logits = torch.cat([emb[r:r + 8192].to(torch.float64) @ h for r in range(0, VOCAB, 8192)])
        return [h, logits, int(logits.argmax())]
    if k == "fm":
        return _fm(_t64(i["h"]), _t64(i["noise"]))
    if k == "prompt":
        emb = _weight(EMB, (VOCAB, DIM))
        ids = torch.from_numpy(np.append(i["toks"], AUDIO_TOKEN).astype(np.int64)).to("cuda")
        x = emb[ids].to(torch.float64)
        if case["voice"]:
            x[VOICE_AT:VOICE_AT + case["voice"]] = _t64(i["voice"])
        r = _backbone(x, case["layers"], case["at"], case["kv16"])
        return [r[-2], r[-1]]
    if k == "codec":
        return [_codec(i["sem"], i["ac"])]
    return None  # generate(): the frames feed each other through quantised codes
