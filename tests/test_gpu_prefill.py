"""Batched prefill (vx_prefill: MFMA GEMMs over chunks of up to 1024 tokens)
against the reference semantics, one backboneStep per prompt token
(src/engine.ts:2457-2472), as restated by the oracle: the KV cache of every
layer, the last token's W.normed and the position afterwards, with voice
rows spliced over [audio_start, audio_start + audio_count)."""
import os

import numpy as np
import pytest
import torch

import oracle as O
from vxtest import gpu_engine, max_rel_err, oracle_engine, tts_prompt, voice_rows

pytestmark = pytest.mark.gpu

SEED = 0


def oracle_prefill(o, tokens, a_start, a_count, voice):
    for i, t in enumerate(tokens):
        if voice is not None and a_start <= i < a_start + a_count:
            o.backbone_step(int(t), 2, voice[i - a_start])
        else:
            o.backbone_step(int(t))


def check_kv(g, o, layers, npos, bar=1e-3):
    for l in range(layers):
        for w in (0, 1):
            got = g.read_kv(l, w, 0, npos)
            ref = o.kv(l, w)[:npos]
            err = max_rel_err(got, ref)
            assert err < bar, (l, w, err)


@pytest.mark.parametrize("n,a_start,a_count,layers", [(40, 5, 8, 2), (7, 0, 0, 2), (256, 2, 64, 2),
                                                    (520, 100, 218, 1)])
def test_prefill_matches_single_steps(n, a_start, a_count, layers):
    """One chunk: GEMM columns sized to the prompt (16, 32 or a multiple of 64, hi and lo)."""
    print(f"[prefill] {layers} layers, {n} tokens, voice rows {a_start}+{a_count}", flush=True)
    g = gpu_engine(n_layers=layers, max_seq=1024)
    o = oracle_engine(n_layers=layers, max_seq=1024)
    try:
        rng = np.random.default_rng(n)
        tokens = rng.integers(0, 131072, n)
        voice = O.gen_f32(SEED + n, "voice", max(a_count, 1) * 3072).reshape(-1, 3072)
        g.prefill(tokens, a_start, a_count, voice if a_count else None)
        oracle_prefill(o, tokens, a_start, a_count, voice if a_count else None)
        assert g.position == n
        check_kv(g, o, layers, n)
        assert max_rel_err(g.debug_read("normed", 3072), o.buffer("normed")) < 1e-3
        # decoding continues from the prefilled state
        _, gn = g.backbone_step(24, 1)
        o.backbone_step(24, 1)
        assert max_rel_err(gn, o.buffer("normed")) < 1e-3
    finally:
        g.destroy()
        o.close()


@pytest.mark.parametrize("n,a_start,a_count,layers", [(40, 5, 8, 2), (256, 2, 64, 1)])
def test_prefill_f16_kv_matches_single_steps(n, a_start, a_count, layers):
    """The same with the f16 KV cache; the oracle rounds each new K/V row to
    f16 as the engine stores it.  Where the f32 value of a K/V element (GEMM
    vs per-token GEMV summation order) lies that close to an f16 rounding
    boundary, the two round to neighbouring halves.  So every element layer 0
    stores must be within one f16 ulp of the oracle's plus the f32 difference
    of the two summation orders (1e-5 of the largest value: several f16 ulps
    near zero, where the f16 spacing is finer than f32 noise at that scale),
    with flips on well under 1% of them.  Later layers see inputs perturbed
    by those flips, so they and the hidden state are held to the 1e-2 bar
    (measured: 3.4e-3 at layer 1, the same with the per-lane attention)."""
    print(f"[prefill f16 KV] {layers} layers, {n} tokens, voice rows {a_start}+{a_count}", flush=True)
    g = gpu_engine(n_layers=layers, max_seq=1024, kv_f16=True)
    o = oracle_engine(n_layers=layers, max_seq=1024)
    try:
        o.set_kv_f16(True)
        rng = np.random.default_rng(n + 1)
        tokens = rng.integers(0, 131072, n)
        voice = O.gen_f32(SEED + n + 1, "voice", a_count * 3072).reshape(-1, 3072)
        g.prefill(tokens, a_start, a_count, voice)
        oracle_prefill(o, tokens, a_start, a_count, voice)
        assert g.position == n
        for l in range(layers):
            for w in (0, 1):
                got, ref = g.read_kv(l, w, 0, n), o.kv(l, w)[:n]
                if l == 0:
                    ulp = np.spacing(np.abs(ref).astype(np.float16)).astype(np.float32)
                    tol = ulp + 1e-5 * np.abs(ref).max()
                    assert np.all(np.abs(got - ref) <= tol), (w, float(np.max(np.abs(got - ref) / tol)))
                    assert np.mean(got != ref) < 0.01, (w, float(np.mean(got != ref)))
                else:
                    assert max_rel_err(got, ref) < 1e-2, (l, w, max_rel_err(got, ref))
        assert max_rel_err(g.debug_read("normed", 3072), o.buffer("normed")) < 1e-2
        _, gn = g.backbone_step(24, 1)
        o.backbone_step(24, 1)
        assert max_rel_err(gn, o.buffer("normed")) < 1e-2
    finally:
        g.destroy()
        o.close()


@pytest.mark.parametrize("n", [1, 15, 16, 17, 32, 33, 64, 65, 129, 193])
def test_prefill_column_widths(n):
    """The edges of the GEMM's column widths: one column up to the whole 16,
    32 or 64 of the thin grids, then the multiples of 64, with the K slices
    each width picks (1e-3, the bar of the other prefill tests: both sides
    are f32 sums, which differ by about 1e-5)."""
    print(f"[prefill] 1 layer, {n} tokens", flush=True)
    g = gpu_engine(n_layers=1, max_seq=256)
    o = oracle_engine(n_layers=1, max_seq=256)
    try:
        tokens = np.random.default_rng(1000 + n).integers(0, 131072, n)
        g.prefill(tokens)
        oracle_prefill(o, tokens, 0, 0, None)
        assert g.position == n
        check_kv(g, o, 1, n)
        assert max_rel_err(g.debug_read("hidden", 3072), o.buffer("hidden")) < 1e-3
        assert max_rel_err(g.debug_read("normed", 3072), o.buffer("normed")) < 1e-3
    finally:
        g.destroy()
        o.close()


def test_prefill_two_chunks_after_context():
    """300 tokens on top of 10 cached positions in 256-token chunks: chunks
    of 256 and 44, the second attending to the first through the cache."""
    print("[prefill] 1 layer, 10 + 300 tokens, 256-token chunks", flush=True)
    os.environ["VX_PREFILL_CHUNK"] = "256"
    try:
        g = gpu_engine(n_layers=1, max_seq=512)
    finally:
        del os.environ["VX_PREFILL_CHUNK"]
    o = oracle_engine(n_layers=1, max_seq=512)
    try:
        rng = np.random.default_rng(7)
        head = rng.integers(0, 131072, 10)
        for t in head:
            g.backbone_step(int(t))
            o.backbone_step(int(t))
        tokens = rng.integers(0, 131072, 300)
        voice = O.gen_f32(SEED + 3, "voice", 20 * 3072).reshape(20, 3072)
        g.prefill(tokens, 250, 20, voice)  # voice rows straddle the chunk boundary
        oracle_prefill(o, tokens, 250, 20, voice)
        assert g.position == 310
        check_kv(g, o, 1, 310)
        assert max_rel_err(g.debug_read("normed", 3072), o.buffer("normed")) < 1e-3
    finally:
        g.destroy()
        o.close()


@pytest.mark.parametrize("kv_f16", [False, True])
def test_prefill_after_long_context(kv_f16):
    """96 prompt tokens on top of 2000 synthetic cache positions: every
    16-token query tile of the prompt attention walks 63-66 key tiles, split
    over its key groups and merged at the end.  The new K/V rows (f32 cache
    to 1e-3; f16 cache within one f16 ulp of the oracle's own f16 rounding,
    to 1e-2) and the last W.normed."""
    print(f"[prefill] 1 layer, 2000 cached + 96 tokens, f16 KV {kv_f16}", flush=True)
    from vxtest import fill_oracle_kv
    g = gpu_engine(n_layers=1, max_seq=2304, kv_f16=kv_f16)
    o = oracle_engine(n_layers=1, max_seq=2304)
    try:
        if kv_f16:
            o.set_kv_f16(True)
        g.fill_kv_synthetic(SEED, 2000)
        fill_oracle_kv(o, SEED, 2000)
        g.position = 2000
        o.position = 2000
        tokens = np.random.default_rng(21).integers(0, 131072, 96)
        g.prefill(tokens)
        oracle_prefill(o, tokens, 0, 0, None)
        assert g.position == 2096
        bar = 1e-2 if kv_f16 else 1e-3
        for w in (0, 1):
            got = g.read_kv(0, w, 2000, 96)
            ref = o.kv(0, w)[2000:2096]
            assert max_rel_err(got, ref) < bar, (w, max_rel_err(got, ref))
        assert max_rel_err(g.debug_read("normed", 3072), o.buffer("normed")) < bar
    finally:
        g.destroy()
        o.close()


@pytest.mark.parametrize("pos0,n", [(1, 3), (31, 1), (32, 33), (45, 20)])
@pytest.mark.parametrize("kv_f16", [False, True])
def test_prefill_context_ends_inside_a_key_tile(pos0, n, kv_f16):
    """The attention's 32-key tiles where old and new positions meet: a tile
    with one old key, one that the prompt only fills up, one that starts with
    it, one that holds both.  New K/V rows (f16 cache to 1e-2, as above), the
    old ones untouched, and the last W.normed."""
    print(f"[prefill] 1 layer, {pos0} cached + {n} tokens, f16 KV {kv_f16}", flush=True)
    from vxtest import fill_oracle_kv
    g = gpu_engine(n_layers=1, max_seq=96, kv_f16=kv_f16)
    o = oracle_engine(n_layers=1, max_seq=96)
    try:
        if kv_f16:
            o.set_kv_f16(True)
        g.fill_kv_synthetic(SEED, pos0)
        fill_oracle_kv(o, SEED, pos0)
        g.position = pos0
        o.position = pos0
        old = [g.read_kv(0, w, 0, pos0) for w in (0, 1)]
        tokens = np.random.default_rng(pos0).integers(0, 131072, n)
        g.prefill(tokens)
        oracle_prefill(o, tokens, 0, 0, None)
        bar = 1e-2 if kv_f16 else 1e-3
        for w in (0, 1):
            assert np.array_equal(g.read_kv(0, w, 0, pos0), old[w])
            assert max_rel_err(g.read_kv(0, w, pos0, n), o.kv(0, w)[pos0:pos0 + n]) < bar
        assert max_rel_err(g.debug_read("normed", 3072), o.buffer("normed")) < bar
    finally:
        g.destroy()
        o.close()


SHAPES = {"attention_norm": (3072,), "attention.wq": (4096, 3072), "attention.wk": (1024, 3072),
          "attention.wv": (1024, 3072), "attention.wo": (3072, 4096), "ffn_norm": (3072,),
          "feed_forward.w1": (9216, 3072), "feed_forward.w3": (9216, 3072), "feed_forward.w2": (3072, 9216)}


def weight_name(layer, part):
    return f"layers.{layer}.{part}.weight"


def layer_f64(g, layer, x, full=True):
    """One backbone layer over the rows x [n][3072] at positions 0 .. n - 1 in
    64-bit torch on the engine's weights: (attention's contribution to each
    row, output rows, K rows, V rows); the first two are None without `full`."""
    def w(part):
        bits = g.read_tensor(weight_name(layer, part), int(np.prod(SHAPES[part])))
        return torch.from_numpy(bits.view(np.float16).astype(np.float64)).reshape(SHAPES[part])

    def norm(x, part):
        return x / torch.sqrt((x * x).mean(-1, keepdim=True) + 1e-5) * w(part)

    def rope(y):
        ang = torch.arange(n, dtype=torch.float64)[:, None] * 1e6 ** (-torch.arange(0, 128, 2, dtype=torch.float64) / 128)
        c, s = torch.cos(ang)[:, None], torch.sin(ang)[:, None]
        y = y.reshape(n, -1, 64, 2)
        return torch.stack([y[..., 0] * c - y[..., 1] * s, y[..., 0] * s + y[..., 1] * c], -1).reshape(n, -1)

    n = x.shape[0]
    h = norm(x, "attention_norm")
    k, v = rope(h @ w("attention.wk").t()), h @ w("attention.wv").t()
    if not full:
        return None, None, k.numpy(), v.numpy()
    q = rope(h @ w("attention.wq").t())
    hide = torch.ones((n, n), dtype=torch.bool).tril().logical_not()
    a = torch.empty_like(q)
    for i in range(32):
        qi, ki, vi = q[:, 128 * i:128 * i + 128], k[:, i // 4 * 128:i // 4 * 128 + 128], v[:, i // 4 * 128:i // 4 * 128 + 128]
        a[:, 128 * i:128 * i + 128] = torch.softmax((qi @ ki.t() / 128 ** 0.5).masked_fill(hide, -np.inf), -1) @ vi
    a = a @ w("attention.wo").t()
    x = x + a
    h = norm(x, "ffn_norm")
    f = torch.nn.functional.silu(h @ w("feed_forward.w1").t()) * (h @ w("feed_forward.w3").t())
    return a.numpy(), x + f @ w("feed_forward.w2").t(), k.numpy(), v.numpy()


def rel_l2(got, ref):
    return float(np.linalg.norm(np.asarray(got, np.float64) - ref) / np.linalg.norm(ref))


@pytest.mark.parametrize("n", [700, 1030])
def test_prefill_long_chunks(n):
    """The GEMM grids of long prompts at the default chunk: shares of whole
    tiles with 256 x 128 tiles over an odd multiple of 64 columns (700 tokens:
    704), and a full 1024-token chunk with a short one behind it.  Layer 1's
    K/V rows depend on every product of layer 0 for every token; all of both
    layers' rows against 64 bits.  4e-5 relative: four times the 9.6e-6 seen,
    in K at the last positions, where the f32 rope angle is that far off; a
    column tile or K slice gone wrong is 1e-2 and more."""
    print(f"[prefill] 2 layers, {n} tokens in default chunks", flush=True)
    g = gpu_engine(n_layers=2, max_seq=1088)
    try:
        x = np.random.default_rng(n).standard_normal((n, 3072)).astype(np.float32)
        g.prefill(np.full(n, 24), 0, n, x)
        _, y, *kv0 = layer_f64(g, 0, torch.from_numpy(x).double())
        kv1 = layer_f64(g, 1, y, full=False)[2:]
        for l, kv in ((0, kv0), (1, kv1)):
            for w in (0, 1):
                got = g.read_kv(l, w, 0, n)
                errs = [rel_l2(got[r:r + 64], kv[w][r:r + 64]) for r in range(0, n, 64)]
                print(f"[prefill] layer {l} {'KV'[w]}: worst 64 rows {max(errs):.3g}", flush=True)
                assert max(errs) < 4e-5, (l, w, errs)
    finally:
        g.destroy()


def test_prompt_attention_small_queries():
    """Queries around 0.02 against keys around 140, so that scores are of
    order 1 although the queries' lo halves are f16 subnormals: their quantum,
    2^-24, must be the query's own and not that of a scaled-down one.  The
    attention's contribution to the last token against 64 bits.  Bound: a lo
    half is off by up to 2^-25, 1.7e-8 rms, against 0.02 a 1e-6 relative error
    of each term and so about that of a score; scores of 2-3 make it 3e-6 of
    the probabilities.  Seen: 1.8e-6, and 1.5e-5 where the queries were split in
    units of 0.13."""
    n = 64
    print(f"[prefill] {n} tokens, small queries", flush=True)
    g = gpu_engine(n_layers=1, max_seq=96)
    try:
        for part, by in (("attention.wq", 1 / 64), ("attention.wk", 128.0), ("feed_forward.w2", 0.0)):
            bits = g.read_tensor(weight_name(0, part), int(np.prod(SHAPES[part])))
            g.load_tensor(weight_name(0, part), (bits.view(np.float16) * np.float16(by)).view(np.uint16).reshape(SHAPES[part]))
        x = np.random.default_rng(4).standard_normal((n, 3072)).astype(np.float32)
        g.prefill(np.full(n, 24), 0, n, x)
        a, _, k, _ = layer_f64(g, 0, torch.from_numpy(x).double())
        assert rel_l2(g.read_kv(0, 0, 0, n), k) < 1e-6
        err = rel_l2(g.debug_read("hidden", 3072).astype(np.float64) - x[-1], a[-1])
        print(f"[prefill] small queries: {err:.3g}", flush=True)
        assert err < 5e-6
    finally:
        g.destroy()


@pytest.mark.parametrize("bad", [16, 29, 32])
@pytest.mark.parametrize("value", [np.inf, np.nan])
@pytest.mark.parametrize("kv_f16", [False, True])
def test_non_finite_token_leaves_earlier_blocks(kv_f16, value, bad):
    """A token whose input is not finite makes its own K/V rows so; the
    attention's blocks of 16 tokens before it hide those keys, and 0 times
    their values must stay 0: every layer's rows of the earlier blocks are
    bit-equal to those of the prompt without it."""
    n = 50
    print(f"[prefill] {n} tokens, token {bad} is {value}, f16 KV {kv_f16}", flush=True)
    g = gpu_engine(n_layers=2, max_seq=64, kv_f16=kv_f16)
    try:
        x = np.random.default_rng(bad).standard_normal((n, 3072)).astype(np.float32)
        first = bad // 16 * 16  # of the bad token's block
        g.prefill(np.full(n, 24), 0, n, x)
        want = [g.read_kv(l, w, 0, first) for l in (0, 1) for w in (0, 1)]
        x[bad] = value
        g.position = 0
        g.prefill(np.full(n, 24), 0, n, x)
        got = [g.read_kv(l, w, 0, first) for l in (0, 1) for w in (0, 1)]
        assert not np.isfinite(g.read_kv(0, 1, bad, 1)).all()
        for a, b in zip(got, want):
            assert np.array_equal(a, b)
    finally:
        g.destroy()


def test_prefill_argument_errors():
    import voxtral_amd as V
    g = gpu_engine(n_layers=1, max_seq=64)
    try:
        with pytest.raises(V.VoxtralError, match="out of range"):
            g.prefill([1, 2, 131072])
        with pytest.raises(V.VoxtralError, match="max_seq_len"):
            g.prefill(np.ones(65, np.int32))
        assert g.position == 0
    finally:
        g.destroy()


@pytest.mark.parametrize("layers,n_tok,n_voice", [(2, 256, 64), (26, 256, 64)])
def test_prompt_then_feedback_decode(layers, n_tok, n_voice):
    """The prompt configuration (a 256-token prompt with 64 voice rows,
    src/engine.ts:2457-2472) at full depth: the prompt laid out as
    buildTTSPrompt makes it with the reference's real voice rows (ar_male)
    spliced at offset 2, prefilled, then decode steps whose input is the
    previous step's W.normed through the precomputed-embedding path (the
    device loop the benchmark times, VX_TIME_FEEDBACK), against the oracle
    doing the same per step.  Checked: W.normed after the prompt and after
    the feedback steps, and every K/V row (prompt and feedback) of the first,
    middle and last layers."""
    steps = 8
    print(f"[prompt] {layers} layers, {n_tok}-token prompt, {n_voice} voice rows, {steps} feedback steps",
          flush=True)
    toks, a0, na = tts_prompt(n_tok, n_voice, seed=7)
    voice = voice_rows(n_voice)
    g = gpu_engine(n_layers=layers, max_seq=512)
    o = oracle_engine(n_layers=layers, max_seq=512)
    try:
        g.prefill(toks, a0, na, voice)
        oracle_prefill(o, toks, a0, na, voice)
        bar = 1e-3 if layers <= 2 else 1e-2
        err = max_rel_err(g.debug_read("normed", 3072), o.buffer("normed"))
        print(f"[prompt] normed after the prompt: max rel err {err:.2e}", flush=True)
        assert err < bar
        g.time_backbone_steps(steps, feedback=True)
        for _ in range(steps):
            o.backbone_step(precomputed=o.buffer("normed").copy())
        assert g.position == o.position == n_tok + steps
        err = max_rel_err(g.debug_read("normed", 3072), o.buffer("normed"))
        print(f"[prompt] normed after the feedback steps: max rel err {err:.2e}", flush=True)
        assert err < bar
        for l in sorted({0, layers // 2 - 1 if layers > 2 else 0, layers - 1}):
            for w in (0, 1):
                got = g.read_kv(l, w, 0, n_tok + steps)
                ref = o.kv(l, w)[:n_tok + steps]
                err_p = max_rel_err(got[:n_tok], ref[:n_tok])
                err_f = max_rel_err(got[n_tok:], ref[n_tok:])
                print(f"[prompt] layer {l} {'KV'[w]}: prompt rows {err_p:.2e}, feedback rows {err_f:.2e}",
                      flush=True)
                assert err_p < bar and err_f < bar, (l, w, err_p, err_f)
    finally:
        g.destroy()
        o.close()
