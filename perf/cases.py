"""The work a transcription service has this library do, as measurable cases.

A request goes: 30 s log-mel chunks through the audio encoder and the adaptor
(`audio_*`), the prompt's rows through the decoder (`prefill_*`), then one
token per step and row (`decode_*`, `logits_*`).  Shapes are those of the
library's own configurations: the Whisper-medium encoder with the adaptor
(fmd.WHISPER_MEDIUM) and the 0.6B decoder (fmd.QWEN3_0_6B), the latter with
fewer layers and a 2048-token vocabulary where one layer is what counts.

Values: linear weights N(0, 0.02^2) (the encoder's q and k 0.04, so that its
softmax is not flat), norm gains around 1, encoder hidden states, cache
contents and prompt rows N(0, 1) (audio rows leave the adaptor's LayerNorm with
unit variance), mel values uniform in the range of normalised log-mel.
"""
from __future__ import annotations

import ctypes
import importlib
import math
import zlib

import numpy as np
import torch

fmd = importlib.import_module("fast-moss-diarization_amd")

DEV = "cuda"
ACT = {"bf16": torch.bfloat16, "f16": torch.float16, "int8": torch.float16}
# dtype of the checkpoint tensors handed to the library
SRC = {"bf16": torch.bfloat16, "f16": torch.float16, "int8": torch.bfloat16}
HALF = 1 << 31  # seeds are folded below 2^31


# --- the cases -----------------------------------------------------------------


def listed():
    return [
        # one short recording: a single 30 s window in an encoder layer
        dict(name="audio_layer_1x1500_bf16", kind="audio_layer", prec="bf16", windows=1, t=1500),
        # a full encoder batch (the default of 16 windows per pass), the audio path's bulk
        dict(name="audio_layer_16x1500_bf16", kind="audio_layer", prec="bf16", windows=16, t=1500),
        # chunks shorter than 30 s, in the int8 precision's f16 audio path
        dict(name="audio_layer_5x1137_f16", kind="audio_layer", prec="f16", windows=5, t=1137),
        # a four-minute recording, mel to decoder rows: stem, 24 layers, adaptor
        dict(name="audio_encode_8_int8", kind="audio_encode", prec="int8", chunks=8, audios=3,
             tokens_seed=7),
        # a single 30 s request to its first two tokens' logits, whole model
        dict(name="prefill_1x450_int8_full", kind="prefill", prec="int8", layers=28, vocab=151936,
             batch=1, lo=450, hi=450, lens_seed=1, chunk=256),
        # a micro-batch of short and medium prompts in the default chunks
        dict(name="prefill_4x310_1890_f16", kind="prefill", prec="f16", layers=2, vocab=2048, batch=4,
             lo=310, hi=1890, lens_seed=2, chunk=256),
        # a micro-batch of long recordings in large chunks, the prefill's bulk
        dict(name="prefill_8x1500_8000_bf16", kind="prefill", prec="bf16", layers=2, vocab=2048,
             batch=8, lo=1500, hi=8000, lens_seed=4, chunk=512),
        # one row's token in one layer: latency
        dict(name="decode_layer_1x450_int8", kind="decode_layer", prec="int8", batch=1, lo=450, hi=450,
             lens_seed=3),
        # the full micro-batch over a 4k context in one layer
        dict(name="decode_layer_8x4096_int8", kind="decode_layer", prec="int8", batch=8, lo=4096,
             hi=4096, lens_seed=3),
        # the largest batch with ragged contexts, bf16 weights
        dict(name="decode_layer_16x1024_4096_bf16", kind="decode_layer", prec="bf16", batch=16, lo=1024,
             hi=4096, lens_seed=6),
        # the head of one decode step: final norm and the whole vocabulary
        dict(name="logits_8_int8", kind="logits", prec="int8", rows=8, vocab=151936),
        # one token for every row of a micro-batch, whole model
        dict(name="decode_step_8x500_1500_int8_full", kind="decode_step", prec="int8", layers=28,
             vocab=151936, batch=8, lo=500, hi=1500, lens_seed=5),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["audio_layer", "audio_layer", "audio_encode", "prefill", "prefill", "prefill",
                       "decode_layer", "decode_layer", "logits", "decode_step"])
    seed = rng.randrange(1 << 20)
    if kind == "audio_layer":
        return dict(kind=kind, prec=rng.choice(["bf16", "f16"]), windows=_log_int(rng, 1, 16),
                    t=rng.randint(100, 1500))
    if kind == "audio_encode":
        chunks = _log_int(rng, 1, 8)
        return dict(kind=kind, prec="int8", chunks=chunks, audios=rng.randint(1, chunks), tokens_seed=seed)
    prec = rng.choice(["bf16", "f16", "int8"])
    if kind == "logits":
        return dict(kind=kind, prec=prec, rows=rng.randint(1, 16), vocab=16 * _log_int(rng, 128, 9496))
    if kind == "decode_step":
        lo = _log_int(rng, 30, 1000)
        return dict(kind=kind, prec="int8", layers=28, vocab=151936, batch=rng.randint(1, 8), lo=lo,
                    hi=min(1500, 3 * lo), lens_seed=seed)
    if kind == "decode_layer":
        lo = _log_int(rng, 30, 4096)
        return dict(kind=kind, prec=prec, batch=_log_int(rng, 1, 16), lo=lo, hi=min(4096, 3 * lo),
                    lens_seed=seed)
    lo = _log_int(rng, 20, 4000)
    return dict(kind=kind, prec=prec, layers=2, vocab=2048, batch=_log_int(rng, 1, 8), lo=lo,
                hi=min(5000, 4 * lo), lens_seed=seed, chunk=rng.choice([256, 512]))


# --- inputs --------------------------------------------------------------------


def _gen(seed, tag):
    g = torch.Generator(device=DEV)
    g.manual_seed((int(seed) * 1000003 + zlib.crc32(tag.encode())) % HALF)
    return g


def _normal(seed, tag, shape, dtype, std=1.0, mean=0.0):
    x = torch.randn(shape, generator=_gen(seed, tag), device=DEV, dtype=torch.float32)
    return (x * std + mean).to(dtype)


def _lens(case):
    r = np.random.default_rng(case["lens_seed"])
    return [int(n) for n in r.integers(case["lo"], case["hi"] + 1, case["batch"])]


def _ids(case, seed, tag, n):
    r = np.random.default_rng([int(seed), zlib.crc32(tag.encode())])
    return [int(v) for v in r.integers(0, case["vocab"], n)]


def _text_config(layers, vocab):
    return fmd.TextConfig(vocab_size=vocab, hidden_size=1024, intermediate_size=3072,
                          num_hidden_layers=layers, num_attention_heads=16, num_key_value_heads=8,
                          head_dim=128, rms_norm_eps=1e-6, rope_theta=1e6,
                          max_position_embeddings=131_072, tie_word_embeddings=True)


def _text_layer(cfg, prec, seed, i):
    """The checkpoint tensors of decoder layer i."""
    H, I, hd, dt = cfg.hidden_size, cfg.intermediate_size, cfg.head_dim, SRC[prec]
    p = f"layers.{i}."
    lin = {"self_attn.q_proj": (cfg.q_dim(), H), "self_attn.k_proj": (cfg.kv_dim(), H),
           "self_attn.v_proj": (cfg.kv_dim(), H), "self_attn.o_proj": (H, cfg.q_dim()),
           "mlp.gate_proj": (I, H), "mlp.up_proj": (I, H), "mlp.down_proj": (H, I)}
    gain = {"input_layernorm": H, "post_attention_layernorm": H, "self_attn.q_norm": hd,
            "self_attn.k_norm": hd}
    w = {p + n + ".weight": _normal(seed, p + n, s, dt, 0.02) for n, s in lin.items()}
    w.update({p + n + ".weight": _normal(seed, p + n, (s,), dt, 0.02, 1.0) for n, s in gain.items()})
    return w


def _text_top(cfg, prec, seed):
    return {"embed_tokens.weight": _normal(seed, "embed", (cfg.vocab_size, cfg.hidden_size), SRC[prec], 0.02),
            "norm.weight": _normal(seed, "norm", (cfg.hidden_size,), SRC[prec], 0.02, 1.0)}


def _decoder(case, seed, layers, vocab, max_len):
    cfg = _text_config(layers, vocab)
    m = fmd.Qwen3(cfg, case["prec"], max_len=max_len)
    torch.cuda.synchronize()
    for i in range(layers):
        for n, t in _text_layer(cfg, case["prec"], seed, i).items():
            torch.cuda.synchronize()
            m.set_weight(n, t)
    for n, t in _text_top(cfg, case["prec"], seed).items():
        torch.cuda.synchronize()
        m.set_weight(n, t)
    return m


AUDIO = "model.whisper_encoder."
ADAPT = "model.vq_adaptor."


def _audio_tensor(cfg, prec, seed, name, shape):
    dt = ACT[prec]
    if "norm" in name or name.startswith(ADAPT + "layers.3"):
        return _normal(seed, name, shape, dt, 0.02, 1.0 if name.endswith("weight") else 0.0)
    if "embed_positions" in name:
        return _normal(seed, name, shape, dt, 0.1)
    if name.endswith("conv1.weight"):
        return _normal(seed, name, shape, dt, 1.0 / math.sqrt(3.0 * cfg.num_mel_bins))
    if "q_proj.weight" in name or "k_proj.weight" in name:
        return _normal(seed, name, shape, dt, 0.04)
    return _normal(seed, name, shape, dt, 0.02)


def _audio_shapes(cfg):
    """Names and shapes of the audio path's checkpoint tensors."""
    d, f, m, H = cfg.d_model, cfg.encoder_ffn_dim, cfg.num_mel_bins, cfg.hidden_size
    s = {AUDIO + "conv1.weight": (d, m, 3), AUDIO + "conv1.bias": (d,),
         AUDIO + "conv2.weight": (d, d, 3), AUDIO + "conv2.bias": (d,),
         AUDIO + "embed_positions.weight": (cfg.max_source_positions, d),
         AUDIO + "layer_norm.weight": (d,), AUDIO + "layer_norm.bias": (d,),
         ADAPT + "layers.0.weight": (H, cfg.adaptor_input_dim), ADAPT + "layers.0.bias": (H,),
         ADAPT + "layers.2.weight": (H, H), ADAPT + "layers.2.bias": (H,),
         ADAPT + "layers.3.weight": (H,), ADAPT + "layers.3.bias": (H,)}
    for i in range(cfg.encoder_layers):
        p = AUDIO + f"layers.{i}."
        for n, shape in (("self_attn.q_proj", (d, d)), ("self_attn.k_proj", (d, d)),
                         ("self_attn.v_proj", (d, d)), ("self_attn.out_proj", (d, d)),
                         ("fc1", (f, d)), ("fc2", (d, f))):
            s[p + n + ".weight"] = shape
            if n != "self_attn.k_proj":
                s[p + n + ".bias"] = shape[:1]
        for n in ("self_attn_layer_norm", "final_layer_norm"):
            s[p + n + ".weight"] = (d,)
            s[p + n + ".bias"] = (d,)
    return s


def _audio_encoder(prec, seed, layers):
    cfg = fmd.AudioConfig(encoder_layers=layers)
    e = fmd.AudioEncoder(cfg, prec)
    for n, shape in _audio_shapes(cfg).items():
        t = _audio_tensor(cfg, prec, seed, n, shape)
        torch.cuda.synchronize()
        e.set_weight(n, t)
    return e


def _chunk_tokens(case):
    """Per 30 s chunk its token count (at most 375) and its audio: the last
    chunk of each audio is cut short."""
    r = np.random.default_rng(case["tokens_seed"])
    n, a = case["chunks"], case["audios"]
    mapping = sorted(list(range(a)) + [int(v) for v in r.integers(0, a, n - a)])
    tokens = [375 if i + 1 < n and mapping[i + 1] == mapping[i] else int(r.integers(40, 376))
              for i in range(n)]
    return tokens, mapping


def _mel(case, seed):
    return torch.rand((case["chunks"], 80, 3000), generator=_gen(seed, "mel"), device=DEV) * 2.5 - 1.0


def _prompt_rows(case, seed, lens):
    """Left-padded (batch, longest, 1024) prompt rows and the pads."""
    total = max(lens)
    pad = [total - n for n in lens]
    x = _normal(seed, "prompt", (len(lens), total, 1024), ACT[case["prec"]])
    for b, p in enumerate(pad):
        x[b, :p] = 0
    return x, pad


def _cache_rows(case, seed, length):
    """(K, V) of one layer: (batch, 8, length, 128)."""
    shape = (case["batch"], 8, length, 128)
    return tuple(_normal(seed, n, shape, ACT[case["prec"]]) for n in ("cache k", "cache v"))


def prepare(case, seed):
    k = case["kind"]
    s = {"case": case}
    if k == "audio_layer":
        s["enc"] = _audio_encoder(case["prec"], seed, 1)
        s["x"] = _normal(seed, "hidden", (case["windows"], case["t"], 1024), ACT[case["prec"]])
        s["out"] = torch.empty_like(s["x"])
    elif k == "audio_encode":
        s["enc"] = _audio_encoder(case["prec"], seed, 24)
        s["mel"] = _mel(case, seed)
        s["tokens"], s["mapping"] = _chunk_tokens(case)
    elif k == "prefill":
        lens = _lens(case)
        cap = max(lens) + 256
        s["dec"] = _decoder(case, seed, case["layers"], case["vocab"], cap)
        s["emb"], s["pad"] = _prompt_rows(case, seed, lens)
        s["kv"] = s["dec"].new_caches(case["batch"], cap)
        s["ids"] = _ids(case, seed, "next", case["batch"])
    elif k == "decode_layer":
        lens = _lens(case)
        L = max(lens)
        s["L"], s["pad"] = L, [L - n for n in lens]
        s["dec"] = _decoder(case, seed, 1, 2048, L + 256)
        s["kv"] = s["dec"].new_caches(case["batch"], L + 256)
        bits = np.uint16 if case["prec"] == "bf16" else np.float16
        for which, t in enumerate(_cache_rows(case, seed, L)):
            full = torch.zeros((case["batch"], 8, L + 256, 128), dtype=t.dtype, device=DEV)
            full[:, :, :L] = t
            s["kv"].write(0, which, full.view(torch.int16).cpu().numpy().view(bits))
        s["kv"].set_len(L)
        s["x0"] = _normal(seed, "hidden", (case["batch"], 1024), ACT[case["prec"]])
        s["x"] = torch.empty_like(s["x0"])
        # the layer runs in place: its input is put back on the same stream
        s["stream"] = torch.cuda.Stream()
        s["dec"].set_stream(s["stream"].cuda_stream)
    elif k == "logits":
        s["dec"] = _decoder(case, seed, 1, case["vocab"], 64)
        s["x"] = _normal(seed, "hidden", (case["rows"], 1024), ACT[case["prec"]])
        s["out"] = torch.empty((case["rows"], case["vocab"]), device=DEV, dtype=torch.float32)
    else:
        lens = _lens(case)
        cap = max(lens) + 256
        s["dec"] = _decoder(case, seed, case["layers"], case["vocab"], cap)
        emb, s["pad"] = _prompt_rows(case, seed, lens)
        s["kv"] = s["dec"].new_caches(case["batch"], cap)
        torch.cuda.synchronize()
        s["dec"].prefill_device(emb, s["kv"], s["pad"], 512)
        s["L"] = max(lens)
        s["ids"] = _ids(case, seed, "next", case["batch"])
    return s


# --- one pass ------------------------------------------------------------------


def run(s):
    case = s["case"]
    k = case["kind"]
    if k == "audio_layer":
        x, out = s["x"], s["out"]
        rc = fmd.lib().fmd_enc_layers(s["enc"].handle, ctypes.c_void_p(x.data_ptr()), 1, case["windows"],
                                      case["t"], 0, 1, 0, ctypes.c_void_p(out.data_ptr()), 1)
        if rc:
            raise RuntimeError(fmd.lib().fmd_last_error().decode())
        return out
    if k == "audio_encode":
        return s["enc"].encode_audio(s["mel"], s["tokens"], s["mapping"], case["audios"])
    if k == "prefill":
        s["kv"].truncate(0)
        first = s["dec"].prefill_device(s["emb"], s["kv"], s["pad"], case["chunk"])
        return [first, s["dec"].decode_step(s["ids"], s["kv"], s["pad"])]
    if k == "decode_layer":
        with torch.cuda.stream(s["stream"]):
            s["x"].copy_(s["x0"])
        s["dec"].op_layer_decode(s["kv"], 0, s["x"].data_ptr(), s["pad"], case["batch"])
        return s["x"]
    if k == "logits":
        s["dec"].op_logits(s["x"].data_ptr(), case["rows"], s["out"].data_ptr())
        return s["out"]
    s["kv"].truncate(s["L"])
    return s["dec"].decode_step(s["ids"], s["kv"], s["pad"])


# --- what a pass cannot do without ---------------------------------------------

LAYER_W = 1024 * 4096 + 2048 * 1024 + 1024 * 6144 + 3072 * 1024  # a decoder layer's weights
ENC_W = 4 * 1024 * 1024 + 2 * 1024 * 4096                        # an encoder layer's weights


def work(case):
    k = case["kind"]
    if k.startswith("audio"):
        n = case["windows"] if k == "audio_layer" else case["chunks"]
        t = case["t"] if k == "audio_layer" else 1500
        layer = n * (2.0 * t * ENC_W + 4.0 * t * t * 1024)
        if k == "audio_layer":
            return {"bytes": 2.0 * ENC_W + 2 * 2.0 * n * t * 1024, "flops": layer}
        tokens, _ = _chunk_tokens(case)
        stem = n * (2.0 * 3000 * 1024 * 240 + 2.0 * 1500 * 1024 * 3072)
        rows = sum(tokens)
        return {"bytes": 2.0 * (24 * ENC_W + 1024 * 3312 + 1024 * 5120) + n * 80 * 3000 * 4.0 + rows * 2048.0,
                "flops": 24 * layer + stem + 2.0 * rows * 1024 * 5120}
    wb = 34.0 / 32.0 if case["prec"] == "int8" else 2.0
    head = case.get("vocab", 0) * 1024.0
    if k == "logits":
        return {"bytes": head * wb + case["rows"] * (2048.0 + 4.0 * case["vocab"]),
                "flops": 2.0 * case["rows"] * head}
    lens = _lens(case)
    B, keys = len(lens), float(sum(lens))
    step_kv = (keys + 2 * B) * 2 * 1024 * 2.0          # cached K and V read, the new rows written
    step_fl = 2.0 * B * LAYER_W + 4.0 * (keys + B) * 2048
    if k == "decode_layer":
        return {"bytes": LAYER_W * wb + step_kv + B * 4096.0, "flops": step_fl}
    n = case["layers"]
    step = {"bytes": n * (LAYER_W * wb + step_kv) + head * wb + 4.0 * B * case["vocab"],
            "flops": n * step_fl + 2.0 * B * head}
    if k == "decode_step":
        return step
    attn = sum(2.0 * m * (m + 1) * 2048 for m in lens)  # each query's keys, scores and values
    return {"bytes": step["bytes"] + keys * 2048.0 + n * (LAYER_W * wb + keys * 4096.0) + head * wb,
            "flops": step["flops"] + n * (2.0 * keys * LAYER_W + attn) + 2.0 * B * head}


def tolerance(case):
    # Relative 2-norm, about four times the library's own distance to the
    # 64-bit result (in brackets): the residual stream carries most of a single
    # layer's output, a whole model's logits carry every layer's roundings.
    k, bf = case["kind"], case["prec"] == "bf16"
    if k in ("audio_layer", "decode_layer"):
        return {"rel": 1.2e-2 if bf else 1.6e-3}       # (3.3e-3; 4.0e-4)
    if k == "logits":
        return {"rel": 1.2e-2 if bf else 2e-3}         # (f16: 5e-4)
    if k == "audio_encode":
        return {"rel": 7e-3}                           # (1.8e-3)
    if k == "prefill" and case["layers"] <= 2:
        return {"rel": 3e-2 if bf else 7e-3}           # (1.1e-2; 1.7e-3)
    return {"rel": 2e-2}                               # (5.4e-3)


# --- the same in 64 bits -------------------------------------------------------


def _q8_0(w):
    """Q8_0 blocks of 32 (f16 scale, int8 values) as the values they stand for."""
    x = w.float().reshape(-1, 32)
    d = x.abs().amax(1, keepdim=True) / 127.0
    q = torch.round(x * torch.where(d > 0, 1.0 / d, torch.zeros_like(d)))
    return (q.double() * d.half().double()).reshape(w.shape)


def _rms(x, g):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + 1e-6) * g


def _ln(x, g, b, eps):
    m = x.mean(-1, keepdim=True)
    v = ((x - m) ** 2).mean(-1, keepdim=True)
    return (x - m) / torch.sqrt(v + eps) * g + b


def _rope(x, pos):
    """x (n, heads, 128) at positions pos; the angles are f32, as the model's are."""
    inv = (1.0 / (1e6 ** (torch.arange(0, 128, 2, dtype=torch.float64) / 128))).float().to(DEV)
    a = (pos.float()[:, None] * inv[None]).double()
    c, s = torch.cos(a)[:, None], torch.sin(a)[:, None]
    lo, hi = x[..., :64], x[..., 64:]
    return torch.cat([lo * c - hi * s, hi * c + lo * s], -1)


def _text_layer64(cfg, prec, seed, i):
    lin = (lambda t: _q8_0(t)) if prec == "int8" else (lambda t: t.double())
    return {n.split(".", 2)[2]: lin(t) if t.ndim == 2 else t.double()
            for n, t in _text_layer(cfg, prec, seed, i).items()}


def _attend(q, k, v, first):
    """q (n, 16, 128) at key indexes first .. first + n - 1; k, v (m, 8, 128)."""
    n, m = q.shape[0], k.shape[0]
    mask = torch.arange(m, device=DEV)[None] > torch.arange(first, first + n, device=DEV)[:, None]
    out = torch.empty_like(q)
    for h in range(16):
        s = (q[:, h] @ k[:, h // 2].t()) * (128 ** -0.5)
        s.masked_fill_(mask, -math.inf)
        out[:, h] = torch.softmax(s, -1) @ v[:, h // 2]
    return out.reshape(n, 2048)


def _layer64(w, x, pos, past):
    """One decoder layer over the rows x at positions pos after `past` (K, V)."""
    n = x.shape[0]
    h = _rms(x, w["input_layernorm.weight"])
    q = _rope(_rms((h @ w["self_attn.q_proj.weight"].t()).reshape(n, 16, 128), w["self_attn.q_norm.weight"]), pos)
    k = _rope(_rms((h @ w["self_attn.k_proj.weight"].t()).reshape(n, 8, 128), w["self_attn.k_norm.weight"]), pos)
    v = (h @ w["self_attn.v_proj.weight"].t()).reshape(n, 8, 128)
    first = 0
    if past is not None:
        first = past[0].shape[0]
        k, v = torch.cat([past[0], k]), torch.cat([past[1], v])
    x = x + _attend(q, k, v, first) @ w["self_attn.o_proj.weight"].t()
    h = _rms(x, w["post_attention_layernorm.weight"])
    g, u = h @ w["mlp.gate_proj.weight"].t(), h @ w["mlp.up_proj.weight"].t()
    return x + (g * torch.sigmoid(g) * u) @ w["mlp.down_proj.weight"].t()


def _head64(cfg, prec, seed):
    top = _text_top(cfg, prec, seed)
    e = top["embed_tokens.weight"]
    return e.to(ACT[prec]).double(), _q8_0(e) if prec == "int8" else e.double(), top["norm.weight"].double()


def _model64(case, seed):
    """Logits after the prompts and after one more token, from one causal pass."""
    cfg, prec, lens = _text_config(case["layers"], case["vocab"]), case["prec"], _lens(case)
    x, pad = _prompt_rows(case, seed, lens)
    embed, head, norm = _head64(cfg, prec, seed)
    ids = _ids(case, seed, "next", case["batch"])
    rows = [torch.cat([x[b, p:].double(), embed[i][None]]) for b, (p, i) in enumerate(zip(pad, ids))]
    for i in range(case["layers"]):
        w = _text_layer64(cfg, prec, seed, i)
        rows = [_layer64(w, r, torch.arange(p, p + r.shape[0], device=DEV), None) for r, p in zip(rows, pad)]
    last = torch.stack([r[-2:] for r in rows])
    return (_rms(last, norm) @ head.t()).cpu().numpy()


def _audio_layer64(cfg, prec, seed, i, x):
    d, p = 1024, AUDIO + f"layers.{i}."

    def t(n, shape):
        return _audio_tensor(cfg, prec, seed, p + n, shape).double()

    def lin(n, h, shape):
        return h @ t(n + ".weight", shape).t() + t(n + ".bias", shape[:1])

    h = _ln(x, t("self_attn_layer_norm.weight", (d,)), t("self_attn_layer_norm.bias", (d,)), 1e-5)
    q, v = lin("self_attn.q_proj", h, (d, d)), lin("self_attn.v_proj", h, (d, d))
    k = h @ t("self_attn.k_proj.weight", (d, d)).t()
    ctx = torch.empty_like(q)
    for n in range(x.shape[0]):
        for c in (slice(64 * j, 64 * j + 64) for j in range(16)):
            ctx[n, :, c] = torch.softmax((q[n, :, c] @ k[n, :, c].t()) * 0.125, -1) @ v[n, :, c]
    x = x + lin("self_attn.out_proj", ctx, (d, d))
    h = _ln(x, t("final_layer_norm.weight", (d,)), t("final_layer_norm.bias", (d,)), 1e-5)
    h = torch.nn.functional.gelu(lin("fc1", h, (4096, d)))
    return x + lin("fc2", h, (d, 4096))


def _audio64(case, seed):
    cfg, prec = fmd.AudioConfig(encoder_layers=24), case["prec"]
    shapes = _audio_shapes(cfg)
    t = lambda n: _audio_tensor(cfg, prec, seed, n, shapes[n]).double()  # noqa: E731
    mel = _mel(case, seed).to(ACT[prec]).double()
    frames = []
    for c in range(case["chunks"]):
        # the convolutions as products over three shifted inputs
        def conv(x, name, stride):
            w = t(AUDIO + name + ".weight")
            xp = torch.nn.functional.pad(x, (1, 1))
            n = (x.shape[1] - 1) // stride + 1
            y = sum(w[:, :, j] @ xp[:, j:j + stride * (n - 1) + 1:stride] for j in range(3))
            return torch.nn.functional.gelu(y + t(AUDIO + name + ".bias")[:, None])

        h = conv(conv(mel[c], "conv1", 1), "conv2", 2).t()
        frames.append(h + t(AUDIO + "embed_positions.weight"))
    x = torch.stack(frames)
    for i in range(24):
        x = _audio_layer64(cfg, prec, seed, i, x)
    x = _ln(x, t(AUDIO + "layer_norm.weight"), t(AUDIO + "layer_norm.bias"), 1e-5)
    tokens, mapping = _chunk_tokens(case)
    out = []
    for a in range(case["audios"]):
        rows = torch.cat([x[i, :min(4 * tokens[i], 1500)] for i in range(case["chunks"]) if mapping[i] == a])
        rows = rows[:rows.shape[0] // 4 * 4].reshape(-1, 4096)
        h = rows @ t(ADAPT + "layers.0.weight").t() + t(ADAPT + "layers.0.bias")
        h = (h * torch.sigmoid(h)) @ t(ADAPT + "layers.2.weight").t() + t(ADAPT + "layers.2.bias")
        out.append(_ln(h, t(ADAPT + "layers.3.weight"), t(ADAPT + "layers.3.bias"), 1e-6))
    return out


def exact(case, seed):
    k, prec = case["kind"], case["prec"]
    if k == "audio_layer":
        cfg = fmd.AudioConfig(encoder_layers=1)
        x = _normal(seed, "hidden", (case["windows"], case["t"], 1024), ACT[prec]).double()
        return _audio_layer64(cfg, prec, seed, 0, x)
    if k == "audio_encode":
        # the embeddings come back in f16
        return [a.cpu().numpy() for a in _audio64(case, seed)]
    if k == "logits":
        cfg = _text_config(1, case["vocab"])
        _, head, norm = _head64(cfg, prec, seed)
        return _rms(_normal(seed, "hidden", (case["rows"], 1024), ACT[prec]).double(), norm) @ head.t()
    if k == "decode_layer":
        cfg, lens = _text_config(1, 2048), _lens(case)
        L = max(lens)
        w = _text_layer64(cfg, prec, seed, 0)
        K, V = _cache_rows(case, seed, L)
        x = _normal(seed, "hidden", (case["batch"], 1024), ACT[prec]).double()
        pos = torch.tensor([L], device=DEV)
        return torch.cat([_layer64(w, x[b:b + 1], pos,
                                   (K[b, :, L - n:].transpose(0, 1).double(), V[b, :, L - n:].transpose(0, 1).double()))
                          for b, n in enumerate(lens)])
    logits = _model64(case, seed)
    return [logits[:, 0], logits[:, 1]] if k == "prefill" else logits[:, 1]
