"""The work a transcription program has this library do, as measurable cases.

The library is the Qwen3-0.6B decoder of an audio transcriber (28 layers, hidden
1024, 16 / 8 heads, SwiGLU 3072, 151,936-row tied vocabulary), its Whisper-shaped
audio encoder (24 layers of 1,024, 3,000 mel frames per chunk) and the standalone
q8_0 matrix product. A program encodes its audio chunks, runs the fused prompt as
one prefill, and then decodes: one row at a time when it samples from logits, or
with drafted rows verified as one batch when it decodes greedily. Weights come as
q8_0 (the usual file), f16, f32 (the converter's default) or q4_K; the KV cache as
f32 or f16.

Kinds of cases:
  matmul   mtg_q8_mul_mat_dev: one packed q8_0 matrix times 1..16 rows on the device
  decode   mtg_append of one embedding row, then mtg_logits of its hidden row
  verify   mtg_verify: a seed and its drafts as one batch over a cached prefix
  prefill  mtg_prefill of fused prompt rows from position 0, every hidden row back
  encode   mtg_encoder_encode of one mel chunk, then mtg_encoder_adapt of its rows

The models' weights are N(0, 0.02) from a fixed seed, one model per weight type and
depth, as a program loads its model file once; prompts, caches, tokens, mel frames
and matmul operands come from the seed that prepare() is given.
"""
import ctypes
import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "moss-transcribe.cpp_amd"))

import mtg  # noqa: E402

TYPES = {"f32": mtg.TYPE_F32, "f16": mtg.TYPE_F16, "q8_0": mtg.TYPE_Q8_0, "q4_K": mtg.TYPE_Q4_K}
BITS = {"f32": 32.0, "f16": 16.0, "q8_0": 8.5, "q4_K": 4.5}
HIDDEN, HEADS, KV_HEADS, HEAD_DIM, FFN, VOCAB = 1024, 16, 8, 128, 3072, 151936
ROPE_BASE, EPS = 1e6, 1e-6
STD = 0.02
LAYER_WEIGHTS = HIDDEN * HEAD_DIM * (2 * HEADS + 2 * KV_HEADS) + 3 * HIDDEN * FFN
ENC_FFN, ENC_HEADS, MELS, MERGE = 4096, 16, 80, 4
PENALTY = 1.1


def listed():
    return [
        # a program that keeps its own graph and hands over single products, one row at a time
        dict(name="matmul_1024x1024_1row", kind="matmul", k=1024, n=1024, rows=1),
        # sampled decoding over a half-minute clip: one row per token, logits to the sampler
        dict(name="decode_q8_613", kind="decode", wtype="q8_0", kv="f32", layers=28, context=613),
        # a short clip decoded with three drafts; the caller looks at the logits too
        dict(name="verify_q8_4rows_512", kind="verify", wtype="q8_0", kv="f32", layers=28, context=512, rows=4,
             penalty=False, logits=True),
        # the benchmark's two-minute recording: seven drafts over 1,600 positions
        dict(name="verify_q8_8rows_1600", kind="verify", wtype="q8_0", kv="f32", layers=28, context=1600, rows=8,
             penalty=True, logits=False),
        # a five-minute recording, f16 cache, the widest batch
        dict(name="verify_q8_16rows_3987", kind="verify", wtype="q8_0", kv="f16", layers=28, context=3987, rows=16,
             penalty=False, logits=False),
        # an f16 model over a ten-minute recording
        dict(name="verify_f16_8rows_8000", kind="verify", wtype="f16", kv="f16", layers=28, context=8000, rows=8,
             penalty=False, logits=False),
        # the converter's default dtype over the two-minute recording
        dict(name="verify_f32_8rows_1600", kind="verify", wtype="f32", kv="f32", layers=28, context=1600, rows=8,
             penalty=False, logits=False),
        # the smallest file over the longest recording
        dict(name="verify_q4k_16rows_16384", kind="verify", wtype="q4_K", kv="f16", layers=28, context=16384, rows=16,
             penalty=False, logits=False),
        # the whole prompt of the two-minute recording
        dict(name="prefill_q8_1600", kind="prefill", wtype="q8_0", kv="f32", layers=28, rows=1600),
        # four layers of the long prompts (blocks of rows over a growing cache; the last block ragged)
        dict(name="prefill_f16_7963", kind="prefill", wtype="f16", kv="f16", layers=4, rows=7963),
        dict(name="prefill_q4k_16384", kind="prefill", wtype="q4_K", kv="f16", layers=4, rows=16384),
        # one 30-second chunk from mel frames to the decoder's audio rows
        dict(name="encode_q8_3000", kind="encode", wtype="q8_0", layers=24, frames=3000),
    ]


def draw(rng):
    """A case of the same ranges: every kind, weight type, cache type and option, sizes spread
    over their logarithm; depths of 2 to 6 layers stand for the whole models."""
    def log_int(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["matmul", "decode", "verify", "verify", "prefill", "prefill", "encode"])
    if kind == "matmul":
        return dict(kind=kind, k=64 * log_int(4, 64), n=16 * log_int(16, VOCAB // 16), rows=rng.randint(1, 16))
    wtype = rng.choice(["q8_0", "q8_0", "f16", "f32", "q4_K"])
    layers = rng.randint(2, 6)
    if kind == "encode":
        return dict(kind=kind, wtype=wtype, layers=layers, frames=log_int(200, 3000))
    kv = rng.choice(["f32", "f16"])
    if kind == "decode":
        return dict(kind=kind, wtype=wtype, kv=kv, layers=layers, context=log_int(16, 8000))
    if kind == "verify":
        return dict(kind=kind, wtype=wtype, kv=kv, layers=layers, context=log_int(16, 12000), rows=rng.randint(2, 16),
                    penalty=rng.random() < 0.5, logits=rng.random() < 0.25)
    return dict(kind=kind, wtype=wtype, kv=kv, layers=layers, rows=log_int(17, 6000))


# ------------------------------------------------------------------ weights --
def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _generator(*seed):
    g = torch.Generator(device=_device())
    g.manual_seed(hash(seed) & 0x7FFFFFFFFFFF)
    return g


def _normal(g, *shape):
    return torch.randn(*shape, generator=g, device=_device(), dtype=torch.float32)


def _pack_q8_0(w):
    n, k = w.shape
    b = w.view(n, k // 32, 32)
    d = (b.abs().amax(-1, keepdim=True) / 127.0)
    q = torch.round(b / d.clamp_min(1e-30)).clamp(-127, 127).to(torch.int8)
    out = torch.cat([d.to(torch.float16).view(torch.uint8), q.view(torch.uint8)], -1)
    return out.reshape(n, k // 32 * 34)


def _pack_q4_k(w):
    n, k = w.shape
    b = w.view(n * k // 256, 8, 32)
    low = (-b.amin(-1)).clamp_min(0)
    step = (b.amax(-1) + low) / 15.0
    d = (step.amax(-1, keepdim=True) / 63.0).to(torch.float16)
    dm = (low.amax(-1, keepdim=True) / 63.0).to(torch.float16)
    sc = torch.round(step / d.float().clamp_min(1e-12)).clamp(0, 63)
    mn = torch.round(low / dm.float().clamp_min(1e-12)).clamp(0, 63)
    q = torch.round((b + (dm.float() * mn).unsqueeze(-1)) / (d.float() * sc).clamp_min(1e-12).unsqueeze(-1))
    q = q.clamp(0, 15).to(torch.uint8)
    sc, mn = sc.to(torch.uint8), mn.to(torch.uint8)
    packed = torch.empty(b.shape[0], 12, dtype=torch.uint8, device=w.device)
    packed[:, 0:4] = sc[:, :4] | ((sc[:, 4:] >> 4) << 6)
    packed[:, 4:8] = mn[:, :4] | ((mn[:, 4:] >> 4) << 6)
    packed[:, 8:12] = (sc[:, 4:] & 15) | ((mn[:, 4:] & 15) << 4)
    qs = (q[:, 0::2] | (q[:, 1::2] << 4)).reshape(b.shape[0], 128)
    return torch.cat([d.view(torch.uint8), dm.view(torch.uint8), packed, qs], -1).reshape(n, k // 256 * 144)


def _pack(w, wtype):
    """The file's bytes of an [n][k] matrix, in host memory."""
    if wtype == "f32":
        out = w
    elif wtype == "f16":
        out = w.to(torch.float16)
    else:
        out = _pack_q8_0(w) if wtype == "q8_0" else _pack_q4_k(w)
    return np.ascontiguousarray(out.cpu().numpy()).view(np.uint8).reshape(w.shape[0], -1)


def _unpack(raw, wtype):
    """[n][k] in 64 bits from the file's bytes."""
    t = torch.from_numpy(raw).to(_device())
    n = t.shape[0]
    if wtype in ("f32", "f16"):
        return t.view(torch.float32 if wtype == "f32" else torch.float16).double()
    if wtype == "q8_0":
        t = t.view(n, -1, 34)
        d = t[:, :, :2].contiguous().view(torch.float16).double()
        return (d * t[:, :, 2:].contiguous().view(torch.int8).double()).view(n, -1)
    t = t.view(-1, 144)
    d = t[:, 0:2].contiguous().view(torch.float16).double()
    dm = t[:, 2:4].contiguous().view(torch.float16).double()
    a, b, c = t[:, 4:8], t[:, 8:12], t[:, 12:16]
    sc = torch.cat([a & 63, (c & 15) | ((a >> 6) << 4)], -1).double()
    mn = torch.cat([b & 63, (c >> 4) | ((b >> 6) << 4)], -1).double()
    qs = t[:, 16:].reshape(-1, 4, 32)
    q = torch.stack([qs & 15, qs >> 4], 2).reshape(-1, 8, 32).double()
    return ((d * sc).unsqueeze(-1) * q - (dm * mn).unsqueeze(-1)).view(n, -1)


class _File:
    """Base of the models held in host memory, as a mapped model file."""

    def matrix(self, g, n, k):
        raw = _pack(_normal(g, n, k) * STD, self.wtype)
        return raw, raw.ctypes.data

    def vector(self, g, n, std, mean=0.0):
        v = (_normal(g, n) * std + mean).cpu().numpy()
        return v, v.ctypes.data


class DecoderFile(_File):
    NAMES = (("attn_norm", "gain", HIDDEN), ("attn_q_norm", "gain", HEAD_DIM), ("attn_k_norm", "gain", HEAD_DIM),
             ("ffn_norm", "gain", HIDDEN), ("attn_q", HEADS * HEAD_DIM, HIDDEN), ("attn_k", KV_HEADS * HEAD_DIM, HIDDEN),
             ("attn_v", KV_HEADS * HEAD_DIM, HIDDEN), ("attn_o", HIDDEN, HEADS * HEAD_DIM), ("ffn_gate", FFN, HIDDEN),
             ("ffn_up", FFN, HIDDEN), ("ffn_down", HIDDEN, FFN))

    def __init__(self, wtype, layers):
        self.wtype, self.layers = wtype, []
        self.hp = mtg.make_hparams(n_layers=layers)
        g = _generator(1, layers)
        self.embd, embd = self.matrix(g, VOCAB, HIDDEN)
        self.out_norm, out_norm = self.vector(g, HIDDEN, 0.05, 1.0)
        self.table = (mtg.LayerTensors * layers)()
        for i in range(layers):
            kept = {}
            for name, n, k in self.NAMES:
                kept[name], at = self.vector(g, k, 0.05, 1.0) if n == "gain" else self.matrix(g, n, k)
                setattr(self.table[i], name, at)
            self.layers.append(kept)
        self._desc = mtg.ModelDesc(self.hp, TYPES[wtype], embd, out_norm, self.table)
        self.desc = ctypes.pointer(self._desc)


class EncoderFile(_File):
    def __init__(self, wtype, layers, frames):
        self.wtype, self.layers = wtype, []
        self.hp = mtg.EncoderHparams(**dict(mtg.ENCODER_DEFAULTS, n_layers=layers, n_frames=frames))
        self.rows = (frames - 1) // 2 + 1
        g = _generator(2, layers, frames)
        self.kept = {}
        d = mtg.EncoderDesc()
        d.hp, d.weight_type = self.hp, TYPES[wtype]
        for name, n, std, mean in (("conv1_w", HIDDEN * MELS * 3, STD, 0), ("conv1_b", HIDDEN, STD, 0),
                                   ("conv2_w", HIDDEN * HIDDEN * 3, STD, 0), ("conv2_b", HIDDEN, STD, 0),
                                   ("pos_embd", self.rows * HIDDEN, 0.2, 0), ("ln_post_w", HIDDEN, 0.05, 1),
                                   ("ln_post_b", HIDDEN, 0.05, 0), ("ad_fc1_b", HIDDEN, STD, 0),
                                   ("ad_fc2_b", HIDDEN, STD, 0), ("ad_ln_w", HIDDEN, 0.05, 1),
                                   ("ad_ln_b", HIDDEN, 0.05, 0)):
            self.kept[name], at = self.vector(g, n, std, mean)
            setattr(d, name, at)
        for name, n, k in (("ad_fc1_w", HIDDEN, HIDDEN * MERGE), ("ad_fc2_w", HIDDEN, HIDDEN)):
            self.kept[name], at = self.matrix(g, n, k)
            setattr(d, name, at)
        self.table = (mtg.EncoderLayer * layers)()
        for i in range(layers):
            kept = {}
            for name, n, k in (("q_w", HIDDEN, HIDDEN), ("k_w", HIDDEN, HIDDEN), ("v_w", HIDDEN, HIDDEN),
                               ("o_w", HIDDEN, HIDDEN), ("fc1_w", ENC_FFN, HIDDEN), ("fc2_w", HIDDEN, ENC_FFN)):
                kept[name], at = self.matrix(g, n, k)
                setattr(self.table[i], name, at)
            for name, n, std, mean in (("attn_ln_w", HIDDEN, 0.05, 1), ("attn_ln_b", HIDDEN, 0.05, 0),
                                       ("q_b", HIDDEN, STD, 0), ("v_b", HIDDEN, STD, 0), ("o_b", HIDDEN, STD, 0),
                                       ("ffn_ln_w", HIDDEN, 0.05, 1), ("ffn_ln_b", HIDDEN, 0.05, 0),
                                       ("fc1_b", ENC_FFN, STD, 0), ("fc2_b", HIDDEN, STD, 0)):
                kept[name], at = self.vector(g, n, std, mean)
                setattr(self.table[i], name, at)
            self.layers.append(kept)
        d.layers = self.table
        self.desc = d


_files = {}  # the model files this process has opened; the largest are dropped first


def _file(case):
    key = ("encoder", case["wtype"], case["layers"], case["frames"]) if case["kind"] == "encode" else \
        ("decoder", case["wtype"], case["layers"])
    if key not in _files:
        while len(_files) >= 3:
            _files.pop(next(iter(_files)))
        _files[key] = EncoderFile(*key[1:]) if case["kind"] == "encode" else DecoderFile(*key[1:])
    return _files[key]


# ------------------------------------------------------------------- inputs --
def _tokens(case, seed):
    r = np.random.default_rng((seed, 12))
    return r.integers(0, VOCAB, case["rows"]).astype(np.int32), r.integers(0, VOCAB, 150).astype(np.int32)


def _rows(case, seed):
    """Fused prompt rows of the embeddings' size (for decode, the row to append last)."""
    n = case["rows"] if case["kind"] == "prefill" else case["context"] + (case["kind"] == "decode")
    return (_normal(_generator(seed, 13), n, HIDDEN) * STD).cpu().numpy()


def _mel(case, seed):
    return (_normal(_generator(seed, 14), MELS, case["frames"]) * 0.5).cpu().numpy()


def _operands(case, seed):
    g = _generator(seed, 15)
    return _pack(_normal(g, case["n"], case["k"]) * STD, "q8_0"), _normal(g, case["rows"], case["k"])


class _Matmul:
    def __init__(self, case, seed):
        raw, self.x = _operands(case, seed)
        self.rows = case["rows"]
        self.y = torch.empty(case["rows"], case["n"], dtype=torch.float32, device="cuda")
        self.w = ctypes.c_void_p()
        self.lib = mtg.lib()
        rc = self.lib.mtg_q8_pack(raw.ctypes.data, case["k"], case["n"], ctypes.byref(self.w))
        if rc:
            raise mtg.MtgError(rc, "pack")

    def __del__(self):
        if getattr(self, "w", None):
            self.lib.mtg_q8_free(self.w)


class _State:
    pass


def prepare(case, seed):
    kind = case["kind"]
    if kind == "matmul":
        s = _Matmul(case, seed)
        s.kind = kind
        torch.cuda.synchronize()
        return s
    s = _State()
    s.kind, f = kind, _file(case)
    if kind == "encode":
        s.enc, s.mel = mtg.Encoder(f), _mel(case, seed)
        return s
    if kind == "prefill":
        s.dec, s.rows = mtg.Decoder(f, case["rows"] + 64, TYPES[case["kv"]]), _rows(case, seed)
        return s
    s.context = case["context"]
    s.dec = mtg.Decoder(f, case["context"] + 64, TYPES[case["kv"]])
    rows = _rows(case, seed)
    s.dec.prefill(rows[:s.context], want_hidden=False)
    if kind == "decode":
        s.row = rows[s.context:]
    else:
        s.tokens, history = _tokens(case, seed)
        s.history = history if case["penalty"] else ()
        s.penalty, s.logits = (PENALTY if case["penalty"] else 1.0), case["logits"]
    return s


def run(s):
    if s.kind == "matmul":
        rc = s.lib.mtg_q8_mul_mat_dev(s.w, s.x.data_ptr(), s.rows, s.y.data_ptr())
        if rc:
            raise mtg.MtgError(rc, "mul_mat")
        return s.y
    if s.kind == "encode":
        rows = s.enc.encode(s.mel)
        return {"rows": rows, "adapted": s.enc.adapt(len(rows))}
    if s.kind == "prefill":
        return s.dec.prefill(s.rows)
    s.dec.rewind(s.context)
    if s.kind == "decode":
        hidden = s.dec.append(s.row)
        return {"hidden": hidden, "logits": s.dec.logits(hidden)}
    choice, n_match, hidden, logits = s.dec.verify(s.tokens, s.history, s.penalty, want_hidden=True, want_logits=s.logits)
    out = {"choice": choice, "n_match": n_match, "hidden": hidden}
    if s.logits:
        out["logits"] = logits
    return out


def work(case):
    kind = case["kind"]
    if kind == "matmul":
        k, n, t = case["k"], case["n"], case["rows"]
        return {"bytes": n * k * 34 / 32 + 4 * t * (k + n), "flops": 2.0 * t * n * k}
    per = BITS[case["wtype"]] / 8
    if kind == "encode":
        frames, layers = case["frames"], case["layers"]
        r = (frames - 1) // 2 + 1
        layer = 4 * HIDDEN * HIDDEN + 2 * HIDDEN * ENC_FFN
        adaptor = HIDDEN * HIDDEN * (MERGE + 1)
        flops = 2.0 * frames * HIDDEN * MELS * 3 + 2.0 * r * HIDDEN * HIDDEN * 3
        flops += layers * (2.0 * r * layer + 4.0 * r * r * HIDDEN) + 2.0 * (r // MERGE) * adaptor
        weights = (layers * layer + adaptor) * per + 4 * (HIDDEN * 3 * (MELS + HIDDEN) + r * HIDDEN)
        return {"bytes": weights + 4 * (MELS * frames + r * HIDDEN + r // MERGE * HIDDEN), "flops": flops}
    layers, kvb = case["layers"], 4 if case["kv"] == "f32" else 2
    pos = layers * 2 * KV_HEADS * HEAD_DIM * kvb
    head = HEADS * HEAD_DIM
    if kind == "prefill":
        s = case["rows"]
        flops = layers * (2.0 * s * LAYER_WEIGHTS + 4.0 * head * s * (s + 1) / 2)
        return {"bytes": layers * LAYER_WEIGHTS * per + s * pos + 8 * s * HIDDEN, "flops": flops}
    t, p = case.get("rows", 1), case["context"]
    flops = 2.0 * t * (layers * LAYER_WEIGHTS + VOCAB * HIDDEN) + layers * 4.0 * t * (p + t) * head
    out = 4 * t * HIDDEN + (4 * t * VOCAB if kind == "decode" or case["logits"] else 0)
    return {"bytes": (layers * LAYER_WEIGHTS + VOCAB * HIDDEN) * per + (p + 2 * t) * pos + out, "flops": flops}


def tolerance(case):
    if case["kind"] == "matmul":  # exact block sums, 32-bit sums over the blocks
        return {"rel": 1e-6}
    # every product rounds its input to the weights' activation type again (8 bits for q8_0 and
    # q4_K, 16 for f16): a difference in a 32-bit sum becomes a step of that rounding. Against
    # exact() the hidden rows are 1.2e-2 .. 3e-2 (q8_0, q4_K), 6e-4 .. 9e-4 (f16) and 1e-5 (f32;
    # 2e-4 with an f16 cache) away.
    rel = {"q8_0": 3e-2, "q4_K": 3e-2, "f16": 3e-3, "f32": 1e-4}[case["wtype"]]
    if case.get("kv") == "f16":
        rel = max(rel, 1e-3)
    return {"rel": rel, "differ": 0.01}


# ------------------------------------------------------------ in 64 bits --
def _rms(x, gain):
    g = torch.from_numpy(gain).to(x.device).double()
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS) * g


def _rope(x, pos):
    i = torch.arange(HEAD_DIM // 2, device=x.device, dtype=torch.float64)
    a = pos.double().unsqueeze(-1) * ROPE_BASE ** (-2.0 * i / HEAD_DIM)
    c, s = torch.cos(a), torch.sin(a)
    x0, x1 = x[..., :HEAD_DIM // 2], x[..., HEAD_DIM // 2:]
    return torch.cat([x0 * c - x1 * s, x0 * s + x1 * c], -1)


def _act(x, wtype):
    """x as the products take it: every product is defined on the weights' activation type (32-bit
    rows, f16 rows, or blocks of 8-bit codes with one scale per 32 or 256 values)."""
    if wtype == "f32":
        return x
    if wtype == "f16":
        return x.to(torch.float16).double()
    b = x.float().view(x.shape[0], -1, 32 if wtype == "q8_0" else 256)
    top = b.abs().amax(-1, keepdim=True)
    if wtype == "q8_0":
        codes = torch.round(b * torch.where(top > 0, 127.0 / top, torch.zeros_like(top)))
        return (codes.double() * (top / 127.0).to(torch.float16).double()).view(x.shape)
    first = b.abs().argmax(-1, keepdim=True)  # the signed largest value takes the code -127
    inv = torch.where(top > 0, -127.0 / b.gather(-1, first), torch.zeros_like(top))
    codes = torch.round(b * inv).clamp_max(127)
    return (codes.double() * torch.where(top > 0, 1.0 / inv, inv).double()).view(x.shape)


def _attend(q, k, v):
    """Causal attention: q [heads][t][d], k / v [kv heads][t][d] -> [t][heads * d]."""
    out = torch.empty_like(q)
    t, group = q.shape[1], q.shape[0] // k.shape[0]
    keys = torch.arange(k.shape[1], device=q.device)
    for h in range(q.shape[0]):
        for r0 in range(0, t, 4096):
            r1 = min(t, r0 + 4096)
            w = q[h, r0:r1] @ k[h // group, :r1].T / math.sqrt(q.shape[2])
            w.masked_fill_(keys[:r1] > torch.arange(r0, r1, device=q.device).unsqueeze(1), -math.inf)
            out[h, r0:r1] = torch.softmax(w, -1) @ v[h // group, :r1]
    return out.transpose(0, 1).reshape(t, -1)


def _decoder(f, x, half):
    """Final-normed hidden rows of x [t][hidden] at positions 0 .. t - 1."""
    t = x.shape[0]
    pos = torch.arange(t, device=x.device)
    for y in f.layers:
        w = {n: _unpack(y[n], f.wtype) for n in ("attn_q", "attn_k", "attn_v", "attn_o", "ffn_gate", "ffn_up", "ffn_down")}
        a = _act(_rms(x, y["attn_norm"]), f.wtype)
        q = (a @ w["attn_q"].T).view(t, HEADS, HEAD_DIM).transpose(0, 1)
        k = (a @ w["attn_k"].T).view(t, KV_HEADS, HEAD_DIM).transpose(0, 1)
        v = (a @ w["attn_v"].T).view(t, KV_HEADS, HEAD_DIM).transpose(0, 1)
        q, k = _rope(_rms(q, y["attn_q_norm"]), pos), _rope(_rms(k, y["attn_k_norm"]), pos)
        if half:  # an f16 cache, whose scores take f16 queries
            q, k, v = (z.to(torch.float16).double() for z in (q, k, v))
        x = x + _act(_attend(q.contiguous(), k, v), f.wtype) @ w["attn_o"].T
        a = _act(_rms(x, y["ffn_norm"]), f.wtype)
        a = torch.nn.functional.silu(a @ w["ffn_gate"].T) * (a @ w["ffn_up"].T)
        x = x + _act(a, f.wtype) @ w["ffn_down"].T
    return _rms(x, f.out_norm)


def _ln(x, w, b, eps):
    dev = x.device
    m = x - x.mean(-1, keepdim=True)
    y = m / torch.sqrt((m * m).mean(-1, keepdim=True) + eps)
    return y * torch.from_numpy(w).to(dev).double() + torch.from_numpy(b).to(dev).double()


def _exact_encode(case, seed):
    f, dev = _file(case), _device()
    t = lambda name, *shape: torch.from_numpy(f.kept[name]).to(dev).double().view(*shape)  # noqa: E731
    gelu = lambda x: 0.5 * x * (1 + torch.erf(x / math.sqrt(2.0)))  # noqa: E731

    def conv(x, w, b, stride):  # [channels][length], kernel 3, pad 1
        p = torch.nn.functional.pad(x, (1, 1)).unfold(1, 3, stride)  # [c][out][3]
        return (w.reshape(w.shape[0], -1) @ p.permute(0, 2, 1).reshape(-1, p.shape[1])) + b.unsqueeze(1)

    x = torch.from_numpy(_mel(case, seed)).to(dev).double()
    x = gelu(conv(x, t("conv1_w", HIDDEN, MELS, 3), t("conv1_b", HIDDEN), 1))
    x = gelu(conv(x, t("conv2_w", HIDDEN, HIDDEN, 3), t("conv2_b", HIDDEN), 2)).T + t("pos_embd", f.rows, HIDDEN)
    for y in f.layers:
        m = lambda a, w, b=None: _act(a, f.wtype) @ _unpack(y[w], f.wtype).T + (torch.from_numpy(y[b]).to(dev).double() if b else 0)  # noqa: E731,B023
        a = _ln(x, y["attn_ln_w"], y["attn_ln_b"], 1e-5)
        heads = lambda z: z.view(f.rows, ENC_HEADS, -1).transpose(0, 1)  # noqa: E731
        q, k, v = heads(m(a, "q_w", "q_b")), heads(m(a, "k_w")), heads(m(a, "v_w", "v_b"))
        z = torch.stack([torch.softmax(q[h] @ k[h].T / 8.0, -1) @ v[h] for h in range(ENC_HEADS)], 1)
        x = x + m(z.reshape(f.rows, HIDDEN), "o_w", "o_b")
        a = _ln(x, y["ffn_ln_w"], y["ffn_ln_b"], 1e-5)
        x = x + m(gelu(m(a, "fc1_w", "fc1_b")), "fc2_w", "fc2_b")
    rows = _ln(x, f.kept["ln_post_w"], f.kept["ln_post_b"], 1e-5)
    n = f.rows // MERGE
    a = _act(rows[:n * MERGE].reshape(n, MERGE * HIDDEN), f.wtype) @ _unpack(f.kept["ad_fc1_w"], f.wtype).T
    a = torch.nn.functional.silu(a + t("ad_fc1_b", HIDDEN))
    a = _act(a, f.wtype) @ _unpack(f.kept["ad_fc2_w"], f.wtype).T + t("ad_fc2_b", HIDDEN)
    return {"rows": rows, "adapted": _ln(a, f.kept["ad_ln_w"], f.kept["ad_ln_b"], EPS)}


def exact(case, seed):
    kind, dev = case["kind"], _device()
    if kind == "encode":
        return _exact_encode(case, seed)
    if kind == "matmul":
        raw, x = _operands(case, seed)
        x = _act(x, "q8_0")
        out = torch.empty(x.shape[0], case["n"], dtype=torch.float64, device=dev)
        for n0 in range(0, case["n"], 16384):
            out[:, n0:n0 + 16384] = x @ _unpack(raw[n0:n0 + 16384], "q8_0").T
        return out
    f, half = _file(case), case["kv"] == "f16"
    x = torch.from_numpy(_rows(case, seed)).to(dev).double()
    if kind == "verify":
        x = torch.cat([x, _unpack(f.embd[_tokens(case, seed)[0]], f.wtype)])
    hidden = _decoder(f, x, half)
    if kind == "prefill":
        return hidden
    hidden = hidden[case["context"]:]
    out = {"hidden": hidden}
    if kind == "decode" or case["logits"]:
        a = _act(hidden, f.wtype)
        out["logits"] = torch.cat([a @ _unpack(f.embd[n:n + 16384], f.wtype).T for n in range(0, VOCAB, 16384)], 1)
    if kind == "verify":
        out.update(choice=None, n_match=None)
    return out
