"""Timing cases: the calls a LoRA training run over a frozen GGUF model makes, at the sizes it makes them.

Kinds: ``linear`` (one adapted projection, forward and / or backward, device pointers), ``frozen`` (a weight
without an adapter), ``host`` (``Linear`` on host arrays, the drop-in call of a CPU trainer), ``loss`` (final
norm, LM head and cross-entropy of a number of targets) and ``model`` (decoder blocks or a whole decoder,
plain or as a packed batch).  Shapes are those of the synthetic presets (Qwen3-0.6B, Qwen3-4B, Llama-3-8B),
formats the GGUF ones and the trainer's own f32-scaled Q8_0.

Weights are N(0, 0.02) in valid blocks of their format.  Activations are N(0, 1) with a few large channels, as
a decoder's hidden states have; gradients span orders of magnitude from token to token.
"""
import ctypes
import math

import numpy as np
import torch
import torch.utils.checkpoint

import rust_trainer_amd as rt
from rust_trainer_amd import _ffi
from rust_trainer_amd import gguf as G
from rust_trainer_amd.head import head_d
from rust_trainer_amd.packing import Packed

DEV = "cuda:0"
FMT = {"q4_0": 2, "q8_0": 8, "q4_k": 12, "q6_k": 14, "tq8_0": 264}
ROW_BYTES = {"q4_0": (32, 18), "q8_0": (32, 34), "q4_k": (256, 144), "q6_k": (256, 210), "tq8_0": (32, 36)}
EPS = 1e-6

# decoder shapes: arch, hidden, heads, kv heads, head dim, ff, RoPE base, vocabulary, format of q .. up, of down, of the embedding
SHAPES = {
    "0.6b": ("qwen3", 1024, 16, 8, 128, 3072, 1e6, 151936, "q4_0", "q4_0", "q4_0"),
    "4b": ("qwen3", 2560, 32, 8, 128, 9728, 1e6, 8192, "q4_k", "q6_k", "q6_k"),
    "8b": ("llama", 4096, 32, 8, 128, 14336, 5e5, 8192, "q8_0", "q8_0", "q8_0"),
}


def listed():
    return [
        # one token through an attention output projection: the smallest call there is, all latency
        {"name": "token_o_q4_0", "kind": "linear", "fmt": "q4_0", "n": 1024, "k": 2048, "t": 1, "r": 16, "dir": "fwd"},
        # one token's logits: the whole vocabulary matrix read once
        {"name": "token_logits_q6_k", "kind": "frozen", "fmt": "q6_k", "n": 151936, "k": 1024, "t": 1, "dir": "fwd"},
        # a training example of one sentence through a wide gate projection, a ragged number of tokens
        {"name": "sentence_gate_q4_k", "kind": "linear", "fmt": "q4_k", "n": 9728, "k": 2560, "t": 37, "r": 16, "dir": "both"},
        # a short sequence through the gate projection of a small model, the size a chat example has
        {"name": "chat_gate_q4_0", "kind": "linear", "fmt": "q4_0", "n": 3072, "k": 1024, "t": 256, "r": 16, "dir": "both"},
        # the same call on host arrays, as a trainer that keeps its tensors on the CPU makes it
        {"name": "chat_gate_host_q4_0", "kind": "host", "fmt": "q4_0", "n": 3072, "k": 1024, "t": 256, "r": 16, "dir": "both"},
        # a model loaded from float weights (f32 block scales, f32 activations)
        {"name": "native_q_tq8_0", "kind": "linear", "fmt": "tq8_0", "n": 2048, "k": 1024, "t": 300, "r": 8, "dir": "both"},
        # a long document, not a multiple of any tile, through a down projection
        {"name": "document_down_q6_k", "kind": "linear", "fmt": "q6_k", "n": 2560, "k": 9728, "t": 1001, "r": 16, "dir": "both"},
        # a full context through the widest projection, a large adapter
        {"name": "context_gate_q8_0", "kind": "linear", "fmt": "q8_0", "n": 14336, "k": 4096, "t": 2048, "r": 64, "dir": "both"},
        # loss and gradient of a short answer
        {"name": "answer_loss_q6_k", "kind": "loss", "fmt": "q6_k", "n": 151936, "k": 1024, "t": 60, "targets": 12},
        # loss and gradient of a long answer
        {"name": "long_loss_q4_0", "kind": "loss", "fmt": "q4_0", "n": 151936, "k": 1024, "t": 512, "targets": 256},
        # two decoder blocks over a packed batch: eight examples that share their prompt, forward and backward
        {"name": "packed_blocks_4b", "kind": "model", "shape": "4b", "layers": 2, "t": 6792, "packed": 8, "shared": 200,
         "targets": 2400, "r": 16, "train": True},
        # a whole training step of a small decoder
        {"name": "step_0.6b", "kind": "model", "shape": "0.6b", "layers": 28, "t": 512, "packed": 0, "shared": 0,
         "targets": 256, "r": 16, "train": True},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("linear", "linear", "linear", "linear", "frozen", "loss", "host", "model", "model"))
    if kind == "model":
        # 1 to 4 blocks of one of the decoders over 40 to 3000 tokens, packed or plain, trained or scored
        packed = rng.choice((0, 0, 3, 6))
        t = _log(rng, 40, 3000)
        c = {"kind": "model", "shape": rng.choice(("0.6b", "4b", "8b")), "layers": rng.randint(1, 4), "t": t, "packed": packed,
             "shared": t // 6 if packed else 0, "targets": max(1, t // rng.choice((2, 3, 7))), "r": rng.choice((8, 16, 32)),
             "train": rng.random() < 0.75}
        if c["shape"] == "8b":
            c.update(layers=min(c["layers"], 2), t=min(t, 2400), targets=min(c["targets"], 800), shared=min(c["shared"], 400))
        return c
    fmt = rng.choice(("q4_0", "q8_0", "q4_k", "q6_k", "q4_0", "q8_0", "q4_k", "q6_k", "tq8_0"))
    unit = 256 if fmt in ("q4_k", "q6_k") else 32
    if kind == "loss":
        if fmt == "tq8_0":
            fmt, unit = "q8_0", 32
        n, k = _log(rng, 20000, 152000), unit * (_log(rng, 768, 2560) // unit)
        m = _log(rng, 1, 700)
        return {"kind": "loss", "fmt": fmt, "n": n, "k": k, "t": m + _log(rng, 1, 500), "targets": m}
    if kind == "frozen":
        if fmt == "tq8_0":
            fmt, unit = "q4_0", 32
        return {"kind": "frozen", "fmt": fmt, "n": _log(rng, 20000, 152000), "k": unit * (_log(rng, 768, 2560) // unit),
                "t": _log(rng, 1, 300), "dir": rng.choice(("fwd", "bwd"))}
    big = 14336 if fmt != "tq8_0" else 4096
    n, k = _log(rng, 512, big), unit * max(1, _log(rng, 512, big) // unit)
    t = _log(rng, 1, 4096 if kind == "linear" and fmt != "tq8_0" else 1024)
    return {"kind": kind, "fmt": fmt, "n": n, "k": k, "t": t, "r": rng.choice((4, 8, 16, 32, 64)),
            "dir": "both" if kind == "host" else rng.choice(("fwd", "bwd", "both"))}


# ------------------------------------------------------------------ blocks of the weight formats
def _gen(seed, part):
    return torch.Generator(device=DEV).manual_seed(seed * 1000003 + part)


def _weights(n, k, seed, part):
    return torch.randn(n, k, device=DEV, generator=_gen(seed, part)) * 0.02


def _half_bytes(d):
    return d.to(torch.float16).contiguous().view(torch.uint8).reshape(d.numel(), 2)


def _q4_0(w):
    x = w.reshape(-1, 32)
    mx = x.gather(1, x.abs().argmax(1, keepdim=True))
    d = mx / torch.full_like(mx, -8.0)
    q = (x * torch.where(d != 0, 1.0 / d, torch.zeros_like(d)) + 8.5).to(torch.int32).clamp(0, 15).to(torch.uint8)
    return torch.cat([_half_bytes(d), q[:, :16] | (q[:, 16:] << 4)], 1)


def _q8_0(w):
    x = w.reshape(-1, 32)
    a = x.abs().amax(1, keepdim=True)
    d = a / torch.full_like(a, 127.0)
    v = x * torch.where(d != 0, 1.0 / d, torch.zeros_like(d))
    q = (v.sign() * (v.abs() + 0.5).floor()).clamp(-127, 127).to(torch.int8)
    return torch.cat([_half_bytes(d), q.view(torch.uint8)], 1)


def _q4_k(w):
    x = w.reshape(-1, 8, 32)
    low, high = x.amin(2).clamp(max=0), x.amax(2)
    scale, mins = (high - low) / 15.0, -low
    dh, mh = (scale.amax(1) / 63.0).to(torch.float16), (mins.amax(1) / 63.0).to(torch.float16)
    d, m = dh.float().clamp(min=1e-12)[:, None], mh.float().clamp(min=1e-12)[:, None]
    sc, mn = (scale / d).round().clamp(0, 63), (mins / m).round().clamp(0, 63)
    es, em = (d * sc).clamp(min=1e-12)[:, :, None], (m * mn)[:, :, None]
    q = ((x + em) / es).round().clamp(0, 15).to(torch.uint8).reshape(-1, 4, 2, 32)
    sc, mn = sc.to(torch.uint8), mn.to(torch.uint8)
    return torch.cat([_half_bytes(dh), _half_bytes(mh), (sc[:, :4] & 63) | ((sc[:, 4:] >> 4) << 6),
                      (mn[:, :4] & 63) | ((mn[:, 4:] >> 4) << 6), (sc[:, 4:] & 15) | ((mn[:, 4:] & 15) << 4),
                      (q[:, :, 0] | (q[:, :, 1] << 4)).reshape(-1, 128)], 1)


def _q6_k(w):
    x = w.reshape(-1, 16, 16)
    s = x.gather(2, x.abs().argmax(2, keepdim=True))[:, :, 0] / -32.0
    top = s.gather(1, s.abs().argmax(1, keepdim=True))
    inv = torch.where(top != 0, -128.0 / top, torch.zeros_like(top))
    dh = torch.where(inv != 0, 1.0 / inv, torch.zeros_like(inv)).to(torch.float16)
    sc = (inv * s).round().clamp(-128, 127)
    es = (dh.float() * sc)[:, :, None]
    q = torch.where(es != 0, x / torch.where(es != 0, es, torch.ones_like(es)), torch.zeros_like(x)).round().clamp(-32, 31)
    q = (q + 32).to(torch.uint8).reshape(-1, 2, 4, 32)
    low = torch.cat([(q[:, :, 0] & 15) | ((q[:, :, 2] & 15) << 4), (q[:, :, 1] & 15) | ((q[:, :, 3] & 15) << 4)], 2)
    top2 = (q[:, :, 0] >> 4) | ((q[:, :, 1] >> 4) << 2) | ((q[:, :, 2] >> 4) << 4) | ((q[:, :, 3] >> 4) << 6)
    return torch.cat([low.reshape(-1, 128), top2.reshape(-1, 64), sc.to(torch.int8).view(torch.uint8), _half_bytes(dh)], 1)


def _tq8_0(w):
    """(f32 scales, int8 codes) of the trainer's own 8-bit storage."""
    x = w.reshape(-1, 32)
    a = x.abs().amax(1, keepdim=True)
    d = a / torch.full_like(a, 127.0)
    v = x * torch.where(d != 0, 1.0 / d, torch.zeros_like(d))
    return d, (v.sign() * (v.abs() + 0.5).floor()).clamp(-127, 127).to(torch.int8)


def _blocks(fmt, w):
    """The packed bytes of a weight, as a loader has them in host memory."""
    if fmt == "tq8_0":
        d, q = _tq8_0(w)
        return np.concatenate([d.cpu().numpy().reshape(-1).view(np.uint8), q.cpu().numpy().reshape(-1).view(np.uint8)])
    if fmt == "f32":
        return w.cpu().numpy().reshape(-1).view(np.uint8)
    return {"q4_0": _q4_0, "q8_0": _q8_0, "q4_k": _q4_k, "q6_k": _q6_k}[fmt](w).cpu().numpy().reshape(-1)


def _halves(b):
    return b.contiguous().view(torch.float16).double()


def _decode(fmt, w):
    """The values that the blocks of ``w`` hold, in 64 bits (``[n, k]``)."""
    n, k = w.shape
    if fmt == "tq8_0":
        d, q = _tq8_0(w)
        return (d.double() * q.double()).reshape(n, k)
    b = {"q4_0": _q4_0, "q8_0": _q8_0, "q4_k": _q4_k, "q6_k": _q6_k}[fmt](w)
    if fmt == "q4_0":
        q = torch.cat([b[:, 2:] & 15, b[:, 2:] >> 4], 1).double() - 8
        return (_halves(b[:, :2]) * q).reshape(n, k)
    if fmt == "q8_0":
        return (_halves(b[:, :2]) * b[:, 2:].contiguous().view(torch.int8).double()).reshape(n, k)
    if fmt == "q4_k":
        d, m = _halves(b[:, 0:2]), _halves(b[:, 2:4])
        s = b[:, 4:16]
        sc = torch.cat([s[:, 0:4] & 63, (s[:, 8:12] & 15) | ((s[:, 0:4] >> 6) << 4)], 1).double()
        mn = torch.cat([s[:, 4:8] & 63, (s[:, 8:12] >> 4) | ((s[:, 4:8] >> 6) << 4)], 1).double()
        q = b[:, 16:].reshape(-1, 4, 1, 32)
        q = torch.cat([q & 15, q >> 4], 2).reshape(-1, 8, 32).double()
        return ((d * sc)[:, :, None] * q - (m * mn)[:, :, None]).reshape(n, k)
    low, top, sc, d = b[:, :128].reshape(-1, 2, 64), b[:, 128:192].reshape(-1, 2, 32), b[:, 192:208], b[:, 208:210]
    q = torch.stack([(low[:, :, :32] & 15) | ((top & 3) << 4), (low[:, :, 32:] & 15) | (((top >> 2) & 3) << 4),
                     (low[:, :, :32] >> 4) | (((top >> 4) & 3) << 4), (low[:, :, 32:] >> 4) | ((top >> 6) << 4)], 2)
    q = q.double().reshape(-1, 16, 16) - 32
    return ((_halves(d) * sc.contiguous().view(torch.int8).double())[:, :, None] * q).reshape(n, k)


def _codes(fmt, x):
    """What a quantised projection multiplies its weight with: the activation's 8-bit blocks, in 64 bits."""
    if fmt == "tq8_0":
        return x.double()
    x = x.float()
    if fmt in ("q4_0", "q8_0"):
        b = x.reshape(-1, 32)
        a = b.abs().amax(1, keepdim=True)
        d = a / torch.full_like(a, 127.0)
        v = (b * torch.where(d != 0, torch.ones_like(d) / d, torch.zeros_like(d))).double()
        q = v.sign() * (v.abs() + 0.5).floor()
        return (q * d.to(torch.float16).double()).reshape(x.shape)
    b = x.reshape(-1, 256)
    top = b.gather(1, b.abs().argmax(1, keepdim=True))
    inv = torch.where(top != 0, torch.full_like(top, -127.0) / top, torch.zeros_like(top))
    d = torch.where(inv != 0, torch.ones_like(inv) / inv, torch.zeros_like(inv))
    return ((inv * b).round().clamp(max=127).double() * d.double()).reshape(x.shape)


# ------------------------------------------------------------------ inputs
def _activations(t, k, seed, part):
    g = _gen(seed, part)
    x = torch.randn(t, k, device=DEV, generator=g)
    big = torch.randint(0, k, (max(1, k // 256),), device=DEV, generator=g)
    x[:, big] *= 12.0
    return x


def _gradients(t, n, seed, part):
    g = _gen(seed, part)
    return torch.randn(t, n, device=DEV, generator=g) * torch.exp(1.5 * torch.randn(t, 1, device=DEV, generator=g)) * 1e-3


def _adapter(n, k, r, seed, part):
    g = _gen(seed, part)
    a = (torch.rand(r, k, device=DEV, generator=g) * 2 - 1) / math.sqrt(k)
    return a, torch.randn(n, r, device=DEV, generator=g) * 0.01


def _linear_inputs(c, seed):
    x, dy = _activations(c["t"], c["k"], seed, 2), _gradients(c["t"], c["n"], seed, 3)
    a, b = _adapter(c["n"], c["k"], c["r"], seed, 4) if c.get("r") else (None, None)
    return x, dy, a, b


def _loss_inputs(c, seed):
    g = _gen(seed, 5)
    x = _activations(c["t"], c["k"], seed, 2)
    norm = 1 + 0.1 * torch.randn(c["k"], device=DEV, generator=g)
    m = c["targets"]
    pos = torch.arange(c["t"] - m, c["t"], device=DEV, dtype=torch.int32)  # the answer ends the sequence
    tok = torch.randint(0, c["n"], (m,), device=DEV, generator=g).to(torch.int32)
    wts = (0.5 + torch.rand(m, device=DEV, generator=g)) / m
    return x, norm, pos, tok, wts


# the linears of a block, in the order in which a model numbers its adapters
def _linears(shape):
    arch, d, nh, nkv, hd, ff, base, vocab, f1, f2, f3 = SHAPES[shape]
    return [("attn_q", nh * hd, d, f1), ("attn_k", nkv * hd, d, f1), ("attn_v", nkv * hd, d, f1), ("attn_output", d, nh * hd, f1),
            ("ffn_gate", ff, d, f1), ("ffn_up", ff, d, f1), ("ffn_down", d, ff, f2)]


def _norm_weight(n, seed, part):
    return 1 + 0.1 * torch.randn(n, device=DEV, generator=_gen(seed, part))


def _block_norms(shape):
    arch, d, nh, nkv, hd = SHAPES[shape][:5]
    return [("attn_norm", d), ("ffn_norm", d)] + ([("attn_q_norm", hd), ("attn_k_norm", hd)] if arch == "qwen3" else [])


def _batch(c, seed):
    """tokens, position and segment of each token, target places, target tokens, weights."""
    vocab = SHAPES[c["shape"]][7]
    r = np.random.RandomState(seed % (1 << 31))
    t, m = c["t"], c["targets"]
    tokens = r.randint(0, vocab, t).astype(np.int32)
    if c["packed"]:
        own = t - c["shared"]
        cut = [c["shared"] + own * i // c["packed"] for i in range(c["packed"] + 1)]
        seg = np.zeros(t, np.int32)
        at = np.arange(t, dtype=np.int32)
        pos = []
        for i in range(c["packed"]):
            seg[cut[i]:cut[i + 1]] = i + 1
            at[cut[i]:cut[i + 1]] = np.arange(cut[i + 1] - cut[i]) + c["shared"]
            n = max(1, min(m * (i + 1) // c["packed"] - m * i // c["packed"], cut[i + 1] - cut[i] - 1))
            pos += range(cut[i + 1] - 1 - n, cut[i + 1] - 1)  # the end of each example is its answer
        pos = np.array(pos, np.int32)
    else:
        seg, at, cut = np.zeros(t, np.int32), np.arange(t, dtype=np.int32), []
        pos = np.arange(t - 1 - m, t - 1, dtype=np.int32)
    tok = tokens[pos + 1].copy()
    wts = ((0.5 + r.rand(len(pos))) / len(pos)).astype(np.float32)
    return tokens, at, seg, cut[:-1], pos, tok, wts


def _image(c, seed):
    """The GGUF file of a decoder of the case's shape."""
    arch, d, nh, nkv, hd, ff, base, vocab, f1, f2, f3 = SHAPES[c["shape"]]
    w = G.GgufWriter()
    V = G.Value
    for key, v in (("general.architecture", V.String(arch)), (f"{arch}.block_count", V.U32(c["layers"])),
                   (f"{arch}.context_length", V.U32(8192)), (f"{arch}.embedding_length", V.U32(d)),
                   (f"{arch}.feed_forward_length", V.U32(ff)), (f"{arch}.attention.head_count", V.U32(nh)),
                   (f"{arch}.attention.head_count_kv", V.U32(nkv)), (f"{arch}.attention.key_length", V.U32(hd)),
                   (f"{arch}.attention.value_length", V.U32(hd)), (f"{arch}.attention.layer_norm_rms_epsilon", V.F32(EPS)),
                   (f"{arch}.rope.dimension_count", V.U32(hd)), (f"{arch}.rope.freq_base", V.F32(base)),
                   (f"{arch}.vocab_size", V.U32(vocab))):
        w.kv(key, v)

    def put(name, fmt, values):
        w.tensor(name, [values.shape[-1]] + ([values.shape[0]] if values.dim() == 2 else []), FMT.get(fmt, 0), _blocks(fmt, values))

    put("token_embd.weight", f3, _weights(vocab, d, seed, 10))
    for i in range(c["layers"]):
        for j, (name, n) in enumerate(_block_norms(c["shape"])):
            put(f"blk.{i}.{name}.weight", "f32", _norm_weight(n, seed, 100 * i + 50 + j))
        for j, (name, n, k, f) in enumerate(_linears(c["shape"])):
            put(f"blk.{i}.{name}.weight", f, _weights(n, k, seed, 100 * i + 20 + j))
    put("output_norm.weight", "f32", _norm_weight(d, seed, 11))
    try:
        return w.to_bytes()
    finally:
        w.close()


class _Memory:
    """Device memory of the model as a tensor (its optimiser reads and writes the adapters in place)."""

    def __init__(self, address, shape, row):
        self.__cuda_array_interface__ = {"shape": shape, "typestr": "<f4", "data": (address, False), "version": 3,
                                         "strides": (4 * row, 4)}

    def tensor(self):
        return torch.as_tensor(self, device=DEV)


def _prepare_model(c, seed):
    model = rt.GpuModel.from_gguf(G.GgufFile.from_bytes(_image(c, seed)))
    model.attach_lora(c["r"], 2.0 * c["r"], seed=1)
    count = model.lora_count()
    for i in range(count):
        layer, j = divmod(i, 7)
        _, n, k, _ = _linears(c["shape"])[j]
        a, b = _adapter(n, k, c["r"], seed, 100 * layer + 70 + j)
        model.set_lora(i, a.cpu().numpy(), b.cpu().numpy())
    tokens, at, seg, cut, pos, tok, wts = _batch(c, seed)
    targets = [rt.Target(int(p), int(q)) for p, q in zip(pos, tok)]
    packed = Packed(tokens, at, seg, c["shared"], cut) if c["packed"] else None
    ga, gb = [], []
    for i in range(count):
        inf = model.lora_info(i)
        _, _, pa, pb, row = model.lora_device(i)
        ga.append(_Memory(pa, (inf["rank"], inf["in_dim"]), inf["in_dim"]).tensor())
        gb.append(_Memory(pb, (inf["out_dim"], inf["rank"]), row).tensor())
    return {"model": model, "tokens": tokens, "packed": packed, "targets": targets, "weights": wts, "ga": ga, "gb": gb,
            "stream": torch.cuda.ExternalStream(model.ctx.stream), "train": c["train"]}


def prepare(case, seed):
    c = case
    if c["kind"] == "model":
        return {"kind": "model", **_prepare_model(c, seed)}
    ctx = rt.default_context()
    w = rt.HipFrozen(FMT[c["fmt"]], _blocks(c["fmt"], _weights(c["n"], c["k"], seed, 1)), c["n"], c["k"], ctx=ctx)
    s = {"kind": c["kind"], "w": w, "t": c["t"], "lib": _ffi.lib(), "ctx": ctx}
    if c["kind"] == "loss":
        s["x"], s["norm"], s["pos"], s["tok"], s["wts"] = _loss_inputs(c, seed)
        s["n"] = c["targets"]
        s["logp"] = torch.empty(c["targets"], device=DEV)
        s["hit"] = torch.empty(c["targets"], device=DEV, dtype=torch.int32)
        s["dx"] = torch.empty(c["t"], c["k"], device=DEV)
        return s
    x, dy, a, b = _linear_inputs(c, seed)
    if c["kind"] == "host":
        lin = rt.Linear("linear", w)
        lin.lora = rt.Lora(c["r"], 2.0 * c["r"], a.cpu().numpy(), b.cpu().numpy())
        s.update(lin=lin, x=x.cpu().numpy(), dy=dy.cpu().numpy())
        return s
    s.update(x=x, dy=dy, dir=c["dir"], y=torch.empty(c["t"], c["n"], device=DEV), dx=torch.empty(c["t"], c["k"], device=DEV))
    if c["kind"] == "linear":
        s.update(a=a, b=b, grads=torch.zeros(c["r"] * (c["n"] + c["k"]), device=DEV),
                 lora=_ffi.RtqLora(c["r"], 2.0 * c["r"], a.data_ptr(), b.data_ptr(), 1))
        s["ga"], s["gb"] = s["grads"][:c["r"] * c["k"]].view(c["r"], c["k"]), s["grads"][c["r"] * c["k"]:].view(c["n"], c["r"])
    return s


# ------------------------------------------------------------------ one pass
def _run_linear(s):
    lib, ctx, w, t = s["lib"], s["ctx"].handle, s["w"].handle, s["t"]
    st = torch.cuda.current_stream().cuda_stream or None
    lora = ctypes.byref(s["lora"])
    out = []
    if s["dir"] != "bwd":
        _ffi.check(lib.rtq_linear_forward_d(ctx, w, None, lora, s["x"].data_ptr(), t, s["y"].data_ptr(), st), "forward")
        out.append(s["y"])
    if s["dir"] != "fwd":
        s["grads"].zero_()
        _ffi.check(lib.rtq_linear_backward_d(ctx, w, lora, s["x"].data_ptr(), s["dy"].data_ptr(), t, s["dx"].data_ptr(),
                                             s["ga"].data_ptr(), s["gb"].data_ptr(), st), "backward")
        out += [s["dx"], s["ga"], s["gb"]]
    return out


def run(state):
    s = state
    if s["kind"] == "linear":
        return _run_linear(s)
    st = torch.cuda.current_stream().cuda_stream
    if s["kind"] == "frozen":
        if s["dir"] == "fwd":
            s["w"].forward_d(s["x"].data_ptr(), s["t"], s["y"].data_ptr(), st)
            return [s["y"]]
        s["dx"].zero_()
        s["w"].backward_input_d(s["dy"].data_ptr(), s["t"], s["dx"].data_ptr(), st)
        return [s["dx"]]
    if s["kind"] == "loss":
        head_d(s["w"], s["norm"].data_ptr(), s["x"].data_ptr(), s["t"], s["pos"].data_ptr(), s["tok"].data_ptr(),
                                      s["wts"].data_ptr(), s["n"], s["logp"].data_ptr(), s["hit"].data_ptr(), s["dx"].data_ptr(),
                                      eps=EPS, stream=st)
        return [s["logp"], s["dx"]]
    if s["kind"] == "host":
        lin = s["lin"]
        lin.lora.zero_grad()
        y = lin.forward(s["x"], s["t"])
        dx = lin.backward(s["x"], s["dy"], s["t"])
        return [y, dx, lin.lora.ga, lin.lora.gb]
    model = s["model"]
    if s["train"]:
        model.zero_grad()
    wts = s["weights"] if s["train"] else None
    if s["packed"] is not None:
        logp, _ = model.forward_backward_packed(s["packed"], s["targets"], wts)
    else:
        logp, _ = model.forward_backward(s["tokens"], s["targets"], wts)
    if not s["train"]:
        return [logp]
    with torch.cuda.stream(s["stream"]):  # the gradients as an optimiser takes them: one matrix of each kind
        return [logp, torch.cat(s["ga"], 1), torch.cat(s["gb"], 0)]


# ------------------------------------------------------------------ work and tolerance
def _nbytes(fmt, n, k):
    e, b = ROW_BYTES[fmt]
    return n * k // e * b


def work(case):
    c = case
    if c["kind"] == "model":
        arch, d, nh, nkv, hd, ff, base, vocab, f1, f2, f3 = SHAPES[c["shape"]]
        t, m, passes = c["t"], c["targets"], 2 if c["train"] else 1
        per = sum(n * k for _, n, k, _ in _linears(c["shape"]))
        lora = sum((n + k) * c["r"] for _, n, k, _ in _linears(c["shape"]))
        wb = sum(_nbytes(f, n, k) for _, n, k, f in _linears(c["shape"]))
        if c["packed"]:
            own = (t - c["shared"]) / c["packed"]
            pairs = c["shared"] ** 2 / 2 + c["packed"] * (own * c["shared"] + own * own / 2)
        else:
            pairs = t * t / 2
        flops = c["layers"] * (2 * t * per * passes + 2 * t * lora * (3 if c["train"] else 1)
                               + 4 * nh * hd * pairs * (3.5 if c["train"] else 1)) + 2 * m * vocab * d * passes
        bytes_ = passes * (c["layers"] * wb + _nbytes(f3, vocab, d)) + (4 * 3 * c["layers"] * lora if c["train"] else 4 * c["layers"] * lora)
        return {"bytes": bytes_, "flops": flops}
    n, k, t, r = c["n"], c["k"], c["t"], c.get("r", 0)
    if c["kind"] == "loss":
        m = c["targets"]
        return {"bytes": 2 * _nbytes(c["fmt"], n, k) + 4 * (m * k + t * k), "flops": 4 * m * n * k}
    fwd, bwd = c["dir"] != "bwd", c["dir"] != "fwd"
    bytes_ = flops = 0
    if fwd:
        bytes_ += _nbytes(c["fmt"], n, k) + 4 * (t * k + t * n + r * (n + k))
        flops += 2 * t * n * k + 2 * t * r * (n + k)
    if bwd:
        bytes_ += _nbytes(c["fmt"], n, k) + 4 * (t * n + t * k * (2 if r else 1) + 2 * r * (n + k))
        flops += 2 * t * n * k + 6 * t * r * (n + k)
    return {"bytes": bytes_, "flops": flops}


def tolerance(case):
    # every projection of a decoder rounds its input to 8 bits, so a last-bit difference in one layer turns codes in the
    # next: the same step with its attention summed in another order measured 0.014 off, single values up to 0.55
    if case["kind"] == "model":
        return {"rel": 3e-2, "max": 0.99}
    if case["kind"] == "loss":
        return {"rel": 1e-3}  # one rounding to 8 bits after the norm
    return {"rel": 1e-5}  # 32-bit sums and split 16-bit products: up to 1.5e-6 off the 64-bit result


# ------------------------------------------------------------------ the same in 64 bits
def _exact_linear(c, seed):
    w = _decode(c["fmt"], _weights(c["n"], c["k"], seed, 1))
    x, dy, a, b = _linear_inputs(c, seed)
    direction = "both" if c["kind"] == "host" else c["dir"]
    out = []
    if direction != "bwd":
        y = _codes(c["fmt"], x) @ w.T
        if a is not None:
            y += 2.0 * ((x.double() @ a.double().T) @ b.double().T)
        out.append(y)
    if direction != "fwd":
        dy, x = dy.double(), x.double()
        dx = dy @ w
        if a is not None:
            g = 2.0 * (dy @ b.double())
            dx += g @ a.double()
            out += [dx, g.T @ x, 2.0 * (dy.T @ (x @ a.double().T))]
        else:
            out.append(dx)
    return [v.reshape(-1) for v in out] if c["kind"] == "host" else out


def _norm(x, w):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + EPS) * w


class _Frozen(torch.autograd.Function):
    """The forward takes the activation's 8-bit blocks, the backward the weight's values alone."""

    @staticmethod
    def forward(ctx, x, w, fmt):
        ctx.save_for_backward(w)
        return _codes(fmt, x) @ w.T

    @staticmethod
    def backward(ctx, dy):
        return dy @ ctx.saved_tensors[0], None, None


class _Half(torch.autograd.Function):
    """Keys and values are kept as 16-bit floats; the gradient passes."""

    @staticmethod
    def forward(ctx, x):
        return x.to(torch.float32).to(torch.float16).double()

    @staticmethod
    def backward(ctx, d):
        return d


def _loss_exact(x, norm, w, fmt, pos, tok):
    rows = _norm(x[pos.long()], norm)
    logits = _Frozen.apply(rows, w, fmt)
    return logits.log_softmax(-1).gather(1, tok.long()[:, None])[:, 0]


def _exact_loss(c, seed):
    w = _decode(c["fmt"], _weights(c["n"], c["k"], seed, 1))
    x, norm, pos, tok, wts = _loss_inputs(c, seed)
    x = x.double().requires_grad_(True)
    logp = _loss_exact(x, norm.double(), w, c["fmt"], pos, tok)
    (-(wts.double() * logp).sum()).backward()
    return [logp.detach(), x.grad]


def _heads(q, k, v, mask):
    s = (q @ k.transpose(-1, -2)).masked_fill(~mask, -math.inf)
    return s.softmax(-1) @ v


def _exact_model(c, seed):
    arch, d, nh, nkv, hd, ff, base, vocab, f1, f2, f3 = SHAPES[c["shape"]]
    tokens, at, seg, _, pos, tok, wts = (torch.from_numpy(v).to(DEV) if isinstance(v, np.ndarray) else v for v in _batch(c, seed))
    t, r, group = c["t"], c["r"], nh // nkv
    embed = _decode(f3, _weights(vocab, d, seed, 10))
    freq = torch.from_numpy(np.power(np.float32(base), np.float32(-2.0) * np.arange(hd // 2, dtype=np.float32) / np.float32(hd))).to(DEV)
    angle = (at.float()[:, None] * freq[None, :]).double()
    cos, sin = angle.cos()[:, None, :], angle.sin()[:, None, :]
    i = torch.arange(t, device=DEV)
    mask = (i[None, :] <= i[:, None]) & ((seg[None, :] == 0) | (seg[None, :] == seg[:, None]))
    adapters = []

    def rope(x):
        if arch == "qwen3":
            a, b = x[..., :hd // 2], x[..., hd // 2:]
            return torch.cat([a * cos - b * sin, b * cos + a * sin], -1)
        a, b = x[..., 0::2], x[..., 1::2]
        return torch.stack([a * cos - b * sin, b * cos + a * sin], -1).reshape(x.shape)

    def block(x, layer):
        ab = []
        for j, (_, n, k, _) in enumerate(_linears(c["shape"])):
            ab.append([v.double().requires_grad_(c["train"]) for v in _adapter(n, k, r, seed, 100 * layer + 70 + j)])
        adapters.extend(ab)

        def linear(j, v):
            _, n, k, f = _linears(c["shape"])[j]
            w = _decode(f, _weights(n, k, seed, 100 * layer + 20 + j))
            return _Frozen.apply(v, w, f) + 2.0 * ((v @ ab[j][0].T) @ ab[j][1].T)

        norms = {name: _norm_weight(n, seed, 100 * layer + 50 + j).double() for j, (name, n) in enumerate(_block_norms(c["shape"]))}
        h = _norm(x, norms["attn_norm"])
        q, k, v = linear(0, h).view(t, nh, hd), linear(1, h).view(t, nkv, hd), linear(2, h).view(t, nkv, hd)
        if arch == "qwen3":
            q, k = _norm(q, norms["attn_q_norm"]), _norm(k, norms["attn_k_norm"])
        q, k, v = rope(q) / math.sqrt(hd), _Half.apply(rope(k)), _Half.apply(v)
        o = [torch.utils.checkpoint.checkpoint(_heads, q[:, n], k[:, n // group], v[:, n // group], mask, use_reentrant=False)
             for n in range(nh)]
        x = x + linear(3, torch.stack(o, 1).reshape(t, nh * hd))
        h = _norm(x, norms["ffn_norm"])
        return x + linear(6, torch.nn.functional.silu(linear(4, h)) * linear(5, h))

    with torch.set_grad_enabled(c["train"]):
        x = embed[tokens.long()]
        for layer in range(c["layers"]):
            x = block(x, layer)
        logp = _loss_exact(x, _norm_weight(d, seed, 11).double(), embed, f3, pos, tok)
        if not c["train"]:
            return [logp]
        (-(wts.double() * logp).sum()).backward()
    return [logp.detach(), torch.cat([a.grad for a, _ in adapters], 1), torch.cat([b.grad for _, b in adapters], 0)]


def exact(case, seed):
    if case["kind"] == "model":
        return _exact_model(case, seed)
    if case["kind"] == "loss":
        return _exact_loss(case, seed)
    return _exact_linear(case, seed)
