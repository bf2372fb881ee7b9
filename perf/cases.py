"""The work that users of this framework have it do, as cases that can be timed: speech-to-text with the whisper models.

Three kinds of work, each through the kernel ABI of include/mi355x_kernels.h in the order in which the ggml plugin's graph
walker issues its launches:

  mel      16 kHz samples -> log-mel spectrogram (mi355x_log_mel_spectrogram), the whole recording in one call
  encode   one window: conv stem, the encoder's layers, the cross-attention K / V of every decoder layer (whisper_encode)
  decode   one call of the decoder (whisper_decode): 1 .. 8 rows are a step of greedy, best-of or beam decoding, more rows
           are a prompt that is read in at once; the logits of every row come out

over the published models (width, heads, layers, vocabulary), the weight types their files come in (F16 as released, Q8_0 and
Q5_0 as quantized by users), windows of 64 to 1500 encoder positions (live transcription shortens the window), and both
attention paths of whisper.cpp: flash attention, and separate products and soft_max, which is what its parameters default to.
Weights are random with the scale of trained ones, and each layer has its own.
"""
from __future__ import annotations

import ctypes as C
import math

import torch

import __graft_entry__

# name: width, heads, encoder layers, decoder layers, mel bands, vocabulary (the sizes of the released model files)
MODELS = {
    "tiny": (384, 6, 4, 4, 80, 51865),
    "base": (512, 8, 6, 6, 80, 51865),
    "small": (768, 12, 12, 12, 80, 51865),
    "medium": (1024, 16, 24, 24, 80, 51865),
    "large-v3": (1280, 20, 32, 32, 128, 51866),
    "large-v3-turbo": (1280, 20, 32, 4, 128, 51866),
}
BYTES = {"f16": 2.0, "q8_0": 34 / 32, "q5_0": 22 / 32}      # per weight
TEXT_CTX = 448
EPS = 1e-5


def listed():
    return [
        # live transcription: three seconds of microphone input every three seconds, one spectrogram each
        {"name": "mel_live_3s", "kind": "mel", "samples": 48000, "bands": 80},
        # a recording of an hour and some: the host computes the spectrogram of the whole file before its first window
        {"name": "mel_file_1h", "kind": "mel", "samples": 58_123_457, "bands": 128},
        # live transcription on the smallest model with the shortened window its users set
        {"name": "encode_tiny_q5_0_ctx487", "kind": "encode", "model": "tiny", "type": "q5_0", "ctx": 487, "attn": "flash"},
        # the model most people try first, as released, a full 30 s window
        {"name": "encode_base_f16", "kind": "encode", "model": "base", "type": "f16", "ctx": 1500, "attn": "flash"},
        # the default parameters of whisper.cpp: no flash attention
        {"name": "encode_small_q8_0_plain", "kind": "encode", "model": "small", "type": "q8_0", "ctx": 1500, "attn": "plain"},
        # the largest model, quantized to fit next to other work: the heaviest single call
        {"name": "encode_large_v3_q5_0", "kind": "encode", "model": "large-v3", "type": "q5_0", "ctx": 1500, "attn": "flash"},
        # greedy decoding with the default parameters, one token
        {"name": "decode_base_f16_greedy_plain", "kind": "decode", "model": "base", "type": "f16", "rows": 1, "past": 61, "ctx": 1500, "attn": "plain"},
        # best-of-three decoding of a short window
        {"name": "decode_small_q5_0_rows3", "kind": "decode", "model": "small", "type": "q5_0", "rows": 3, "past": 118, "ctx": 617, "attn": "flash"},
        # beam search with five beams, late in a window, on the model made for fast decoding
        {"name": "decode_turbo_q8_0_beam5", "kind": "decode", "model": "large-v3-turbo", "type": "q8_0", "rows": 5, "past": 300, "ctx": 1500, "attn": "flash"},
        # beam search on the largest model as released: 1.6 GB of weights for every step
        {"name": "decode_large_v3_f16_beam5", "kind": "decode", "model": "large-v3", "type": "f16", "rows": 5, "past": 200, "ctx": 1500, "attn": "flash"},
        # an initial prompt of a sentence or two
        {"name": "prompt_small_q5_0_27", "kind": "decode", "model": "small", "type": "q5_0", "rows": 27, "past": 0, "ctx": 1500, "attn": "flash"},
        # the longest prompt there is: the text of the window before (half the text context) and the start tokens
        {"name": "prompt_turbo_q8_0_227", "kind": "decode", "model": "large-v3-turbo", "type": "q8_0", "rows": 227, "past": 0, "ctx": 1500, "attn": "flash"},
    ]


def log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["mel", "encode", "encode", "decode", "decode", "prompt"])
    if kind == "mel":
        return {"kind": "mel", "samples": log_int(rng, 16000, 58_000_000), "bands": rng.choice([80, 128])}
    # (without flash attention up to the middle-sized models: the largest call stays the largest listed one)
    attn = rng.choice(["flash", "flash", "plain"])
    model = rng.choice(["tiny", "base", "small"] if attn == "plain" else list(MODELS))
    case = {"kind": "encode" if kind == "encode" else "decode", "model": model, "type": rng.choice(["f16", "q8_0", "q5_0"])}
    if kind == "encode":
        case["ctx"] = log_int(rng, 64, 1500)
    else:
        case["rows"] = rng.randint(1, 8) if kind == "decode" else log_int(rng, 9, 227)
        case["past"] = log_int(rng, 4, TEXT_CTX - 8) if kind == "decode" else 0
        case["ctx"] = rng.choice([1500, log_int(rng, 64, 1500)])
    case["attn"] = attn
    return case


def work(case):
    if case["kind"] == "mel":
        n_len = (case["samples"] + 480000) // 160
        frames = case["samples"] // 160 + 2
        # a frame's transform as a real fast Fourier transform, its power spectrum and the filter bank's two entries per bin
        return {"bytes": 4 * case["samples"] + 4 * case["bands"] * n_len, "flops": frames * (2.5 * 400 * math.log2(400) + 7 * 201)}
    d, _, enc, dec, mels, vocab = MODELS[case["model"]]
    t, wb = case["ctx"], BYTES[case["type"]]
    if case["kind"] == "encode":
        weights = 3 * mels * d + 3 * d * d
        flops = 2 * (2 * t) * 3 * mels * d + 2 * t * 3 * d * d + enc * (24 * t * d * d + 4 * t * t * d) + dec * 4 * t * d * d
        return {"bytes": 2 * weights + wb * (enc * 12 + dec * 2) * d * d + 4 * 2 * t * mels + 4 * t * d + 2 * dec * 2 * t * d, "flops": flops}
    n, kv = case["rows"], case["past"] + case["rows"]
    weights = 14 * d * d * dec + vocab * d
    return {"bytes": wb * weights + 4 * dec * (kv + t) * d + 4 * n * vocab, "flops": 2 * n * weights + 4 * n * (kv + t) * d * dec}


def tolerance(case):
    if case["kind"] == "mel":
        return {"rel": 1e-5}
    # f16 operands and f16 attention sums through every layer of a model: 1e-3 to 2e-3 between two correct forms
    if case["type"] == "f16":
        return {"rel": 4e-3}
    # Products over quantized weights round their activations to Q8_0 first (one part in 254 of a block's largest value): one
    # f32 sum in another order draws every later rounding anew, which comes to 1.3e-2 .. 3.1e-2 at the end of a model (the
    # library's two forms of the attention step, x86 and Arm order of operations, over 50 cases)
    return {"rel": 4e-2}


# ---- what a user's program holds ------------------------------------------------------------------------------------------

class Program:
    """Device memory, weights and the list of library calls of one pass.

    Buffers are torch tensors in torch's order of dimensions; descriptors are in ggml's (first dimension contiguous)."""

    def __init__(self, seed):
        self.p = __graft_entry__.package()
        self.lib = self.p.kernels()
        self.gen = torch.Generator(device="cuda").manual_seed(seed)
        self.stream = C.c_void_p(torch.cuda.current_stream().cuda_stream)
        self.keep, self.calls, self.out = [], [], {}

    # -- memory
    def zeros(self, *shape, dtype=torch.float32):
        t = torch.zeros(shape, dtype=dtype, device="cuda")
        self.keep.append(t)
        return t

    def randn(self, *shape, std=1.0, mean=0.0, dtype=torch.float32):
        t = (torch.randn(shape, generator=self.gen, device="cuda") * std + mean).to(dtype)
        self.keep.append(t)
        return t

    def desc(self, t, ne=None, nb=None, type_=None):
        if type_ is None:
            type_ = {torch.float32: self.p.F32, torch.float16: self.p.F16, torch.int32: self.p.I32}[t.dtype]
        d = self.p.tensor(t, type_, ne, nb)
        self.keep.append(d)
        return d

    # -- weights: a [rows, k] matrix as blocks of 32, and the forms of it that the plugin keeps beside it
    def quantize(self, w, type_):
        b = w.reshape(-1, 32)
        if type_ == "q8_0":
            d = (b.abs().amax(1) / 127.0).to(torch.float16)
            s = d.float()
            q = torch.round(b / torch.where(s == 0, torch.ones_like(s), s)[:, None]).clamp(-127, 127).to(torch.int8)
            blocks = torch.cat([d.view(torch.uint8).reshape(-1, 2), q.view(torch.uint8)], 1)
        else:
            top = b.gather(1, b.abs().argmax(1, keepdim=True))[:, 0]
            d = (top / -16.0).to(torch.float16)
            s = d.float()
            q = torch.floor(b / torch.where(s == 0, torch.ones_like(s), s)[:, None] + 16.5).clamp(0, 31).to(torch.int64)
            nib = ((q[:, :16] & 15) | ((q[:, 16:] & 15) << 4)).to(torch.uint8)
            bits = ((q >> 4) << torch.arange(32, device="cuda")).sum(1)
            qh = torch.stack([(bits >> (8 * i)) & 255 for i in range(4)], 1).to(torch.uint8)
            blocks = torch.cat([d.view(torch.uint8).reshape(-1, 2), qh, nib], 1)
        return blocks.contiguous()

    def matrix(self, rows, k, type_, image, gain=1.0):
        """Descriptor of random weights; with `image`, quantized ones as their f16 image (what products over many columns read)."""
        w = torch.randn((rows, k), generator=self.gen, device="cuda") * (gain / math.sqrt(k))
        if type_ == "f16":
            w = w.to(torch.float16)
            self.keep.append(w)
            return self.desc(w)
        t = self.p.Q8_0 if type_ == "q8_0" else self.p.Q5_0
        blocks = self.quantize(w, type_)
        if not image:
            self.keep.append(blocks)
            return self.desc(blocks, [k, rows], None, t)
        half = self.zeros(rows, k, dtype=torch.float16)
        self.now("mi355x_dequantize_row_f16", t, blocks.data_ptr(), half.data_ptr(), rows * k, self.stream)
        torch.cuda.synchronize()
        return self.desc(half)

    # -- calls
    def now(self, name, *args):
        status = getattr(self.lib, name)(*args)
        self.p.check(status, name)

    def call(self, name, *args):
        fn = getattr(self.lib, name)
        fixed = tuple(C.byref(a) if isinstance(a, C.Structure) else a for a in args)
        self.keep.append(args)
        self.calls.append((fn, fixed))

    def call_or(self, name, args, otherwise):
        """The fused entry where the library takes these shapes, what it asks for instead where it says that it does not."""
        status = getattr(self.lib, name)(*args)
        if status == 0:
            self.call(name, *args)
        elif status == -1:
            otherwise()
        else:
            self.p.check(status, name)
        return status == 0

    def epilogue(self, flags, scale=1.0, bias=None, residual=None, image=None):
        ptr = [None if t is None else t.data_ptr() for t in (bias, residual, image)]
        e = self.p.Epilogue(flags, scale, *ptr)
        self.keep.append(e)
        return e

    def items(self, triples):
        arr = (self.p.MulMatItem * len(triples))(*[self.p.MulMatItem(C.pointer(w), C.pointer(d), C.pointer(e)) for w, d, e in triples])
        self.keep.append(arr)
        return arr

    def many(self, triples, x, flags, ws):
        """Products over the same activations: one launch where the library takes the shapes, else one after the other."""
        arr = self.items(triples)

        def singles():
            ready = flags & self.p.MM_WS_READY
            for w, d, e in triples:
                e.flags |= ready | (flags & ~self.p.MM_WS_READY)
                self.call("mi355x_mul_mat", w, x, d, e, ws.data_ptr(), ws.numel(), self.stream)
                ready = self.p.MM_WS_READY
        if len(triples) < 2:
            singles()
        else:
            self.call_or("mi355x_mul_mat_group", (arr, len(triples), x, flags, ws.data_ptr(), ws.numel(), self.stream), singles)


def pad(n, m):
    return (n + m - 1) // m * m


def heads_view(pr, t, n, h, esz):
    """[n, width] rows as ggml's [64, n, h]."""
    return pr.desc(t, [64, n, h], [esz, 64 * h * esz, 64 * esz])


def attention_plain(pr, q, k, v_t, mask, n, kv, h, scale, out):
    """KQ, soft_max, KQV and the merge of the heads as separate calls; k: descriptor [64, kv, h], v_t: [kv, 64, h]."""
    d = 64 * h
    kq, o = pr.zeros(h, n, kv), pr.zeros(h, n, 64)
    ws = pr.zeros(max(pr.lib.mi355x_mul_mat_workspace_size(k, q), pr.lib.mi355x_mul_mat_workspace_size(v_t, pr.desc(kq)), 256), dtype=torch.uint8)
    pr.call("mi355x_mul_mat", k, q, pr.desc(kq), None, ws.data_ptr(), ws.numel(), pr.stream)
    pr.call("mi355x_soft_max", pr.desc(kq), mask, pr.desc(kq), scale, pr.stream)
    pr.call("mi355x_mul_mat", v_t, pr.desc(kq), pr.desc(o), None, ws.data_ptr(), ws.numel(), pr.stream)
    pr.call("mi355x_cpy", pr.desc(o, [64, h, n], [4, 256 * n, 256]), pr.desc(out, [64, h, n], [4, 256, 4 * d]), pr.stream)


def layer_norm(pr, d):
    return pr.randn(d, std=0.2, mean=1.0), pr.randn(d, std=0.1)


# ---- mel ------------------------------------------------------------------------------------------------------------------

def prepare_mel(pr, case):
    n, bands = case["samples"], case["bands"]
    # speech-like level: noise under a slow envelope with pauses, and a few tones
    t = torch.arange(n, device="cuda", dtype=torch.float64) / 16000.0
    env = (0.5 + 0.5 * torch.sin(2 * math.pi * 0.31 * t)).square()
    x = 0.1 * env * torch.randn(n, generator=pr.gen, device="cuda")
    for f in (140.0, 733.0, 2310.0):
        x += 0.05 * env * torch.sin(2 * math.pi * f * t)
    x = x.to(torch.float32)
    # triangular bands on the mel scale over the 201 bins, as in the model files
    edges = 700.0 * (torch.pow(10.0, torch.linspace(0, 2595.0 * math.log10(1 + 8000.0 / 700.0), bands + 2) / 2595.0) - 1)
    freq = torch.linspace(0, 8000.0, 201)
    lo, mid, hi = edges[:-2, None], edges[1:-1, None], edges[2:, None]
    bank = torch.minimum((freq - lo) / (mid - lo), (hi - freq) / (hi - mid)).clamp_min(0) * (2.0 / (hi - lo))
    bank = bank.to(torch.float32).contiguous().cuda()
    mel = pr.zeros(bands, pr.lib.mi355x_log_mel_n_len(n))
    ws = pr.zeros(pr.lib.mi355x_log_mel_workspace_size(bands), dtype=torch.uint8)
    pr.keep += [x, bank]
    pr.call("mi355x_log_mel_spectrogram", x.data_ptr(), n, bank.data_ptr(), bands, mel.data_ptr(), ws.data_ptr(), ws.numel(), pr.stream)
    pr.out = {"mel": mel}


# ---- encode ---------------------------------------------------------------------------------------------------------------

def prepare_encode(pr, case):
    p, lib = pr.p, pr.lib
    d, h, enc, dec, mels, _ = MODELS[case["model"]]
    t, type_, flash = case["ctx"], case["type"], case["attn"] == "flash"
    quant = type_ != "f16"
    act = p.MM_ACT_Q8_0 if quant else 0
    tp = pad(t, 256) if flash else t
    ws = [pr.zeros(pad(2 * t * 4 * d, 256) + 256, dtype=torch.uint8) for _ in range(2)]
    w0 = (ws[0].data_ptr(), ws[0].numel(), pr.stream)
    w1 = (ws[1].data_ptr(), ws[1].numel(), pr.stream)

    # conv stem: two 1-d convolutions with GELU, then the sum with the positional embedding
    mel = pr.randn(mels, 2 * t, std=0.5, mean=0.1)
    col1, col2 = pr.zeros(2 * t, 3 * mels, dtype=torch.float16), pr.zeros(t, 3 * d, dtype=torch.float16)
    y1, y2, x0, pos = pr.zeros(d, 2 * t), pr.zeros(d, t), pr.zeros(t, d), pr.randn(t, d, std=0.5)
    for src, col, y, k, stride in ((mel, col1, y1, 3 * mels, 1), (y1, col2, y2, 3 * d, 2)):
        e = pr.epilogue(p.EPI_BIAS_COL | p.EPI_GELU, bias=pr.randn(d, std=0.1))
        pr.call("mi355x_im2col_1d", pr.desc(src), pr.desc(col), 3, stride, 1, 1, pr.stream)
        pr.call("mi355x_mul_mat", pr.desc(col), pr.matrix(d, k, "f16", False), pr.desc(y), e, *w0)
    xt = pr.zeros(t, d)
    pr.call("mi355x_cpy", pr.desc(y2, [d, t], [4 * t, 4]), pr.desc(xt), pr.stream)
    pr.call("mi355x_binary", 0, pr.desc(pos), pr.desc(xt), pr.desc(x0), pr.stream)

    x1, normed, q, vf, ao, up = pr.zeros(t, d), pr.zeros(t, d), pr.zeros(t, d), pr.zeros(t, d), pr.zeros(t, d), pr.zeros(t, 4 * d)
    k16, v16 = pr.zeros(tp, d, dtype=torch.float16), pr.zeros(tp, d, dtype=torch.float16)
    tx0, tx1, tn, ta, tu = pr.desc(x0), pr.desc(x1), pr.desc(normed), pr.desc(ao), pr.desc(up)
    nowhere = pr.desc(normed)
    nowhere.data = None
    nowhere_attn = pr.desc(ao, [64, h, t])
    nowhere_attn.data = None
    rows16 = lambda buf: pr.desc(buf, [d, t], [2, 2 * d])

    def norm(src):
        w, b = layer_norm(pr, d)
        if quant:
            pr.call("mi355x_norm_emit_f16", src, nowhere, EPS, w.data_ptr(), b.data_ptr(), ws[0].data_ptr(), pr.stream)
            return p.MM_WS_READY
        pr.call("mi355x_norm", src, tn, EPS, w.data_ptr(), b.data_ptr(), pr.stream)
        return 0

    for _ in range(enc):
        ready = norm(tx0)
        wq, wk, wv, wo = (pr.matrix(d, d, type_, True, g) for g in (1.5, 1.5, 1.0, 0.5))
        eq, ev = (pr.epilogue(p.EPI_BIAS, bias=pr.randn(d, std=0.1)) for _ in range(2))
        if flash:
            ev.flags |= p.EPI_OUT_F16
            pr.many([(wk, rows16(k16), pr.epilogue(p.EPI_OUT_F16)), (wv, rows16(v16), ev), (wq, pr.desc(q), eq)], tn, act | ready, ws[0])
            tq, tk, tv = heads_view(pr, q, t, h, 4), heads_view(pr, k16, tp, h, 2), heads_view(pr, v16, tp, h, 2)
            if quant:
                pr.call("mi355x_flash_attn_ext", tq, tk, tv, None, nowhere_attn, 0.125, p.FA_F16_PK | p.FA_EMIT_F16, *w0)
                ready = p.MM_WS_READY
            else:
                pr.call("mi355x_flash_attn_ext", tq, tk, tv, None, pr.desc(ao, [64, h, t]), 0.125, p.FA_F16_PK, *w0)
                ready = 0
        else:
            pr.many([(wv, pr.desc(vf), ev)], tn, act | ready, ws[0])
            vt = pr.desc(v16, [t, 64, h], [2, 2 * t, 128 * t])
            pr.call("mi355x_cpy", pr.desc(vf, [t, 64, h], [4 * d, 4, 256]), vt, pr.stream)
            pr.many([(wk, rows16(k16), pr.epilogue(p.EPI_OUT_F16)), (wq, pr.desc(q), eq)], tn, act | p.MM_WS_READY, ws[0])
            attention_plain(pr, heads_view(pr, q, t, h, 4), heads_view(pr, k16, t, h, 2), vt, None, t, t, h, 0.125, ao)
            ready = 0
        pr.call("mi355x_mul_mat", wo, ta, tx1, pr.epilogue(p.EPI_BIAS | p.EPI_RESIDUAL | act | ready, bias=pr.randn(d, std=0.1), residual=x0), *w0)
        ready = norm(tx1)
        eu = pr.epilogue(p.EPI_BIAS | p.EPI_GELU | act | ready, bias=pr.randn(4 * d, std=0.1), image=ws[1])
        ed = pr.epilogue(p.EPI_BIAS | p.EPI_RESIDUAL | act, bias=pr.randn(d, std=0.1), residual=x1)
        if quant:
            eu.flags |= p.EPI_EMIT_F16 | p.EPI_IMAGE_ONLY
            ed.flags |= p.MM_WS_READY
        pr.call("mi355x_mul_mat", pr.matrix(4 * d, d, type_, True), tn, tu, eu, *w0)
        pr.call("mi355x_mul_mat", pr.matrix(d, 4 * d, type_, True, 0.5), tu, tx0, ed, *w1)
    embd = pr.zeros(t, d)
    w, b = layer_norm(pr, d)
    pr.call("mi355x_norm", tx0, pr.desc(embd), EPS, w.data_ptr(), b.data_ptr(), pr.stream)

    # K and V of every decoder layer's cross-attention
    kc, vc = pr.zeros(dec, tp, d, dtype=torch.float16), pr.zeros(dec, tp, d, dtype=torch.float16)
    first, group = 0, []
    for i in range(dec):
        ek = pr.epilogue(p.EPI_SCALE | p.EPI_OUT_F16, scale=64 ** -0.25)
        ev = pr.epilogue(p.EPI_BIAS | (p.EPI_OUT_F16 if flash else 0), bias=pr.randn(d, std=0.1))
        group += [(pr.matrix(d, d, type_, True, 1.5), rows16(kc[i]), ek), (pr.matrix(d, d, type_, True), rows16(vc[i]) if flash else pr.desc(vf), ev)]
        if flash and i + 1 < dec:
            continue
        pr.many(group, pr.desc(embd), act | first, ws[0])
        first, group = p.MM_WS_READY, []
        if not flash:
            pr.call("mi355x_cpy", pr.desc(vf, [t, d], [4 * d, 4]), pr.desc(vc[i], [t, d], [2, 2 * t]), pr.stream)
    pr.out = {"embd": embd, "k": kc[dec - 1], "v": vc[dec - 1]}


# ---- decode ---------------------------------------------------------------------------------------------------------------

def prepare_decode(pr, case):
    p, lib = pr.p, pr.lib
    d, h, _, dec, _, vocab = MODELS[case["model"]]
    n, past, t, type_, flash = case["rows"], case["past"], case["ctx"], case["type"], case["attn"] == "flash"
    quant, few = type_ != "f16", n <= 8
    image = not few                                     # many columns: the f16 images of quantized weights
    act = p.MM_ACT_Q8_0 if quant and image else 0
    tp = pad(t, 256) if flash else t
    cells = 512                                         # the self-attention cache: the text context, padded
    kv = min(cells, pad(past + n, 256 if flash else 32))
    qtype = {"f16": p.F16, "q8_0": p.Q8_0, "q5_0": p.Q5_0}[type_]

    # the token matrix serves the embedding and the logits
    te = torch.randn((vocab, d), generator=pr.gen, device="cuda") * 0.04
    te = te.to(torch.float16) if not quant else pr.quantize(te, type_)
    pr.keep.append(te)
    tte = pr.desc(te, [d, vocab], None, qtype)
    pos = pr.randn(TEXT_CTX, d, std=0.02)
    ids = torch.randint(0, vocab, (n,), generator=pr.gen, device="cuda", dtype=torch.int32)
    # a step's rows are alternatives for one position, a prompt's follow each other
    at = torch.full((n,), past, device="cuda", dtype=torch.int32) if few else torch.arange(past, past + n, device="cuda", dtype=torch.int32)
    mask = torch.full((pad(n, 64), kv), -math.inf, device="cuda")
    mask[:n, :past] = 0
    mask[:n, past:past + n] = torch.where(torch.eye(n, device="cuda") > 0, 0.0, -math.inf) if few else torch.triu(torch.full((n, n), -math.inf, device="cuda"), 1)
    mask16 = pr.zeros(pad(n, 64), kv, dtype=torch.float16)
    pr.keep += [ids, at, mask]
    tm, tm16 = pr.desc(mask), pr.desc(mask16)

    big = max(pad(2 * n * 4 * d, 256) + 256, 1 << 16)
    ws = [pr.zeros(big, dtype=torch.uint8) for _ in range(2)]
    w0 = (ws[0].data_ptr(), ws[0].numel(), pr.stream)
    w1 = (ws[1].data_ptr(), ws[1].numel(), pr.stream)
    x0, x1, normed, q, vf, ao, up, logits = (pr.zeros(n, w) for w in (d, d, d, d, d, d, 4 * d, vocab))
    tx0, tx1, tn, ta, tu, tl = (pr.desc(b) for b in (x0, x1, normed, ao, up, logits))
    nowhere, nowhere_attn = pr.desc(normed), pr.desc(ao, [64, h, n])
    nowhere.data = nowhere_attn.data = None
    embed = (tte, pr.desc(ids), pr.desc(pos), pr.desc(at))

    def gather():
        pr.call("mi355x_get_rows_add", *embed, tx0, pr.stream)

    def norm(src):
        """LayerNorm on its own; returns the flags of the products that take its result."""
        w, b = layer_norm(pr, d)
        if quant and few:
            pr.call("mi355x_norm_emit_q8_0", src, tn, EPS, w.data_ptr(), b.data_ptr(), ws[0].data_ptr(), pr.stream)
        elif quant:
            pr.call("mi355x_norm_emit_f16", src, nowhere, EPS, w.data_ptr(), b.data_ptr(), ws[0].data_ptr(), pr.stream)
        else:
            pr.call("mi355x_norm", src, tn, EPS, w.data_ptr(), b.data_ptr(), pr.stream)
        return p.MM_WS_READY if quant else 0

    def norm_products(src, triples, with_embedding=False):
        """LayerNorm and the products over it: one launch for the few rows of a step over quantized weights."""
        def apart():
            if with_embedding:
                gather()
            pr.many(triples, tn, act | norm(src), ws[0])
        if not (quant and few):
            return apart()
        w, b = layer_norm(pr, d)
        tail = (src, tn, EPS, w.data_ptr(), b.data_ptr(), pr.items(triples), len(triples)) + w0

        def two():
            if with_embedding:
                gather()
            pr.call_or("mi355x_norm_mul_mat_group", tail, lambda: pr.many(triples, tn, act | norm(src), ws[0]))
        if with_embedding:
            pr.call_or("mi355x_embed_norm_mul_mat_group", embed + tail, two)
        else:
            two()

    def attention(tq, tk, tv, m, scale, cast):
        """Returns the flags of the output projection."""
        if not flash:
            attention_plain(pr, tq, tk, tv, m, n, tk.ne[1], h, scale, ao)
            return 0
        mode, dst = p.FA_F16_PK, pr.desc(ao, [64, h, n])
        if quant:
            mode |= p.FA_EMIT_Q8_0 if few else p.FA_EMIT_F16
            dst = dst if few else nowhere_attn
        if cast:
            pr.call("mi355x_flash_attn_ext_cast_mask", tq, tk, tv, tm, tm16, dst, scale, mode, *w0)
        else:
            pr.call("mi355x_flash_attn_ext", tq, tk, tv, m, dst, scale, mode, *w0)
        return p.MM_WS_READY if quant else 0

    def project(src, into, residual, ready, rows_in, w_in):
        e = pr.epilogue(p.EPI_BIAS | p.EPI_RESIDUAL | act | ready, bias=pr.randn(d, std=0.1), residual=residual)
        pr.call("mi355x_mul_mat", pr.matrix(d, rows_in, type_, image, 0.5), src, into, e, *w_in)

    kq_scale = 64 ** -0.25
    if flash and not few:
        pr.call("mi355x_cpy", tm, tm16, pr.stream)
    for layer in range(dec):
        ks, kc = (pr.randn(rows, d, std=0.5, dtype=torch.float16) for rows in (cells, tp))
        vs, vc = (pr.randn(rows, d, dtype=torch.float16) for rows in (cells, tp))
        if flash:
            kc[t:], vc[t:] = 0, 0
        eq = pr.epilogue(p.EPI_BIAS | p.EPI_SCALE, scale=kq_scale, bias=pr.randn(d, std=0.1))
        ek = pr.epilogue(p.EPI_SCALE | p.EPI_OUT_F16, scale=kq_scale)
        ev = pr.epilogue(p.EPI_BIAS | (p.EPI_OUT_F16 if flash else 0), bias=pr.randn(d, std=0.1))
        wq, wk, wv = (pr.matrix(d, d, type_, image, g) for g in (1.5, 1.5, 1.0))
        new_k = pr.desc(ks[past:past + n])
        new_v = pr.desc(vs[past:past + n]) if flash else pr.desc(vf)
        norm_products(tx0, [(wq, pr.desc(q), eq), (wk, new_k, ek), (wv, new_v, ev)], with_embedding=layer == 0)
        tq = heads_view(pr, q, n, h, 4)
        if flash:
            tv = heads_view(pr, vs, kv, h, 2)
        else:
            pr.call("mi355x_cpy", pr.desc(vf, [n, d], [4 * d, 4]), pr.desc(vs.reshape(-1)[past:], [n, d], [2, 2 * cells]), pr.stream)
            tv = pr.desc(vs, [kv, 64, h], [2, 2 * cells, 128 * cells])
        ready = attention(tq, heads_view(pr, ks, kv, h, 2), tv, tm16 if flash else tm, 1.0, flash and few and layer == 0)
        project(ta, tx1, x0, ready, d, w0)

        # cross-attention over the encoder's positions
        ecq = pr.epilogue(p.EPI_BIAS, bias=pr.randn(d, std=0.1))
        norm_products(tx1, [(pr.matrix(d, d, type_, image, 1.5), pr.desc(q), ecq)])
        tv = heads_view(pr, vc, tp, h, 2) if flash else pr.desc(vc, [t, 64, h], [2, 2 * t, 128 * t])
        ready = attention(tq, heads_view(pr, kc, tp, h, 2), tv, None, kq_scale, False)
        project(ta, tx0, x1, ready, d, w0)

        # the two products of the feed-forward part; the first leaves its result in the form that the second reads
        wu = pr.matrix(4 * d, d, type_, image)
        eu = pr.epilogue(p.EPI_BIAS | p.EPI_GELU, bias=pr.randn(4 * d, std=0.1))
        ready = 0
        shape = pr.desc(up)
        wd_probe = p.tensor(up, qtype, [4 * d, d])
        if quant and (not few or lib.mi355x_mul_mat_workspace_size(wd_probe, shape) > 0):
            eu.flags |= p.EPI_EMIT_Q8_0 if few else p.EPI_EMIT_F16 | p.EPI_IMAGE_ONLY
            eu.image = ws[1].data_ptr()
            ready = p.MM_WS_READY
        norm_products(tx0, [(wu, tu, eu)])
        project(tu, tx1, x0, ready, 4 * d, w1)
        x0, x1, tx0, tx1 = x1, x0, tx1, tx0

    # the last LayerNorm and the logits
    if quant and few and type_ == "q8_0" and vocab * d * BYTES[type_] >= 32e6:
        tiles = pr.zeros(lib.mi355x_q8_0_tiles_size(d, vocab), dtype=torch.uint8)
        pr.now("mi355x_q8_0_tiles_pack", tte, tiles.data_ptr(), pr.stream)
        w, b = layer_norm(pr, d)
        pr.call("mi355x_norm_mul_mat_q8_0_tiles", tiles.data_ptr(), d, vocab, tx0, tn, EPS, w.data_ptr(), b.data_ptr(), tl, 0, *w0)
    else:
        wl = tte
        if quant and not few:
            half = pr.zeros(vocab, d, dtype=torch.float16)
            pr.now("mi355x_dequantize_row_f16", qtype, te.data_ptr(), half.data_ptr(), vocab * d, pr.stream)
            wl = pr.desc(half)
        ready = norm(tx0)
        pr.call("mi355x_mul_mat", wl, tn, tl, pr.epilogue(act | ready), *w0)
    pr.out = {"logits": logits}


# ---- entry points ---------------------------------------------------------------------------------------------------------

def prepare(case, seed):
    pr = Program(seed)
    {"mel": prepare_mel, "encode": prepare_encode, "decode": prepare_decode}[case["kind"]](pr, case)
    torch.cuda.synchronize()
    return pr


def run(state):
    for fn, args in state.calls:
        status = fn(*args)
        if status:
            state.p.check(status, fn.__name__)
    return state.out
