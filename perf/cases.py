"""The work that is timed: a model's linear-layer steps through the command stream.

A case is one step of a decoder's linear layers, recorded as the planner records it and run
as one submit: the tokens' embeddings gathered from the (tied) vocabulary table, then, a layer,
the attention-shaped projections dim -> attn -> dim, the stacked gate / up projection with its
SiLU product, and the down projection, each pair added to the residual, and for a decode step
the vocabulary projection behind the final RMSNorm. There is no attention between the two
attention-shaped projections (the backend has no such kernel), so every output of every
multiply feeds the next one and nothing is computed that the results do not depend on.

Three ways through the layers, as the planner has them:

  decode  1 .. 8 tokens: matvec_<type> with the RMSNorm prologue, the SILU_PAIR and ACCUMULATE
          epilogues; what comes back is the logits. `id` names the MatvecVariant the tuner
          would have picked ("default", or "matrix_core" for deployments that verify several
          tokens); `wide` opens the device with ZHIP_OPTION_WIDE_DECODE.
  int8    5 .. 512 tokens: the default prefill, quantize_q8 (behind its RMSNorm and SiLU-pair
          modes) and matmul_<type>; what comes back is the hidden state of every token.
  float   5 .. 512 tokens: matmul_q8_0_float / matmul_bf16 / matmul_f16 on a rung of the
          precision ladder with silu_mul between; what comes back is the hidden state of
          every token.

and `layers` = 0 for a single projection (a kernel check, a tuner's probe, a draft head): the
input is written, one decode multiply runs, its output is read.

A step's command words are recorded once and executed again for every step, as a plan's
prebuilt launches are; each pass writes the step's token ids (or inputs) and reads its results.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from zllm_amd import Device, Host, cmd
from zllm_amd import kernels as K
from zllm_amd.kernels import Kernel, TensorType, params as P

EPS = 1e-6
MATRIX_CORE = K.MatvecVariant(wg=512, lanes=64, rows=16)
K_FORMATS = ("q3_k", "q4_k", "q5_k", "q6_k")

# What every case states; a case names what differs.
_DEFAULTS = dict(path="decode", fmt="q8_0", alt="", head="", id="default", wide=False, rung="", tokens=1, dim=1024, attn=2048, ffn=3072,
                 vocab=151936, layers=28)


def listed():
    def case(name, **kw):
        return dict(_DEFAULTS, name=name, **kw)

    big = dict(dim=4096, attn=4096, ffn=14336)
    return [
        # The smallest call: one 1024 -> 3072 projection of one token, where latency is everything.
        case("one_projection_q8", layers=0),
        # A token of a model of 0.6 - 0.8 B weights, all 28 layers: 113 short launches.
        case("decode1_small_q8"),
        # The same model as published in bf16.
        case("decode1_small_bf16", fmt="bf16"),
        # A token through a quarter of an 8 B model, the usual mixed file: Q4_K, half of the down
        # projections and the vocabulary in Q6_K.
        case("decode1_8b_q4", fmt="q4_k", alt="q6_k", head="q6_k", vocab=128256, layers=8, **big),
        # Four speculated tokens verified in one step on the id that the tuner picks for it.
        case("verify4_8b_q4", fmt="q4_k", alt="q6_k", head="q6_k", vocab=128256, layers=8, id="matrix_core", tokens=4, **big),
        # Two tokens (one drafted) on the default id, a middle-sized model with a vocabulary that
        # is no multiple of anything, Q5_K.
        case("decode2_mid_q5", fmt="q5_k", alt="q6_k", head="q5_k", tokens=2, dim=2560, attn=4096, ffn=9728, vocab=50257, layers=12),
        # Eight sequences decoded together: f16 weights read once for all of them.
        case("decode8_mid_f16", fmt="f16", wide=True, tokens=8, dim=2048, attn=2048, ffn=8192, vocab=32003, layers=8),
        # The scheduler's first chunk of a prompt, 64 tokens.
        case("prefill64_8b_q4", path="int8", fmt="q4_k", alt="q6_k", tokens=64, vocab=32000, layers=8, **big),
        # A full prefill step, 512 tokens: the largest work of all.
        case("prefill512_8b_q4", path="int8", fmt="q4_k", alt="q6_k", tokens=512, vocab=32000, layers=8, **big),
        # A full prefill step of the small model, Q8_0.
        case("prefill512_small_q8", path="int8", tokens=512, vocab=32000),
        # A prompt's last, ragged chunk through the smallest files (Q3_K with Q5_K downs).
        case("prefill201_mid_q3", path="int8", fmt="q3_k", alt="q5_k", tokens=201, dim=2560, attn=4096, ffn=9728, vocab=32003, layers=6),
        # Q8_0 on the bf16 matrix cores, where the precision ladder allows it.
        case("prefill512_8b_q8_bf16", path="float", rung="bf16_mfma", tokens=512, vocab=32000, layers=6, **big),
    ]


def _log(rng, low, high):
    return math.exp(rng.uniform(math.log(low), math.log(high)))


def draw(rng):
    while True:
        path = rng.choice(("one", "decode", "decode", "decode", "int8", "int8", "int8", "float"))
        c = dict(_DEFAULTS)
        unit = 256
        if path == "float":
            c["fmt"] = rng.choice(("q8_0", "q8_0", "bf16", "f16"))
            c["rung"] = rng.choice(("fp16_single", "fp16_compensated", "bf16_mfma") if c["fmt"] == "q8_0" else ("fp16_single",))
            unit = 128 if c["fmt"] == "q8_0" else 64
        elif path == "int8":
            c["fmt"] = rng.choice(("q8_0",) + K_FORMATS)
        else:
            c["fmt"] = rng.choice(("q8_0", "bf16", "f16") + K_FORMATS)
        if c["fmt"] in K_FORMATS:
            c["alt"] = rng.choice(("", "q5_k", "q6_k"))
            c["head"] = rng.choice(("", "q6_k")) if path == "decode" else ""
        elif c["fmt"] == "q8_0" and path != "float":
            unit = 64
        elif path != "float":
            unit = 128
        c["dim"] = unit * round(_log(rng, 768, 5120) / unit)
        c["attn"] = unit * round(c["dim"] * rng.uniform(0.8, 2.0) / unit)
        c["ffn"] = unit * round(c["dim"] * rng.uniform(2.2, 4.0) / unit)
        c["vocab"] = int(_log(rng, 5000, 152000)) if path == "decode" else int(_log(rng, 5000, 50000))
        c["layers"] = 0 if path == "one" else rng.randint(4, 24)
        if path in ("one", "decode"):
            c["path"] = "decode"
            c["tokens"] = rng.choice((1, 1, 1, 2, 2, 3, 4, 5, 8))
            if c["fmt"] in ("bf16", "f16"):
                c["wide"] = c["tokens"] > 1
            elif c["tokens"] > 2:
                c["id"] = rng.choice(("default", "matrix_core", "matrix_core"))
        else:
            c["path"] = path
            c["tokens"] = rng.choice((64, 128, 256, 512, int(_log(rng, 9, 512)), int(_log(rng, 9, 512))))
        w = work(c)
        stored = sum(n * k for _, n, k in _matrices(c)) * 2.2
        if w["flops"] <= work(_LARGEST)["flops"] * (0.5 if c["path"] == "float" else 0.7) and stored <= 4e9 and (c["rung"] != "fp16_compensated" or w["flops"] < 5e11):
            return c


def _formats(c):
    """The storage type of each role in layer i: (projections, down, vocabulary)."""
    body = c["fmt"]
    return body, c["alt"] or body, c["head"] or body


def _matrices(c):
    """(storage type, rows, columns) of every matrix a pass multiplies by, in order."""
    body, alt, head = _formats(c)
    if c["layers"] == 0:
        return [(body, c["ffn"], c["dim"])]
    out = []
    for i in range(c["layers"]):
        out += [(body, c["attn"], c["dim"]), (body, c["dim"], c["attn"]), (body, 2 * c["ffn"], c["dim"]), (alt if i % 2 else body, c["dim"], c["ffn"])]
    if c["path"] == "decode":
        out.append((head, c["vocab"], c["dim"]))
    return out


def _file_bytes(fmt, n, k):
    e, b = K.LAYOUT[TensorType[fmt]]
    return n * k // e * b


def work(case):
    c = dict(_DEFAULTS, **case)
    mats = _matrices(c)
    t = c["tokens"]
    size = sum(_file_bytes(f, n, k) for f, n, k in mats)
    flops = 2.0 * t * sum(n * k for _, n, k in mats)
    if c["layers"] == 0:
        return {"bytes": size + 4 * t * (c["dim"] + c["ffn"]), "flops": flops}
    norms = 4 * c["dim"] * (0 if c["path"] == "float" else 2 * c["layers"] + (c["path"] == "decode"))
    _, _, head = _formats(c)
    out = 4 * t * (c["vocab"] if c["path"] == "decode" else c["dim"])
    return {"bytes": size + norms + 4 * t + t * _file_bytes(head, 1, c["dim"]) + out, "flops": flops}


def tolerance(case):
    """Four times what a pass differs by from the same pass worked out in 64 bits, every rounding
    that the path itself prescribes kept (measured over the listed cases and models of 24 layers)."""
    c = dict(_DEFAULTS, **case)
    if c["path"] == "int8":
        # An activation within an f32 rounding of a half moves by one of its 127 steps, and a
        # layer later that has moved a few in a hundred of the others: the layers' roundings
        # are then independent ones (0.8e-2 over eight layers, and over twenty-four).
        return {"rel": 0.03, "max": 0.3}
    if c["path"] == "float":
        # The same with the rung's own rounding of every input: 8 bits, 11 bits, or 22.
        return {"bf16_mfma": {"rel": 0.025, "max": 0.14}, "fp16_single": {"rel": 0.008, "max": 0.15},
                "fp16_compensated": {"rel": 5e-6, "max": 5e-5}}[c["rung"]]
    return {"rel": 6e-6, "max": 3e-5}


_LARGEST = dict(_DEFAULTS, path="int8", fmt="q4_k", alt="q6_k", tokens=512, vocab=32000, layers=8, dim=4096, attn=4096, ffn=14336)


# ---- inputs ------------------------------------------------------------------------------


class _Make:
    """Seeded tensors in GGUF storage formats, drawn on the GPU and handed over as host bytes."""

    def __init__(self, seed):
        self.dev = torch.device("cuda") if torch.cuda.is_available() else torch.device("cpu")
        self.g = torch.Generator(device=self.dev).manual_seed(seed)

    def bytes(self, *shape):
        words = torch.randint(-(2**31), 2**31 - 1, (-(-math.prod(shape) // 4),), dtype=torch.int32, device=self.dev, generator=self.g)
        return words.view(torch.uint8)[: math.prod(shape)].view(*shape)

    def normal(self, *shape):
        return torch.randn(*shape, device=self.dev, generator=self.g)

    def halves(self, value):
        return value.to(torch.float16).view(torch.uint8).view(*value.shape, 2)

    def rows(self, fmt, n, k, std):
        """n rows of k weights of root mean square ~std as the file stores them: block scales
        within a quarter of each other, minimums about the middle of a block's range."""
        e, b = K.LAYOUT[TensorType[fmt]]
        if fmt in ("bf16", "f16"):
            w = (self.normal(n, k) * std).to(torch.bfloat16 if fmt == "bf16" else torch.float16)
            return w.view(torch.uint8).reshape(-1).cpu().numpy()
        blocks = n * k // e
        out = self.bytes(blocks, b)
        spread = 1 + 0.125 * self.normal(blocks)
        if fmt == "q8_0":
            out[:, 0:2] = self.halves(spread * (std / 73.9))
        elif fmt in ("q4_k", "q5_k"):
            mid, rms = (7.5, 4.61) if fmt == "q4_k" else (15.5, 9.23)
            sc = 32 + out[:, 4:12] % 32
            m = (sc.to(torch.int16) + (out[:, 12:16].repeat(1, 2) % 7).to(torch.int16) - 3).clamp(0, 63).to(torch.uint8)
            d = spread * (std / (48.4 * rms))
            out[:, 0:2], out[:, 2:4] = self.halves(d), self.halves(d * mid)
            out[:, 4:8] = sc[:, 0:4] | ((sc[:, 4:8] >> 4) << 6)
            out[:, 8:12] = m[:, 0:4] | ((m[:, 4:8] >> 4) << 6)
            out[:, 12:16] = (sc[:, 4:8] & 15) | ((m[:, 4:8] & 15) << 4)
        elif fmt == "q6_k":
            s = out[:, 192:208].view(torch.int8)
            s[:] = torch.where(s < 0, s // 2 - 63, s // 2 + 63).clamp(-127, 127)
            out[:, 208:210] = self.halves(spread * (std / (96.6 * 18.5)))
        else:  # q3_k
            out[:, 108:110] = self.halves(spread * (std / (18.5 * 2.29)))
        return out.reshape(-1).cpu().numpy()


class State:
    """A device, the step's weights and buffers on it, and its command words."""

    def __init__(self, case, seed):
        c = self.c = dict(_DEFAULTS, **case)
        self.make = _Make(seed)
        self.device = Device.open(0, Device.WIDE_DECODE if c["wide"] else 0)
        self.host = Host(self.device)
        self.rec = cmd.Recorder()
        self.set = K.Set.create(self.rec)
        if c["rung"]:
            self.set.select_prefill(self.rec, K.Prefill[c["rung"]])
        self.token = 0
        self.build()
        self.make = None

    def execute(self):
        self.token += 1
        self.rec.submit(self.token)
        self.host.execute(self.rec.batch(), [])
        self.rec.clear()

    def buffer(self, size):
        size = (size + 15) & ~15
        return K.Arg(self.rec.create_buffer(size, cmd.Usage.storage | cmd.Usage.copy_dst | cmd.Usage.copy_src), size)

    def floats(self, n):
        return self.buffer(4 * n)

    def upload(self, data):
        raw = np.ascontiguousarray(data).reshape(-1).view(np.uint8)
        if raw.size % 4:
            raw = np.concatenate([raw, np.zeros(-raw.size % 4, np.uint8)])
        a = self.buffer(raw.size)
        self.rec.write_buffer(a.buffer, 0, raw)
        return a

    def weights(self, fmt, n, k, gain):
        """A matrix laid out as the kernels read it, as the loader does it."""
        t = TensorType[fmt]
        a = self.upload(self.make.rows(fmt, n, k, gain / math.sqrt(k)))
        if not K.is_half(t) and K.needs_layout(t):
            raw, a = a, self.buffer(n * K.row_bytes(t, k))
            K.Launcher(self.rec, self.set).layout(t, raw, a, n, k)
            self.rec.destroy(cmd.Kind.buffer, raw.buffer)
        self.execute()
        return a

    def norm(self, k):
        return self.upload((1 + 0.1 * self.make.normal(k)).cpu().numpy().astype(np.float32))

    def build(self):
        c, t = self.c, self.c["tokens"]
        dim, attn, ffn = c["dim"], c["attn"], c["ffn"]
        body, alt, head_fmt = _formats(c)
        self.b = K.Builder(self.rec, self.set)
        self.launches = []
        if c["layers"] == 0:
            self.input = self.make.normal(t, dim).cpu().numpy().astype(np.float32)
            x, out = self.floats(t * dim), self.floats(t * ffn)
            w = self.weights(body, ffn, dim, 1.0)
            self.vector(body, w, ffn, dim, x, out)
            self.result = np.empty((t, ffn), np.float32)
            return self.record(x, out)
        rows = torch.randint(0, c["vocab"], (t,), device=self.make.dev, generator=self.make.g)
        self.input = rows.cpu().numpy().astype(np.uint32)
        ids, x, a, act = self.buffer(4 * t), self.floats(t * dim), self.floats(t * attn), self.floats(t * ffn)
        # (a vocabulary projection gives logits of about one; a prefill step only gathers from the table)
        head = self.weights(head_fmt, c["vocab"], dim, 1.0 if c["path"] == "decode" else math.sqrt(dim))
        self.add(K.weight_kernel("embed", TensorType[head_fmt]), P.EmbedBf16(dim=dim, row0=0, chunk_rows=c["vocab"]), [ids, head, x], (t, 1, 1))
        if c["path"] != "decode":
            self.gu = self.floats(t * 2 * ffn)
            self.qx, self.dx = self.buffer(t * max(dim, attn, ffn)), self.floats(t * max(dim, attn, ffn) // 32)
        out_gain = 1 / math.sqrt(2 * c["layers"])
        for i in range(c["layers"]):
            down_fmt = alt if i % 2 else body
            w_in, w_out = self.weights(body, attn, dim, 1.0), self.weights(body, dim, attn, out_gain)
            w_gu, w_down = self.weights(body, 2 * ffn, dim, 1.0), self.weights(down_fmt, dim, ffn, 2 * out_gain)
            if c["path"] == "decode":
                self.vector(body, w_in, attn, dim, x, a, norm=self.norm(dim))
                self.vector(body, w_out, dim, attn, a, x, accumulate=True)
                self.vector(body, w_gu, ffn, dim, x, act, norm=self.norm(dim), pair=True)
                self.vector(down_fmt, w_down, dim, ffn, act, x, accumulate=True)
            elif c["path"] == "int8":
                self.tiled(body, w_in, attn, dim, x, a, norm=self.norm(dim))
                self.tiled(body, w_out, dim, attn, a, x, accumulate=True)
                self.tiled(body, w_gu, 2 * ffn, dim, x, self.gu, norm=self.norm(dim))
                self.tiled(down_fmt, w_down, dim, ffn, self.gu, x, accumulate=True, pair=True)
            else:
                self.plain(body, w_in, attn, dim, x, a)
                self.plain(body, w_out, dim, attn, a, x, accumulate=True)
                self.plain(body, w_gu, 2 * ffn, dim, x, self.gu)
                self.add(Kernel.silu_mul, P.SiluMul(t * ffn, ffn), [self.gu, act], K.elementwise(t * ffn))
                self.plain(down_fmt, w_down, dim, ffn, act, x, accumulate=True)
        if c["path"] != "decode":
            self.result = np.empty((t, dim), np.float32)
            return self.record(ids, x)
        logits = self.floats(t * c["vocab"])
        self.vector(head_fmt, head, c["vocab"], dim, x, logits, norm=self.norm(dim))
        self.result = np.empty((t, c["vocab"]), np.float32)
        self.record(ids, logits)

    def add(self, kernel, p, args, grid, variant=None):
        if variant is None:
            self.launches.append(self.b.add(kernel, p, args, K.Grid.fixed_(grid)))
        else:
            self.launches.append(self.b.add_matvec(kernel, variant, p, args, K.Grid.fixed_(grid)))

    def vector(self, fmt, w, n, k, x, out, norm=None, pair=False, accumulate=False):
        """A decode multiply (Mm.vector)."""
        t = TensorType[fmt]
        kernel = K.weight_kernel("matvec", t)
        variant = None if K.is_half(t) or self.c["id"] == "default" else MATRIX_CORE
        per_group = K.matvec_rows if variant is None else variant.group_rows()
        p = P.MatvecBf16(n=n, k=k, col0=0, out_stride=n, eps=EPS, norm=norm is not None, accumulate=accumulate, silu_pair=pair, half=n if pair else 0)
        self.add(kernel, p, [x, w, out, norm or w], (K.div_ceil(n, per_group), self.c["tokens"], 1), variant)

    def tiled(self, fmt, w, n, k, x, out, norm=None, pair=False, accumulate=False):
        """The default prefill multiply (Mm.tiled): the inputs rounded to 8-bit blocks, then the product."""
        t, rows = TensorType[fmt], self.c["tokens"]
        mode = 1 if norm is not None else 2 if pair else 0
        self.add(Kernel.quantize_q8, P.QuantizeQ8(k=k, block=K.act_block(t), mode=mode, eps=EPS), [x, self.qx, self.dx, norm or x], (K.div_ceil(k, 256), rows, 1))
        self.add(K.weight_kernel("matmul", t), P.MatmulQuant(rows=rows, n=n, k=k, col0=0, out_stride=n, accumulate=int(accumulate), k_slice=-(-k // 32) * 32),
                 [self.qx, w, out, self.dx], (K.div_ceil(n, K.matmul_quant_tile_n), K.div_ceil(rows, K.matmul_quant_tile_t), 1))

    def plain(self, fmt, w, n, k, x, out, accumulate=False):
        """A prefill multiply on a rung of the precision ladder."""
        rows = self.c["tokens"]
        grid = (K.div_ceil(n, K.matmul_tile_n), K.div_ceil(rows, K.matmul_tile_t), 1)
        if fmt == "q8_0":
            self.add(Kernel.matmul_q8_0_float, P.MatmulQuant(rows=rows, n=n, k=k, col0=0, out_stride=n, accumulate=int(accumulate), k_slice=k), [x, w, out], grid)
        else:
            self.add(Kernel["matmul_" + fmt], P.MatmulBf16(rows=rows, n=n, k=k, col0=0, out_stride=n, accumulate=int(accumulate)), [x, w, out], grid)

    def record(self, source, out):
        """The step's command words, once for every pass."""
        self.b.finish()
        self.execute()
        self.rec.write_buffer(source.buffer, 0, self.input)
        for l in self.launches:
            l.record(self.rec, K.Extent(rows=self.c["tokens"]))
        self.rec.read_buffer(1, out.buffer, 0, self.result)
        self.rec.submit(2)
        self.words = self.rec.batch()


def prepare(case, seed):
    return State(case, seed)


def run(state):
    state.host.execute(state.words, [])
    return state.result
