"""A multiply on a float rung whose activations the dispatch right before it wrote reads them
packed by that dispatch: the same bits as with every dispatch in a submit of its own, where
each multiply packs its activations itself. How many do so is counted: every one that may, and none that may not."""
import numpy as np
import pytest

from gpucheck import Ctx
from zllm_amd import Device, synth
from zllm_amd import kernels as K
from zllm_amd.kernels import Kernel, TensorType, params as P

pytestmark = pytest.mark.gpu


class Chain:
    """x -> a -> x (added) -> gu -> act -> x (added) -> out, five multiplies and the SwiGLU between two of them."""

    def __init__(self, c: Ctx, weights, rung, rows, dim, attn, ffn, change):
        self.c = c
        c.set.select_prefill(c.rec, K.Prefill[rung])
        b = K.Builder(c.rec, c.set)
        self.launches = []
        self.x, self.a, self.gu, self.act, self.out = (c.output(rows * n + 8) for n in (dim, attn + 4, 2 * ffn, ffn, 96))

        def multiply(n, k, x, out, accumulate=0, rows=rows, pad=0):
            grid = K.Grid.fixed_((K.div_ceil(n, K.matmul_tile_n), K.div_ceil(rows, K.matmul_tile_t), 1))
            if weights == "q8_0":
                w = c.gpu_weights(TensorType.q8_0, synth.q8_0_rows(synth.rng(n + k), n, k), k)
                self.launches.append(b.add(Kernel.matmul_q8_0_float, P.MatmulQuant(rows=rows, n=n, k=k, col0=0, out_stride=n + pad, accumulate=accumulate, k_slice=k), [x, w, out], grid))
            else:
                bits = synth.to_bf16_bits(c.random(n * k, 0.1)) if weights == "bf16" else c.random(n * k, 0.1).astype(np.float16).view(np.uint16)
                self.launches.append(b.add(Kernel["matmul_" + weights], P.MatmulBf16(rows=rows, n=n, k=k, col0=0, out_stride=n + pad, accumulate=accumulate), [x, c.upload(bits), out], grid))

        fewer = rows - 1 if change == "rows" else rows
        multiply(attn, dim, self.x, self.a, pad=4 if change == "stride" else 0)
        multiply(dim, attn, self.a, self.x, accumulate=1, rows=fewer)
        multiply(2 * ffn, dim, self.x, self.gu)
        self.launches.append(b.add(Kernel.silu_mul, P.SiluMul(rows * ffn, ffn), [self.gu, self.act], K.Grid.fixed_(K.elementwise(fewer * ffn))))
        multiply(dim, ffn, self.act, self.x, accumulate=1, rows=rows)
        multiply(96, dim, self.x, self.out)
        b.finish()
        c.flush()

    def run(self, x, apart):
        """The bytes of every buffer; handed: the packed activations handed over meanwhile."""
        c = self.c
        before = c.host.handed_over()
        c.rec.write_buffer(self.x.buffer, 0, x.reshape(-1).view(np.uint8))
        c.flush()
        for l in self.launches:
            l.record(c.rec, K.Extent(rows=1))
            if apart:
                c.flush()
        c.flush()
        after = c.host.handed_over()
        assert after[1] == before[1]
        self.handed = after[0] - before[0]
        return [c.read(t).tobytes() for t in (self.x, self.a, self.gu, self.act, self.out)]


@pytest.mark.parametrize("weights,rung,rows,dim,attn,ffn,change,handed", [
    ("q8_0", "bf16_mfma", 19, 256, 384, 640, "", 4),       # whole 128-deep steps
    ("q8_0", "bf16_mfma", 133, 256, 320, 352, "", 4),      # a ragged k between
    ("q8_0", "bf16_mfma", 67, 128, 8192, 256, "", 4),      # 128-row tiles
    ("q8_0", "bf16_mfma", 520, 256, 256, 5504, "", 4),     # more tokens than a planner records
    ("q8_0", "bf16_mfma", 1, 256, 256, 256, "", 4),
    ("q8_0", "bf16_mfma", 35, 256, 384, 640, "rows", 1),
    ("q8_0", "bf16_mfma", 35, 256, 384, 640, "stride", 3),
    ("bf16", "bf16_mfma", 300, 320, 448, 704, "", 4),
    ("f16", "fp16_single", 133, 256, 320, 384, "", 4),
    ("q8_0", "fp16_single", 260, 256, 512, 384, "", 4),
    ("q8_0", "fp16_compensated", 35, 256, 384, 640, "", 4),
    ("bf16", "fp16_compensated", 133, 192, 320, 448, "rows", 1),
])
def test_activations_packed_by_their_writer(weights, rung, rows, dim, attn, ffn, change, handed):
    devices = [Device.open(0), Device.open(0, Device.NO_REPLAY)]
    together, apart = (Chain(Ctx(d), weights, rung, rows, dim, attn, ffn, change) for d in devices)
    g = synth.rng(rows)
    for i in range(5):  # the first ones launch by launch, the later ones replayed
        x = np.zeros((rows, dim), np.float32)
        x[:] = synth.activations(g, rows, dim) * 0.1
        x[0, :3] = [np.inf, 7e4, 1e-7] if i == 3 else [1.0009765625 + 2.0 ** -12, -7e4, 1e-7]
        assert together.run(x, False) == apart.run(x, True)
        assert (together.handed, apart.handed) == (handed, 0)
    for d in devices:
        d.deinit()


@pytest.mark.parametrize("rung,rows,k,handed", [("bf16_mfma", 504, 65664, 1), ("bf16_mfma", 512, 65664, 0), ("fp16_compensated", 504, 32896, 1), ("fp16_compensated", 512, 32896, 0)])
def test_more_activations_than_their_place_holds_are_packed_by_their_reader(rung, rows, k, handed):
    """64 MB of them, in one plane or in two."""
    got = []
    for apart in (False, True):
        c = Ctx(Device.open(0))
        c.set.select_prefill(c.rec, K.Prefill[rung])
        b = K.Builder(c.rec, c.set)
        x, y, out = c.upload(c.random(rows * 128, 1)), c.output(rows * k), c.output(rows * 32)
        launches = []
        for n, depth, source, to in ((k, 128, x, y), (32, k, y, out)):
            w = c.gpu_weights(TensorType.q8_0, synth.q8_0_rows(synth.rng(n), n, depth), depth)
            launches.append(b.add(Kernel.matmul_q8_0_float, P.MatmulQuant(rows=rows, n=n, k=depth, col0=0, out_stride=n, k_slice=depth), [source, w, to],
                                  K.Grid.fixed_((K.div_ceil(n, K.matmul_tile_n), K.div_ceil(rows, K.matmul_tile_t), 1))))
        b.finish()
        c.flush()
        for l in launches:
            l.record(c.rec, K.Extent(rows=1))
            if apart:
                c.flush()
        c.flush()
        assert c.host.handed_over() == (0 if apart else handed, 0)
        got.append(c.read(out).tobytes())
        c.device.deinit()
    assert got[0] == got[1]
