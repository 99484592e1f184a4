"""An int8 Q8_0 multiply whose outputs the next dispatch rounds for another such multiply rounds
them itself: the same bits in every buffer as with each dispatch in a submit of its own, where
quantize_q8 is launched."""
import numpy as np
import pytest

from gpucheck import Ctx
from zllm_amd import Device, synth
from zllm_amd import kernels as K
from zllm_amd.kernels import Kernel, TensorType, params as P

pytestmark = pytest.mark.gpu


class Chain:
    """A layer: x -> a -> x (added) behind the RMSNorm, then gate | up -> x (added) through the SiLU pair, then x -> out and
    once more from the last rounding."""

    def __init__(self, c: Ctx, rows, dim, attn, ffn, change):
        self.c, self.rows, self.dim = c, rows, dim
        b = K.Builder(c.rec, c.set)
        self.launches = []
        self.x, self.a, self.gu, self.out, self.more = (c.output(rows * n + 8) for n in (dim, attn + 4, 2 * ffn, 96, 40))
        widest = max(dim, attn, ffn)
        self.qx, self.dx = c.output((rows * widest + 3) // 4 + 4), c.output(rows * widest // 32 + 4)
        norm = c.upload(c.random(dim, 0.5) + 1)

        def rounded(k, x, mode=0, rows=rows):
            # (with scales that lie off 16-byte lines every dispatch does its own work)
            dx = K.Arg(self.dx.buffer, self.dx.size - 4, offset=4) if change == "scales" else self.dx
            self.launches.append(b.add(Kernel.quantize_q8, P.QuantizeQ8(k=k, block=32, mode=mode, eps=1e-6), [x, self.qx, dx, norm if mode == 1 else x], K.Grid.fixed_((K.div_ceil(k, 256), rows, 1))))
            return dx

        def multiply(n, k, dx, out, accumulate=0, rows=rows, pad=0):
            w = c.gpu_weights(TensorType.q8_0, synth.q8_0_rows(synth.rng(n + k), n, k), k)
            p = P.MatmulQuant(rows=rows, n=n, k=k, col0=0, out_stride=n + pad, accumulate=accumulate, k_slice=k)
            self.launches.append(b.add(Kernel.matmul_q8_0, p, [self.qx, w, out, dx], K.Grid.fixed_((K.div_ceil(n, K.matmul_quant_tile_n), K.div_ceil(rows, K.matmul_quant_tile_t), 1))))

        fewer = rows - 1 if change == "rows" else rows
        multiply(attn, dim, rounded(dim, self.x, 1), self.a, pad=4 if change == "stride" else 0)
        multiply(dim, attn, rounded(attn, self.a), self.x, 1, rows=fewer)
        multiply(2 * ffn, dim, rounded(dim, self.x), self.gu)
        multiply(dim, ffn, rounded(ffn, self.gu, 2), self.x, 1)
        dx = rounded(dim, self.x)
        multiply(96, dim, dx, self.out)
        multiply(40, dim, dx, self.more)
        b.finish()
        c.flush()

    def run(self, x, apart):
        c = self.c
        c.rec.write_buffer(self.x.buffer, 0, x.reshape(-1).view(np.uint8))
        c.flush()
        for l in self.launches:
            l.record(c.rec, K.Extent(rows=1))
            if apart:
                c.flush()
        c.flush()
        return [c.read(t).tobytes() for t in (self.x, self.a, self.gu, self.qx, self.dx, self.out, self.more)]


@pytest.mark.parametrize("rows,dim,attn,ffn,change", [
    (19, 256, 384, 640, ""),
    (133, 256, 128, 384, ""),    # a last tile of five tokens
    (64, 128, 1152, 256, ""),    # a matrix of two tiles, the rounding carried home in several turns
    (512, 1024, 2048, 3072, ""), # tiles of 64 tokens
    (201, 2560, 4096, 1280, ""),
    (33, 256, 320, 672, ""),     # k of no whole 128s between: the general kernel
    (1, 128, 128, 128, ""),
    (35, 256, 384, 640, "rows"),
    (35, 256, 384, 640, "stride"),
    (35, 256, 384, 640, "scales"),
])
def test_activations_rounded_by_their_writer(rows, dim, attn, ffn, change):
    devices = [Device.open(0), Device.open(0, Device.NO_REPLAY)]
    together, apart = (Chain(Ctx(d), rows, dim, attn, ffn, change) for d in devices)
    g = synth.rng(rows)
    for i in range(5):  # the first ones launch by launch, the later ones replayed
        x = np.zeros((rows, dim), np.float32)
        x[:] = synth.activations(g, rows, dim) * 0.1
        x[0, :3] = [np.inf, 7e4, 1e-7] if i == 3 else [1.0009765625 + 2.0 ** -12, -7e4, 1e-7]
        if i == 2:
            x[rows // 2] = 0
        assert together.run(x, False) == apart.run(x, True)
    for d in devices:
        d.deinit()
