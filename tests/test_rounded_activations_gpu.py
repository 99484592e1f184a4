"""An int8 Q8_0 multiply whose outputs the next dispatch rounds for another such multiply rounds
them itself: the same bits in every buffer as with each dispatch in a submit of its own, where
quantize_q8 is launched. How many do so is counted: every one that may, and none that may not."""
import numpy as np
import pytest

from gpucheck import Ctx
from zllm_amd import Device, cmd, synth
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
        """The bytes of every buffer; handed: the roundings handed over meanwhile."""
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
        assert after[0] == before[0]
        self.handed = after[1] - before[1]
        return [c.read(t).tobytes() for t in (self.x, self.a, self.gu, self.qx, self.dx, self.out, self.more)]


@pytest.mark.parametrize("rows,dim,attn,ffn,change,handed", [
    (19, 256, 384, 640, "", 4),
    (133, 256, 128, 384, "", 4),    # a last tile of five tokens
    (64, 128, 1152, 256, "", 4),    # a matrix of two tiles, the rounding carried home in several turns
    (512, 1024, 2048, 3072, "", 4), # tiles of 64 tokens
    (201, 2560, 4096, 1280, "", 4),
    (33, 256, 320, 672, "", 0),     # k of no whole 128s between: the general kernel
    (1, 128, 128, 128, "", 4),
    (35, 256, 384, 640, "rows", 2),
    (35, 256, 384, 640, "stride", 3),
    (35, 256, 384, 640, "scales", 0),
])
def test_activations_rounded_by_their_writer(rows, dim, attn, ffn, change, handed):
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
        assert (together.handed, apart.handed) == (handed, 0)
    for d in devices:
        d.deinit()


def test_under_a_profile_every_dispatch_rounds_for_itself():
    devices = [Device.open(0), Device.open(0, Device.NO_REPLAY)]
    together, apart = (Chain(Ctx(d), 19, 256, 384, 640, "") for d in devices)
    host = together.c.host
    for i, profiled in enumerate((False, False, True, False, True, True, False)):
        x = synth.activations(synth.rng(i), 19, 256) * np.float32(0.1)
        if profiled:
            host.start_profile()
        assert together.run(x, False) == apart.run(x, True)
        assert together.handed == (0 if profiled else 4)
        if profiled:
            assert sum(t.count for t in host.timings().totals.values()) == len(together.launches)
            host.stop_profile()
    for d in devices:
        d.deinit()


class Pair:
    """x -> y, its rounding, y -> out, with the ranges of every dispatch and the buffer of its parameters to choose."""

    def __init__(self, c: Ctx, rows, k, n, last, fillers=0):
        self.c, self.rows, self.k, self.n, self.last = c, rows, k, n, last
        self.x, self.qx, self.dx = c.upload(c.random(rows * k, 1)), c.output(rows * k // 4), c.output(rows * k // 32)
        self.y, self.out = c.output(rows * n), c.output(rows * last)
        self.q, self.d = c.output(rows * n // 4), c.output(rows * n // 32)
        self.w = c.gpu_weights(TensorType.q8_0, synth.q8_0_rows(synth.rng(1), n, k), k)
        self.w2 = c.gpu_weights(TensorType.q8_0, synth.q8_0_rows(synth.rng(2), last, n), n)
        self.stride, self.col0 = last, 0
        self.params = [None, None, None]
        self.others = [c.output(64) for _ in range(fillers)]

    def run(self, apart):
        c, rows = self.c, self.rows
        c.launcher().launch(Kernel.quantize_q8, P.QuantizeQ8(k=self.k, block=32, mode=0, eps=0), [self.x, self.qx, self.dx, self.x], (K.div_ceil(self.k, 256), rows, 1))
        c.flush()
        tiles = lambda n: (K.div_ceil(n, K.matmul_quant_tile_n), K.div_ceil(rows, K.matmul_quant_tile_t), 1)
        three = (
            (Kernel.matmul_q8_0, P.MatmulQuant(rows=rows, n=self.n, k=self.k, col0=0, out_stride=self.n, k_slice=self.k), [self.qx, self.w, self.y, self.dx], tiles(self.n)),
            (Kernel.quantize_q8, P.QuantizeQ8(k=self.n, block=32, mode=0, eps=0), [self.y, self.q, self.d, self.y], (K.div_ceil(self.n, 256), rows, 1)),
            (Kernel.matmul_q8_0, P.MatmulQuant(rows=rows, n=self.last, k=self.n, col0=self.col0, out_stride=self.stride, k_slice=self.n), [self.q, self.w2, self.out, self.d], tiles(self.last)),
        )
        groups = []
        for (kernel, p, args, grid), at in zip(three, self.params):
            raw = np.frombuffer(p.pack(), np.uint8)
            at = at or K.Arg(c.rec.create_buffer(raw.size, cmd.Usage.uniform | cmd.Usage.copy_dst), raw.size)
            c.rec.write_buffer(at.buffer, at.offset, raw)
            groups.append((c.set.pipelines[kernel], grid, K.bind_group(c.rec, c.set.pipelines[kernel], K.Arg(at.buffer, raw.size, offset=at.offset), args)))
        c.flush()
        before = c.host.handed_over()[1]
        for pipeline, grid, group in groups:
            c.rec.dispatch(pipeline, grid, [group])
            if apart:
                c.flush()
        c.flush()
        self.handed = c.host.handed_over()[1] - before
        return [c.read(t).tobytes() for t in (self.y, self.out, self.q, self.d)]


def both(change, shape=(19, 256, 384, 96)):
    """Whether the rounding was handed over, the same bytes either way."""
    devices = [Device.open(0), Device.open(0, Device.NO_REPLAY)]
    together, apart = (Pair(Ctx(d), *shape) for d in devices)
    for p in (together, apart):
        change(p)
    handed = []
    for _ in range(2):
        assert together.run(False) == apart.run(True)
        handed.append(together.handed)
        assert apart.handed == 0
    for d in devices:
        d.deinit()
    assert handed in ([0, 0], [1, 1])
    return handed[0] == 1


def test_a_rounding_that_overlaps_what_the_multiplies_hold_is_not_handed_over():
    """Placed ahead of the second multiply's first column but within its output range, among the first one's weights (which it has
    read by then) and among the second one's, and next to each of them."""
    def ahead_of_the_outputs(gap):
        def change(p):
            size = p.rows * p.n
            p.col0 = size // 4
            p.stride = p.col0 + p.last
            whole = p.c.output(gap // 4 + p.rows * p.stride)
            p.q, p.out = K.Arg(whole.buffer, size), K.Arg(whole.buffer, whole.size - gap, offset=gap)
        return change

    def among_the_weights(name, rows, behind):
        def change(p):
            k = p.k if name == "w" else p.n
            raw, size = K.row_bytes(TensorType.q8_0, k) * rows, p.rows * p.n
            small, whole = getattr(p, name), p.c.output((raw + 256 + size) // 4)
            p.c.rec.copy_buffer(small.buffer, 0, whole.buffer, 0, min(raw, small.size))
            p.c.flush()
            start = (raw + 255) // 256 * 256 if behind else raw // 2 // 256 * 256
            assert raw % 4 == 0 and start + size <= whole.size and (behind or start + size <= raw)
            setattr(p, name, K.Arg(whole.buffer, raw))
            p.q = K.Arg(whole.buffer, size, offset=start)
        return change

    assert both(lambda p: None)
    assert not both(ahead_of_the_outputs(0))
    assert both(ahead_of_the_outputs(7424))  # (the rounding's 7296 bytes, to the next 256)
    assert not both(among_the_weights("w", 384, False))
    assert both(among_the_weights("w", 384, True))
    assert not both(among_the_weights("w2", 96, False))
    assert both(among_the_weights("w2", 96, True))


def test_no_rounding_is_handed_over_past_a_buffer_that_holds_parameters():
    """A buffer that one of the three dispatches writes and one of the later two has its parameters in: what the
    host would look at ahead of time may not be what the dispatch finds."""
    def shared(name, floats, which):
        def change(p):
            size = 4 * floats(p)
            buffer = p.c.rec.create_buffer(size + 512, cmd.Usage.uniform | cmd.Usage.storage | cmd.Usage.copy_dst | cmd.Usage.copy_src)
            setattr(p, name, K.Arg(buffer, size, offset=256))
            if which is not None:
                p.params[which] = K.Arg(buffer, 256)
        return change

    sizes = {"y": lambda p: p.rows * p.n, "q": lambda p: p.rows * p.n // 4, "d": lambda p: p.rows * p.n // 32}
    for name, floats in sizes.items():
        assert both(shared(name, floats, None))
        for which in (1, 2):
            assert not both(shared(name, floats, which)), (name, which)


@pytest.mark.parametrize("rows,handed", [(480, True), (512, False)])
def test_a_rounding_of_more_than_its_place_holds_is_not_handed_over(rows, handed):
    """64 MB: 480 tokens of 118,784 values and their scales, not 512."""
    assert both(lambda p: None, (rows, 128, 118784, 32)) == handed
