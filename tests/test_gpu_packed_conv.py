"""Plan nodes on a packed filter (kxc_hip_plan_add_conv2d_packed): the three-part kernels for 3x3 stride-2 convolutions, with
and without the second output, and for 7x7 stride-2 convolutions of three channels, with and without the column maxima, at the
edges of their tiles, against float64; their values that are not finite; their filters.  And single calls on a filter that
they pack themselves."""
import ctypes
import threading

import numpy as np
import pytest
import torch

from gpu_util import assert_bit_exact, dev, host

pytestmark = pytest.mark.gpu


def _want(x, w, bias, residual, relu, stride, pad):
    t = lambda a: torch.from_numpy(a).double()
    y = torch.nn.functional.conv2d(t(x), t(w), t(bias) if bias is not None else None, stride, pad).numpy()
    if residual is not None:
        y = y + residual
    return np.maximum(y, 0.0) if relu else y


class _Node:
    """One packed convolution with its operands on the GPU; `run` returns its outputs."""

    def __init__(self, pkg, xs, o, second, residual=False, bias=True, relu=True, seed=0, k=3, pad=1, hpool=False):
        rng = np.random.default_rng(seed)
        n, c, h, w = xs
        f32 = lambda s, k=1.0: (rng.standard_normal(s) * k).astype(np.float32)
        self.pkg, self.second, self.relu, self.k, self.pad, self.hpool = pkg, second, relu, k, pad, hpool
        ys = (n, o, (h + 2 * pad - k) // 2 + 1, (w + 2 * pad - k) // 2 + 1)
        if hpool:
            ys = ys[:3] + (ys[3] // 2,)
        self.x, self.w, self.w2 = f32(xs), f32((o, c, k, k), (2 / (k * k * c)) ** 0.5), f32((o, c, 1, 1), (2 / c) ** 0.5)
        self.b, self.b2 = (f32((o,)), f32((o,))) if bias else (None, None)
        self.res = f32(ys) if residual else None
        flags = (pkg.CONV_BIAS if bias else 0) | (pkg.CONV_RESIDUAL if residual else 0) | (pkg.CONV_RELU if relu else 0) | (pkg.CONV_HPOOL if hpool else 0)
        self.desc = pkg.ConvDesc(n, c, h, w, o, k, k, 2, 2, pad, pad, 1, 1, flags)
        self.bytes = pkg.conv2d_node_filter_bytes(self.desc, second)
        z = lambda a, s: dev(a) if a is not None else torch.empty(s, device="cuda")
        self.args = [dev(self.x), dev(self.w), z(self.b, (o,)), z(self.res, ys), torch.empty(ys, device="cuda"), dev(self.w2), z(self.b2, (o,)),
                     torch.empty(ys, device="cuda")]
        A, none = pkg.Buf.arg, pkg.Buf.none()
        self.plan = pkg.Plan(8)
        self.plan.add_conv2d_packed(self.desc, A(0), A(1), A(2) if bias else none, A(3) if residual else none, A(4), A(5) if second else none,
                                    A(6) if second and bias else none, A(7) if second else none, pkg.Buf.ws(0), self.bytes or 256)
        self.plan.finalize(self.bytes or 256)

    def outputs(self, run):
        for k in (4, 7):
            self.args[k].fill_(float("nan"))
        run()
        torch.cuda.synchronize()
        return [host(self.args[4])] + ([host(self.args[7])] if self.second else [])

    def run(self, plan=None, stream=None):
        return self.outputs(lambda: (plan or self.plan).run(self.args, stream))

    def want(self):
        y = [_want(self.x, self.w, self.b, self.res, self.relu, 2, self.pad)]
        if self.hpool:
            left = np.concatenate([y[0][..., :1], y[0][..., 1:-1:2]], axis=-1)
            y = [np.maximum(np.maximum(left, y[0][..., ::2]), y[0][..., 1::2])]
        return y + ([_want(self.x, self.w2, self.b2, None, False, 2, 0)] if self.second else [])

    def check(self, got):
        # sums of k k c (c) products and a few more terms in float32, against float64
        c = self.x.shape[1]
        for y, want, terms in zip(got, self.want(), (self.k * self.k * c + 16, c + 16)):
            assert np.isfinite(y).all()
            assert np.linalg.norm(y - want) <= terms ** 0.5 * 2.0 ** -23 * np.linalg.norm(want)


@pytest.mark.parametrize("xs, o, second, residual, bias, relu", [
    ((1, 16, 13, 13), 32, True, False, True, True),         # one step of channels, one tile of 49 pixels
    ((3, 80, 13, 13), 300, True, True, True, True),         # rows of 13, images meet inside a tile, the last block 12 channels
    ((3, 80, 13, 13), 300, False, True, False, False),
    ((1, 32, 100, 90), 64, True, False, False, True),       # the widest rows; half of the workgroup's channels absent
    ((7, 32, 6, 6), 128, True, False, True, False),         # eight images in a tile
    ((2, 48, 30, 37), 160, False, False, True, True),       # 37 = 9 pieces of four columns and one more
    ((8, 64, 1, 9), 128, True, False, True, True),          # one row: the rows above and below are padding
    ((2, 512, 8, 8), 128, True, True, True, True),          # the reduction in eight parts
    ((16, 64, 56, 56), 128, True, False, True, True),       # a launch that fills the GPU, whole reductions
])
def test_conv_on_a_packed_filter(pkg, monkeypatch, xs, o, second, residual, bias, relu):
    monkeypatch.setenv("KXC_HIP_CONV_BF16X3", "1")
    node = _Node(pkg, xs, o, second, residual, bias, relu, seed=sum(xs) + o)
    assert node.bytes > 0 and "bf16x3" in node.plan.node_symbol(0)
    first = node.run()
    node.check(first)
    for a, b in zip(first, node.run()):
        assert_bit_exact(b, a, "second run")
    # without scratch the reduction stays in one piece
    monkeypatch.setenv("KXC_HIP_SCRATCH_MAX", "0")
    fresh = torch.cuda.Stream()
    node.check(node.run(stream=fresh.cuda_stream))
    node.plan.close()


@pytest.mark.parametrize("xs, o, second, k, hpool, packed", [
    ((16, 64, 56, 56), 128, True, 3, False, True), ((2, 64, 56, 56), 128, True, 3, False, False),
    ((21, 96, 26, 16), 512, False, 3, False, True), ((14, 512, 8, 38), 160, False, 3, False, False),
    ((8, 48, 74, 74), 64, False, 3, False, True), ((2, 48, 74, 74), 64, False, 3, False, False),      # fewer than 64 channels
    ((38, 64, 60, 38), 8, False, 3, False, False),                                                    # few output channels
    ((18, 3, 224, 224), 64, False, 7, False, True), ((4, 3, 224, 224), 64, False, 7, False, False),
    ((7, 3, 104, 112), 24, False, 7, True, True), ((24, 3, 30, 56), 64, False, 7, True, False),
])
def test_nodes_on_both_sides_of_the_lines(pkg, monkeypatch, xs, o, second, k, hpool, packed):
    """What a plan's stride-2 nodes launch when no switch is set."""
    for name in ("KXC_HIP_CONV_BF16X3", "KXC_HIP_WINOGRAD_BF16X3"):
        monkeypatch.delenv(name, raising=False)
    node = _Node(pkg, xs, o, second, seed=o, k=k, pad=k // 2, hpool=hpool)
    assert (node.bytes > 0) == packed == ("bf16x3" in node.plan.node_symbol(0))
    node.check(node.run())
    node.plan.close()


@pytest.mark.parametrize("xs, o, pad, residual, bias, relu, hpool", [
    ((1, 3, 224, 224), 64, 3, False, True, True, True),     # two rows of 112 columns a tile
    ((7, 3, 64, 64), 40, 3, False, True, True, True),       # seven rows of 32; the second block of channels ends after 8
    ((7, 3, 32, 56), 8, 3, False, False, True, True),       # eight rows of 28, one block of channels
    ((3, 3, 224, 224), 96, 3, False, True, True, False),
    ((2, 3, 33, 61), 20, 3, True, True, False, False),      # odd maps, channels and pixels short of a block
    ((1, 3, 7, 9), 64, 0, False, False, True, False),       # two outputs a channel
    ((5, 3, 40, 231), 33, 1, True, True, True, False),      # 114 columns: the last word of the widest rows
    ((9, 3, 16, 123), 64, 2, False, True, True, False),     # 61: the widest of the narrow rows
])
def test_first_layer_on_a_packed_filter(pkg, monkeypatch, xs, o, pad, residual, bias, relu, hpool):
    monkeypatch.setenv("KXC_HIP_CONV_BF16X3", "1")
    node = _Node(pkg, xs, o, False, residual, bias, relu, seed=sum(xs) + o, k=7, pad=pad, hpool=hpool)
    assert node.bytes > 0 and "k7x7s2_bf16x3" in node.plan.node_symbol(0)
    first = node.run()
    node.check(first)
    assert_bit_exact(node.run()[0], first[0], "second run")
    again = pkg.Plan.deserialize(node.plan.serialize(), 0)
    assert_bit_exact(node.run(again)[0], first[0], "from its text")
    again.close()
    node.plan.close()


@pytest.mark.parametrize("xs, o, pad, residual, bias, relu, packed", [
    ((6, 3, 193, 193), 64, 3, False, True, True, True),     # two rows of 97: four blocks of pixels to a wave, the last tile a row
    ((3, 3, 37, 189), 64, 3, False, False, True, True),     # two rows of 95: three blocks
    ((2, 3, 21, 150), 48, 3, True, True, True, True),       # the second block of channels ends after 16
    ((5, 3, 9, 50), 96, 0, False, True, False, True),       # narrow rows, an image a tile; the last 64 channels half empty
    ((1, 3, 46, 226), 72, 3, True, False, False, True),     # rows of 113
    ((3, 3, 7, 2), 64, 3, False, True, True, True),         # the narrowest images: one column of four pixels
    ((4, 3, 150, 150), 32, 3, False, True, True, False),
    ((9, 3, 213, 213), 32, 3, False, True, True, False), ((32, 3, 213, 213), 32, 3, False, True, True, True),
])
def test_first_layers_on_tiles_of_whole_rows(pkg, monkeypatch, xs, o, pad, residual, bias, relu, packed):
    """Selected by the rule, at the edges of their tiles, and no further from float64 than on the fp32 instructions."""
    for name in ("KXC_HIP_CONV_BF16X3", "KXC_HIP_WINOGRAD_BF16X3"):
        monkeypatch.delenv(name, raising=False)
    node = _Node(pkg, xs, o, False, residual, bias, relu, seed=sum(xs) + o, k=7, pad=pad)
    assert (node.bytes > 0) == packed == ("k7x7s2_bf16x3" in node.plan.node_symbol(0))
    first = node.run()
    node.check(first)
    assert_bit_exact(node.run()[0], first[0], "second run")
    if packed and sum(xs) < 450:
        monkeypatch.setenv("KXC_HIP_CONV_BF16X3", "0")
        plain, want = _Node(pkg, xs, o, False, residual, bias, relu, seed=sum(xs) + o, k=7, pad=pad), node.want()[0]
        assert "bf16x3" not in plain.plan.node_symbol(0)
        assert np.linalg.norm(first[0] - want) <= np.linalg.norm(plain.run()[0] - want)
        plain.plan.close()
    node.plan.close()


@pytest.mark.parametrize("xs, o, second, k, hpool", [((2, 128, 13, 18), 96, True, 3, False), ((2, 3, 45, 50), 96, False, 7, False),
                                                     ((7, 3, 64, 64), 96, False, 7, True)])
def test_conv_on_a_packed_filter_keeps_values_that_are_not_finite(pkg, monkeypatch, xs, o, second, k, hpool):
    """Infinities, NaN and operands next to the largest float reach the outputs that the operator's definition says."""
    monkeypatch.setenv("KXC_HIP_CONV_BF16X3", "1")
    node = _Node(pkg, xs, o, second, relu=hpool, seed=5, k=k, pad=k // 2, hpool=hpool)
    x, (n, c, h, w) = node.x, xs
    x[0, c // 2, 4, 5] = np.inf
    x[0, c // 3, 9, 0] = -np.inf
    x[1, c - 1, h - 1, w - 1] = np.nan
    x[1, 0, 0, 0] = 3.4e38
    node.w[40, 0, k // 2, k // 2] = 2.0 ** -20
    node.w[7, c // 2, 0, 2] = np.inf
    node.w2[8, c // 2, 0, 0] = -np.inf
    for i, a in ((0, x), (1, node.w), (5, node.w2)):
        node.args[i].copy_(torch.from_numpy(a))
    largest = float(np.finfo(np.float32).max)
    finite = lambda a: np.where(np.abs(a) > largest, np.sign(a) * np.inf, a)
    if hpool:      # relu(NaN) is 0 in the operator's definition; numpy's maximum would keep it
        y = finite(_want(node.x, node.w, node.b, None, False, 2, k // 2))
        y = np.where(y > 0, y, 0.0)
        wants = [np.maximum(np.maximum(np.concatenate([y[..., :1], y[..., 1:-1:2]], axis=-1), y[..., ::2]), y[..., 1::2])]
    else:
        wants = [finite(y) for y in node.want()]
    for got, want in zip(node.run(), wants):
        assert (np.isnan(got) == np.isnan(want)).all()
        inf = np.isinf(want)
        assert (np.isinf(got) == inf).all() and (got[inf] == want[inf]).all()
        m = np.isfinite(want)
        assert (np.abs(got[m] - want[m]) <= 1e-5 * np.maximum(np.abs(want[m]), 1.0)).all()
    node.plan.close()


@pytest.mark.parametrize("xs, o, second, k, hpool", [((2, 64, 13, 18), 96, True, 3, False), ((2, 512, 8, 8), 128, True, 3, False),
                                                     ((2, 3, 45, 50), 40, False, 7, False), ((7, 3, 64, 64), 40, False, 7, True)])
@pytest.mark.parametrize("sx, sw", [(2.0 ** -122, 1.0), (1.0, 2.0 ** -122), (2.0 ** -128, 2.0 ** 20), (2.0 ** 100, 1.0), (1.0, 2.0 ** 100)])
def test_conv_on_a_packed_filter_at_both_ends_of_the_range(pkg, monkeypatch, xs, o, second, k, hpool, sx, sw):
    """Operands that bf16 parts hold in fewer bits than float32 does unless they are scaled, and sums that then overflow: the
    error of a float32 sum, as for operands of ordinary size.  (2^-128: float32 holds a value within 2^-150.)"""
    monkeypatch.setenv("KXC_HIP_CONV_BF16X3", "1")
    node = _Node(pkg, xs, o, second, bias=False, relu=hpool, seed=9, k=k, pad=k // 2, hpool=hpool)
    for i, name, scale in ((0, "x", sx), (1, "w", sw), (5, "w2", sw)):
        a = getattr(node, name) * np.float32(scale)
        setattr(node, name, a)
        node.args[i].copy_(torch.from_numpy(a))
    node.check(node.run())
    node.plan.close()


def test_packed_filters_follow_their_weights(pkg, monkeypatch):
    """Rewritten in place they are read in the next run; frozen, only another pointer or an invalidation counts, for either
    of the two filters; the plan's text keeps the node; a graph replays it."""
    monkeypatch.setenv("KXC_HIP_CONV_BF16X3", "1")
    node = _Node(pkg, (2, 64, 14, 14), 128, True, seed=11)
    node.check(node.run())
    scale = lambda k, f: (node.args[k].mul_(f), None)[1]
    scale(1, 2.0); node.w *= 2
    scale(5, 0.5); node.w2 *= np.float32(0.5)
    node.check(node.run())
    node.plan.freeze_constants(True)
    frozen = node.run()
    node.check(frozen)
    scale(5, 4.0)
    for a, b in zip(frozen, node.run()):
        assert_bit_exact(b, a, "frozen")
    node.w2 *= 4
    node.plan.invalidate_constants()
    node.check(node.run())
    node.w2 = node.w2[::-1].copy()
    node.args[5] = dev(node.w2)
    now = node.run()
    node.check(now)
    text = node.plan.serialize()
    assert text.startswith("kxc_hip_plan 5 ")
    again = pkg.Plan.deserialize(text, 0)
    assert again.serialize() == text and "bf16x3" in again.node_symbol(0)
    for a, b in zip(now, node.run(again)):
        assert_bit_exact(b, a, "from its text")
    again.close()
    node.plan.enable_graph(True)
    stream = torch.cuda.Stream()
    for replay in range(5):
        for a, b in zip(now, node.run(stream=stream.cuda_stream)):
            assert_bit_exact(b, a, "replay %d" % replay)
        assert torch.isfinite(pkg.conv2d(node.args[0], node.args[1], None, None, 2, 1)).all()
    node.plan.close()
    # switched off when the plan is finalized: the node reads its weights as they are
    monkeypatch.setenv("KXC_HIP_CONV_BF16X3", "0")
    again = pkg.Plan.deserialize(text, 0)
    assert "bf16x3" not in again.node_symbol(0)
    node.check(node.run(again))
    again.close()
    assert pkg.conv2d_node_filter_bytes(node.desc, True) == 0


@pytest.mark.parametrize("xs, o, k, stride, pad, residual, bias, relu", [
    ((1, 16, 5, 6), 32, 5, 1, 2, False, True, True),        # one step
    ((2, 50, 27, 27), 96, 5, 1, 2, True, True, True),       # channels short of a step, images meet inside a tile
    ((3, 33, 20, 31), 64, 5, 2, 2, True, False, False),     # stride 2, an odd number of rows per phase
    ((1, 20, 23, 21), 40, 7, 1, 3, False, True, True),
    ((2, 10, 30, 30), 20, 7, 2, 0, True, True, True),       # no padding
    ((2, 48, 15, 40), 130, 3, 1, 1, True, True, True),      # the second block of channels holds two
    ((1, 35, 9, 14), 24, 3, 2, 2, False, True, False),
    ((3, 96, 4, 5), 200, 1, 1, 0, True, True, True),        # images of 20 pixels: tiles across four of them, whole quads
    ((2, 70, 5, 5), 33, 1, 1, 0, False, True, True),        # 25: pixel by pixel; six channels of a step of 64
    ((4, 64, 13, 18), 64, 1, 2, 0, True, True, True),
    ((1, 130, 8, 8), 32, 1, 1, 1, False, False, False),     # a padded 1x1 filter
    ((2, 512, 6, 6), 256, 3, 1, 1, True, True, True),       # a reduction in parts
    ((16, 64, 33, 36), 256, 1, 1, 0, True, True, True),     # a launch that fills the GPU
])
def test_single_convolution_on_a_packed_filter(pkg, monkeypatch, xs, o, k, stride, pad, residual, bias, relu):
    rng = np.random.default_rng(sum(xs) + o + k)
    n, c, h, w = xs
    f32 = lambda s, scale=1.0: (rng.standard_normal(s) * scale).astype(np.float32)
    oh, ow = (h + 2 * pad - k) // stride + 1, (w + 2 * pad - k) // stride + 1
    x, wt, b = f32(xs), f32((o, c, k, k), (2 / (k * k * c)) ** 0.5), f32((o,)) if bias else None
    res = f32((n, o, oh, ow)) if residual else None
    gpu = lambda a: dev(a) if a is not None else None
    run = lambda: host(pkg.conv2d(gpu(x), gpu(wt), gpu(b), gpu(res), stride, pad, 1, relu))
    monkeypatch.setenv("KXC_HIP_CONV_BF16X3", "0")
    assert "bf16x3" not in pkg.conv2d_variant(x.shape, wt.shape, stride, pad)
    monkeypatch.setenv("KXC_HIP_CONV_WINOGRAD", "0")
    monkeypatch.setenv("KXC_HIP_CONV_BF16X3", "1")
    assert pkg.conv2d_variant(x.shape, wt.shape, stride, pad) == "mfma_k%dx%ds%d_bf16x3" % (k, k, stride)
    first = run()
    want = _want(x, wt, b, res, relu, stride, pad)
    assert np.linalg.norm(first - want) <= (k * k * c + 16) ** 0.5 * 2.0 ** -23 * np.linalg.norm(want)
    assert_bit_exact(run(), first, "second run")
    wt *= 2                                                 # the filter is read by every call
    want = _want(x, wt, b, res, relu, stride, pad)
    assert np.linalg.norm(run() - want) <= (k * k * c + 16) ** 0.5 * 2.0 ** -23 * np.linalg.norm(want)
    # values that are not finite
    x[0, c - 1, h // 2, w // 2], x[n - 1, 0, 0, 0], wt[o - 1, c // 2, 0, 0] = np.inf, np.nan, -np.inf
    want, got = _want(x, wt, b, res, False, stride, pad), run()
    want = np.where(want > 0, want, 0.0) if relu else want
    assert (np.isnan(got) == np.isnan(want)).all() and (got[np.isinf(want)] == want[np.isinf(want)]).all()
    m = np.isfinite(want)
    assert (np.abs(got[m] - want[m]) <= 1e-5 * np.maximum(np.abs(want[m]), 1.0)).all()


@pytest.mark.parametrize("xs, o, k", [((2, 50, 27, 27), 96, 5), ((2, 512, 6, 6), 256, 3), ((3, 96, 4, 5), 200, 1)])
@pytest.mark.parametrize("sx, sw", [(2.0 ** -122, 1.0), (1.0, 2.0 ** -122), (2.0 ** 100, 1.0)])
def test_single_convolution_on_a_packed_filter_at_both_ends_of_the_range(pkg, monkeypatch, xs, o, k, sx, sw):
    monkeypatch.setenv("KXC_HIP_CONV_WINOGRAD", "0")
    monkeypatch.setenv("KXC_HIP_CONV_BF16X3", "1")
    rng = np.random.default_rng(k)
    x = rng.standard_normal(xs).astype(np.float32) * np.float32(sx)
    w = (rng.standard_normal((o, xs[1], k, k)) * (2 / (k * k * xs[1])) ** 0.5).astype(np.float32) * np.float32(sw)
    assert "bf16x3" in pkg.conv2d_variant(x.shape, w.shape, 1, k // 2)
    want = _want(x, w, None, None, False, 1, k // 2)
    got = host(pkg.conv2d(dev(x), dev(w), None, None, 1, k // 2))
    assert np.isfinite(got).all()
    assert np.linalg.norm(got - want) <= (k * k * xs[1] + 16) ** 0.5 * 2.0 ** -23 * np.linalg.norm(want)


def _filters(pkg, xs, o, k, count, seed):
    """Input, `count` filters of one shape and what a stride-1 call gives for each in float64; the tolerance of a float32 sum."""
    rng = np.random.default_rng(seed)
    n, c, h, w = xs
    x = rng.standard_normal(xs).astype(np.float32)
    wt = [(rng.standard_normal((o, c, k, k)) * (2 / (k * k * c)) ** 0.5).astype(np.float32) for _ in range(count)]
    want = [_want(x, v, None, None, False, 1, k // 2) for v in wt]
    close = lambda got, i: np.linalg.norm(host(got) - want[i]) <= (k * k * c + 16) ** 0.5 * 2.0 ** -23 * np.linalg.norm(want[i])
    return dev(x), [dev(v) for v in wt], want[0].shape, close


@pytest.mark.parametrize("xs, o, k, variant", [
    ((1, 226, 26, 33), 161, 7, "mfma_k7x7s1_bf16x3"),       # 113 chunks of the reduction on four wave groups
    ((19, 232, 8, 14), 343, 7, "mfma_k7x7s1_bf16x3"), ((17, 370, 9, 8), 363, 3, "mfma_k3x3s1_bf16x3"), ((18, 124, 53, 7), 100, 5, "mfma_k5x5s1_bf16x3"),
    ((11, 26, 27, 44), 78, 1, "mfma_k1x1s1_bf16x3"),        # too few channels for the kernel that splits over wave groups
    ((13, 731, 37, 22), 94, 3, "winograd_f2k3_bf16x3")])
def test_calls_with_a_filter_in_the_scratch_keep_it_out_of_graphs(pkg, monkeypatch, xs, o, k, variant):
    """The kernels that take these shapes' place under capture and on hipStreamPerThread would split their reductions into the very
    buffer that the eager calls keep their filters in: a graph, captured before any call, replays on another stream beside eager
    calls with another filter on the capture stream; captured again after those, and on hipStreamPerThread, the bits are the same."""
    x, w, shape, close = _filters(pkg, xs, o, k, 2, sum(xs) + o)
    assert pkg.conv2d_variant(xs, tuple(w[0].shape), 1, k // 2) == variant
    need = ctypes.c_size_t(0)
    assert pkg.lib().kxc_hip_conv2d_scratch_needed(ctypes.byref(pkg.conv_desc(xs, tuple(w[0].shape), 1, k // 2)), ctypes.byref(need)) == 0
    assert need.value > 0
    y = [torch.empty(shape, device="cuda") for _ in range(3)]
    call = lambda i, out: pkg.conv2d(x, w[i], None, None, 1, k // 2, out=out)
    capture, other = torch.cuda.Stream(), torch.cuda.Stream()
    graphs = [torch.cuda.CUDAGraph() for _ in range(2)]
    torch.cuda.synchronize()
    with torch.cuda.graph(graphs[0], stream=capture):
        call(0, y[0])
    for replay in range(5):
        y[0].zero_(); y[1].zero_()
        torch.cuda.synchronize()
        with torch.cuda.stream(other):
            graphs[0].replay()
        with torch.cuda.stream(capture):
            call(1, y[1])
        torch.cuda.synchronize()
        if replay == 0:
            first, eager = y[0].clone(), y[1].clone()
            assert close(first, 0) and close(eager, 1)
        assert torch.equal(y[0], first) and torch.equal(y[1], eager), "replay %d" % replay
    with torch.cuda.graph(graphs[1], stream=capture):
        call(0, y[2])
    graphs[1].replay()
    torch.cuda.synchronize()
    assert torch.equal(y[2], first)
    monkeypatch.setattr(pkg.hipabi, "_stream", lambda: ctypes.c_void_p(2))        # hipStreamPerThread
    outs = [[torch.zeros(shape, device="cuda") for _ in range(3)] for _ in range(2)]
    torch.cuda.synchronize()
    # (a thread waits for its stream itself: nothing does once it has ended)
    _in_threads(2, lambda i: ([call(0, out) for out in outs[i]], torch.cuda.synchronize()))
    assert all(torch.equal(out, first) for per_thread in outs for out in per_thread)


def _in_threads(count, f):
    errors = []

    def body(i):
        try:
            f(i)
        except Exception as e:      # (an exception of a thread would pass unseen)
            errors.append(e)
    threads = [threading.Thread(target=body, args=(i,)) for i in range(count)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors


@pytest.mark.parametrize("xs, o, k", [((8, 64, 27, 27), 96, 5), ((32, 128, 28, 28), 512, 1)])
def test_packed_calls_from_threads_and_streams(pkg, xs, o, k):
    """Eager calls with filters of their own, four threads on two streams at once: the buffer for a call's packed filter (and, at
    5x5 here, its partial sums) is kept per stream, whose order keeps the calls of its two threads apart."""
    x, w, shape, close = _filters(pkg, xs, o, k, 4, 78)
    assert pkg.conv2d_variant(xs, tuple(w[0].shape), 1, k // 2) == "mfma_k%dx%ds1_bf16x3" % (k, k)
    want = [pkg.conv2d(x, v, None, None, 1, k // 2) for v in w]
    assert all(close(y, i) for i, y in enumerate(want))
    out = [[torch.empty(shape, device="cuda") for _ in range(6)] for _ in w]
    streams = [torch.cuda.Stream() for _ in range(2)]
    torch.cuda.synchronize()

    def calls(i):
        with torch.cuda.stream(streams[i % 2]):
            for y in out[i]:
                pkg.conv2d(x, w[i], None, None, 1, k // 2, out=y)
    _in_threads(4, calls)
    torch.cuda.synchronize()
    assert all(torch.equal(y, want[i]) for i in range(4) for y in out[i])


@pytest.mark.parametrize("xs, o, residual, bias, relu", [
    ((1, 1, 2, 2), 1, True, True, True),                    # one channel, four pixels of a tile of 64
    ((3, 17, 4, 5), 33, True, True, False),                 # images meet inside a tile; one channel in the second step and the second block
    ((2, 64, 10, 18), 96, False, False, True),              # the last channels of the kernel of four steps; three blocks, a wave without one
    ((2, 65, 6, 14), 130, True, False, True),               # ... the first of the kernel of eight; waves with two blocks and one
    ((5, 128, 7, 12), 1000, True, True, True),              # workgroups that share their pixels, the last with fewer blocks
    ((1, 20, 8, 8), 2100, False, True, False),
    ((400, 33, 8, 8), 160, True, True, True),               # more tiles than workgroups that share them: one to a tile
])
def test_pointwise_convolution_of_few_channels(pkg, monkeypatch, xs, o, residual, bias, relu):
    """conv_point.h at the edges of its tiles, on operands that are aligned and that are not, with the residual in the output's place, and
    no further from float64 than the fp32 instructions beyond what the last roundings differ by."""
    rng = np.random.default_rng(sum(xs) + o)
    n, c, h, w = xs
    f32 = lambda s, scale=1.0: (rng.standard_normal(s) * scale).astype(np.float32)
    x, wt, b, ys = f32(xs), f32((o, c, 1, 1), (2 / c) ** 0.5), f32((o,)) if bias else None, (n, o, h, w)
    res = f32(ys) if residual else None

    def gpu(a, shift):
        if a is None:
            return None
        t = torch.empty(a.size + 4, device="cuda")[shift:shift + a.size].view(a.shape)
        return t.copy_(dev(a))

    want = _want(x, wt, b, res, relu, 1, 0)
    error = lambda y: np.linalg.norm(y - want) / np.linalg.norm(want)
    monkeypatch.setenv("KXC_HIP_CONV_BF16X3", "0")
    plain = error(host(pkg.conv2d(gpu(x, 0), gpu(wt, 0), gpu(b, 0), gpu(res, 0), 1, 0, 1, relu)))
    monkeypatch.setenv("KXC_HIP_CONV_BF16X3", "1")
    assert pkg.conv2d_variant(x.shape, wt.shape, 1, 0) == "mfma_k1x1s1_bf16x3"
    first = None
    for shift in (0, 1):
        r, out = gpu(res, shift), gpu(np.zeros(ys, np.float32), shift)
        for y in (out, r) if residual else (out,):
            y = pkg.conv2d(gpu(x, shift), gpu(wt, shift), gpu(b, shift), r, 1, 0, 1, relu, out=y)
            first = host(y) if first is None else first
            assert_bit_exact(host(y), first, "shift %d" % shift)
    assert error(first) <= (c + 16) ** 0.5 * 2.0 ** -23
    assert error(first) <= max(1.05 * plain, 2.0 ** -24)     # (of few terms both are the last rounding's)
    x[n - 1, c - 1, h - 1, w - 1], x[0, 0, 0, 1], wt[o - 1, c // 2, 0, 0] = np.inf, np.nan, -np.inf
    want = _want(x, wt, b, res, False, 1, 0)
    got, want = host(pkg.conv2d(dev(x), dev(wt), gpu(b, 0), gpu(res, 0), 1, 0, 1, relu)), np.where(want > 0, want, 0.0) if relu else want
    assert (np.isnan(got) == np.isnan(want)).all() and (got[np.isinf(want)] == want[np.isinf(want)]).all()
    m = np.isfinite(want)
    assert (np.abs(got[m] - want[m]) <= 1e-5 * np.maximum(np.abs(want[m]), 1.0)).all()


@pytest.mark.parametrize("xs, o", [
    ((16, 250, 14, 14), 500),       # 256 tiles of the filter, the last: four workgroups to a tile; channels short of a tile on both sides
    ((12, 257, 14, 14), 512),       # 272: one; one channel in the last tile
])
def test_single_winograd_convolution_transforms_its_filter(pkg, monkeypatch, xs, o):
    for name in ("KXC_HIP_CONV_BF16X3", "KXC_HIP_WINOGRAD_BF16X3"):
        monkeypatch.delenv(name, raising=False)
    x, wt, _, close = _filters(pkg, xs, o, 3, 2, o)
    assert pkg.conv2d_variant(xs, tuple(wt[0].shape), 1, 1) == "winograd_f2k3_bf16x3"
    for i in (0, 1, 0):             # the filter is read by every call
        assert close(pkg.conv2d(x, wt[i], None, None, 1, 1), i)
