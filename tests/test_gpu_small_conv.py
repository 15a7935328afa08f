"""Small convolutions that load the three values of a filter row at once, with four and with eight waves: at the ends of rows,
where the load moves, against float64 bit for bit on small integers, whose sums are exact in any order."""
import numpy as np
import pytest
import torch

from gpu_util import assert_bit_exact, dev, host

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("variant", ["mfma_k3x3_small_o1", "mfma_k3x3_small_o2"])
@pytest.mark.parametrize("xs, o, stride, pad", [
    ((1, 64, 5, 3), 20, 1, (1, 1)),         # rows of three values: every load is the whole row
    ((2, 64, 4, 4), 33, 1, (1, 1)),
    ((3, 64, 3, 5), 16, 2, (1, 1)),
    ((1, 64, 9, 37), 48, 1, (0, 0)),        # no padding
    ((1, 64, 9, 38), 48, 3, (2, 1)),        # rows above and below, windows that skip columns
    ((1, 128, 9, 33), 40, 1, (1, 1)),       # a chunk for each of eight waves
    ((2, 144, 13, 18), 32, 2, (1, 1)),      # one wave has two
    ((1, 240, 7, 20), 70, 1, (1, 0)),
    ((40, 128, 15, 16), 32, 1, (1, 1)),     # more workgroups than compute units: four waves with two chunks
    ((1, 64, 9, 30), 24, 1, (1, 2)),        # two columns of padding and
    ((1, 64, 9, 2), 24, 1, (1, 1)),         # rows of two values: one load per value
])
def test_conv_loads_filter_rows(pkg, monkeypatch, variant, xs, o, stride, pad):
    monkeypatch.setenv("KXC_HIP_CONV_VARIANT", variant)
    rng = np.random.default_rng(sum(xs) + o)
    n, c, h, w = xs
    ints = lambda *s: rng.integers(-3, 4, s).astype(np.float32)
    oh, ow = (h + 2 * pad[0] - 3) // stride + 1, (w + 2 * pad[1] - 3) // stride + 1
    x, wt, b, w2, r = ints(*xs), ints(o, c, 3, 3), ints(o), ints(o, c, 1, 1), ints(n, o, oh, ow)
    t = lambda a: torch.from_numpy(a).double()
    conv = lambda k, p: torch.nn.functional.conv2d(t(x), t(k), None, stride, p).numpy()
    want = np.maximum(conv(wt, pad) + b[:, None, None] + r, 0).astype(np.float32)
    d = pkg.ConvDesc(n, c, h, w, o, 3, 3, stride, stride, pad[0], pad[1], 1, 1, pkg.CONV_BIAS | pkg.CONV_RESIDUAL | pkg.CONV_RELU)
    arg = pkg.Buf.arg
    y, y2 = (torch.full((n, o, oh, ow), float("nan"), device="cuda") for _ in range(2))
    plan = pkg.Plan(5)
    plan.add_conv2d(d, *[arg(i) for i in range(5)])
    plan.finalize(0)
    assert variant in plan.node_symbol(0)
    plan.run([dev(x), dev(wt), dev(b), dev(r), y]); torch.cuda.synchronize()
    assert_bit_exact(host(y), want, "%s %s" % (variant, xs))
    plan.close()
    if pad != (1, 1) or o < 32 or n * oh * ow < 32:
        return
    plan = pkg.Plan(8)
    monkeypatch.delenv("KXC_HIP_CONV_VARIANT")          # (the name is one of the launches with one output)
    plan.add_conv2d_pair(d, *[arg(i) for i in range(8)])
    monkeypatch.setenv("KXC_HIP_CONV_VARIANT", variant)
    plan.finalize(256)
    assert variant in plan.node_symbol(0)
    y.fill_(float("nan"))
    plan.run([dev(x), dev(wt), dev(b), dev(r), y, dev(w2), dev(b), y2]); torch.cuda.synchronize()
    assert_bit_exact(host(y), want, "%s %s, first output" % (variant, xs))
    assert_bit_exact(host(y2), (conv(w2, 0) + b[:, None, None]).astype(np.float32), "%s %s, second output" % (variant, xs))
    plan.close()


@pytest.mark.parametrize("xs, o, stride, second, small", [
    ((2, 64, 56, 56), 64, 1, False, True),          # 1568 tiles
    ((5, 64, 56, 56), 64, 1, False, True),          # 3920: 2.26 million tiles * k, the last batch below the line
    ((6, 64, 56, 56), 64, 1, False, False),
    ((2, 64, 56, 56), 72, 1, False, True),          # a last block of 8 channels, more than 800 tiles
    ((10, 64, 56, 56), 128, 2, True, True),         # with the second output
    ((11, 64, 56, 56), 128, 2, True, False),
    ((6, 256, 14, 14), 512, 2, True, True),
    ((2, 256, 14, 14), 512, 2, False, True),        # as few tiles as staged rows take with stride 1
])
def test_where_filter_rows_in_one_load_reach(pkg, xs, o, stride, second, small):
    """The rule's line and both sides of it against float64: 9 c + 16 roundings of at most 2^-23, of independent signs."""
    rng = np.random.default_rng(sum(xs) + o)
    n, c, h, w = xs
    oh, ow = (h - 1) // stride + 1, (w - 1) // stride + 1
    f32 = lambda *s: rng.standard_normal(s).astype(np.float32)
    x, wt, b, w2 = f32(*xs), f32(o, c, 3, 3) / np.float32(3 * c ** 0.5), f32(o), f32(o, c, 1, 1) / np.float32(c ** 0.5)
    d = pkg.ConvDesc(n, c, h, w, o, 3, 3, stride, stride, 1, 1, 1, 1, pkg.CONV_BIAS)
    arg, none = pkg.Buf.arg, pkg.Buf.none()
    plan = pkg.Plan(6)
    if second:
        plan.add_conv2d_pair(d, arg(0), arg(1), arg(2), none, arg(3), arg(4), none, arg(5))
    else:
        plan.add_conv2d(d, arg(0), arg(1), arg(2), none, arg(3))
    plan.finalize(0)
    assert ("_small_o1" in plan.node_symbol(0)) == small, plan.node_symbol(0)
    y, y2 = (torch.full((n, o, oh, ow), float("nan"), device="cuda") for _ in range(2))
    plan.run([dev(x), dev(wt), dev(b), y, dev(w2), y2]); torch.cuda.synchronize()
    t = lambda a: torch.from_numpy(a).double()
    conv = lambda k, bias, p: torch.nn.functional.conv2d(t(x), t(k), bias, stride, p).numpy()
    pairs = [(y, conv(wt, t(b), 1), 9 * c + 16)] + ([(y2, conv(w2, None, 0), c + 16)] if second else [])
    for got, want, terms in pairs:
        assert np.linalg.norm(host(got) - want) <= terms ** 0.5 * 2.0 ** -23 * np.linalg.norm(want)
    plan.close()
    # the operator by itself takes the same side of the line
    if not second and stride == 1:
        assert ("_small_o1" in pkg.conv2d_variant(xs, wt.shape, 1, 1)) == small
        got = host(pkg.conv2d(dev(x), dev(wt), dev(b), None, 1, 1))
        assert np.linalg.norm(got - pairs[0][1]) <= pairs[0][2] ** 0.5 * 2.0 ** -23 * np.linalg.norm(pairs[0][1])
