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
