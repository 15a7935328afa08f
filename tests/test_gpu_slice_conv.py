"""Plan nodes of small 3x3 convolutions on the kernel whose waves split the input channels (conv_slice.h), at the edges of its
tiles and patches, against float64; sums that are not finite; nodes that share a filter buffer; which nodes take it."""
import numpy as np
import pytest
import torch

from gpu_util import assert_bit_exact, dev, host

pytestmark = pytest.mark.gpu
VARIANTS = ["mfma_k3x3_slice_o%d_k%d" % v for v in ((1, 4), (1, 8), (2, 4), (2, 8))]


class _Node:
    """One Winograd node with its operands on the GPU."""

    def __init__(self, pkg, xs, o, pad=1, residual=True, bias=True, relu=True, seed=0, room=None):
        rng = np.random.default_rng(seed)
        n, c, h, w = xs
        ys = (n, o, h + 2 * pad - 2, w + 2 * pad - 2)
        f32 = lambda s, k=1.0: (rng.standard_normal(s) * k).astype(np.float32)
        self.pkg, self.pad, self.relu = pkg, pad, relu
        self.x, self.w = f32(xs), f32((o, c, 3, 3), (2 / (9 * c)) ** 0.5)
        self.b, self.res = f32((o,)) if bias else None, f32(ys) if residual else None
        flags = (pkg.CONV_BIAS if bias else 0) | (pkg.CONV_RESIDUAL if residual else 0) | (pkg.CONV_RELU if relu else 0)
        self.desc = pkg.ConvDesc(n, c, h, w, o, 3, 3, 1, 1, pad, pad, 1, 1, flags)
        y = torch.empty(ys, device="cuda")
        self.args = [dev(self.x), dev(self.w), y, dev(self.b) if bias else y, dev(self.res) if residual else y]
        self.room = pkg.conv2d_winograd_node_bytes(self.desc) if room is None else room
        A, none = pkg.Buf.arg, pkg.Buf.none()
        self.plan = pkg.Plan(5)
        self.plan.add_conv2d_winograd(self.desc, A(0), A(1), A(3) if bias else none, A(4) if residual else none, A(2), pkg.Buf.ws(0), self.room)
        self.plan.finalize(max(self.room, 256))

    def run(self, plan=None):
        self.args[2].fill_(float("nan"))
        (plan or self.plan).run(self.args)
        torch.cuda.synchronize()
        return host(self.args[2])

    def want(self):
        t = lambda a: torch.from_numpy(a).double()
        y = torch.nn.functional.conv2d(t(self.x), t(self.w), t(self.b) if self.b is not None else None, 1, self.pad).numpy()
        if self.res is not None:
            y = y + self.res
        return np.maximum(y, 0.0) if self.relu else y

    def check(self, got):
        # 9 c + 16 roundings of at most 2^-23 of a sum, of independent signs
        want = self.want()
        assert np.isfinite(got).all()
        assert np.linalg.norm(got - want) <= (9 * self.x.shape[1] + 16) ** 0.5 * 2.0 ** -23 * np.linalg.norm(want)


@pytest.mark.parametrize("variant", VARIANTS)
@pytest.mark.parametrize("xs, o, pad, residual, bias, relu", [
    ((1, 64, 1, 1), 32, 1, False, True, True),            # one pixel, all of its neighbours padding
    ((3, 128, 13, 13), 40, 1, True, True, True),          # whole rows; images meet inside a tile; a block of channels that ends after 8
    ((5, 132, 7, 7), 33, 1, True, False, False),          # a last step of four channels; one channel in the last block
    ((2, 64, 25, 25), 96, 1, False, True, True),          # columns under each output row, three rows in a tile
    ((1, 68, 9, 203), 64, 2, True, True, True),           # wide rows, two columns of padding
    ((1, 64, 3, 3), 64, 0, False, False, True),           # no padding, one output a channel
    ((2, 192, 31, 37), 70, 1, True, True, False),
    ((4, 256, 3, 2), 256, 1, False, True, True),          # five images in a tile
    ((2, 512, 7, 7), 512, 1, True, True, True),           # four steps a wave
])
def test_slice_kernel_at_its_edges(pkg, monkeypatch, variant, xs, o, pad, residual, bias, relu):
    monkeypatch.setenv("KXC_HIP_CONV_SLICE", variant)
    node = _Node(pkg, xs, o, pad, residual, bias, relu, seed=sum(xs) + o)
    assert variant in node.plan.node_symbol(0)
    first = node.run()
    node.check(first)
    assert_bit_exact(node.run(), first, "second run")
    again = pkg.Plan.deserialize(node.plan.serialize(), 0)
    assert variant in again.node_symbol(0)
    assert_bit_exact(node.run(again), first, "from its text")
    again.close()
    node.plan.close()


@pytest.mark.parametrize("variant", VARIANTS)
def test_slice_kernel_forms_sums_that_are_not_finite_again(pkg, monkeypatch, variant):
    """An infinity or NaN reaches the nine outputs whose windows hold it, as the definition's loop gives them, and a value of 2^113
    that leaves the scaled sums' range comes out as it is; the residual is the output's own buffer."""
    monkeypatch.setenv("KXC_HIP_CONV_SLICE", variant)
    node = _Node(pkg, (2, 128, 9, 11), 48, seed=5, relu=False)
    for at, v in (((0, 3, 4, 5), np.inf), ((1, 100, 0, 0), np.nan), ((1, 7, 8, 3), np.float32(2.0 ** 113))):
        node.x[at] = v
    node.args[0].copy_(torch.from_numpy(node.x))
    t = lambda a: torch.from_numpy(a).double()
    with np.errstate(all="ignore"):
        want = (torch.nn.functional.conv2d(t(node.x), t(node.w), t(node.b), 1, 1).numpy() + node.res).astype(np.float32)
    got = node.run()
    assert (np.isnan(got) == np.isnan(want)).all() and (np.isinf(got) == np.isinf(want)).all()
    ok = np.isfinite(want)
    assert (np.abs(got[ok] - want[ok]) <= (9 * 128 + 16) * 2.0 ** -24 * np.maximum(np.abs(want[ok]), 8)).all()
    plan = pkg.Plan(3)
    A, none = pkg.Buf.arg, pkg.Buf.none()
    plan.add_conv2d_winograd(pkg.ConvDesc(2, 128, 9, 11, 48, 3, 3, 1, 1, 1, 1, 1, 1, pkg.CONV_RESIDUAL), A(0), A(1), none, A(2), A(2), pkg.Buf.ws(0), node.room)
    plan.finalize(node.room)
    y = dev(node.res)
    plan.run([node.args[0], node.args[1], y]); torch.cuda.synchronize()
    node.b[:] = 0
    node.args[3].zero_()
    assert_bit_exact(host(y), node.run(), "residual in place")
    plan.close()
    node.plan.close()


def test_nodes_of_different_kernels_that_share_a_filter_fall_back_to_one_form(pkg, monkeypatch):
    for name in ("KXC_HIP_CONV_SLICE", "KXC_HIP_CONV_BF16X3", "KXC_HIP_WINOGRAD_BF16X3"):
        monkeypatch.delenv(name, raising=False)
    rng = np.random.default_rng(3)
    c, h = 64, 56
    d = lambda n: pkg.ConvDesc(n, c, h, h, c, 3, 3, 1, 1, 1, 1, 1, 1, 0)
    x, w = rng.standard_normal((16, c, h, h)).astype(np.float32), (rng.standard_normal((c, c, 3, 3)) / 24).astype(np.float32)
    both = pkg.conv2d_winograd_weight_bytes(x.shape, w.shape)
    args = [dev(x), dev(w), torch.empty(x.shape, device="cuda"), torch.empty((2, c, h, h), device="cuda")]
    A, none = pkg.Buf.arg, pkg.Buf.none()
    want = torch.nn.functional.conv2d(torch.from_numpy(x).double(), torch.from_numpy(w).double(), None, 1, 1).numpy()
    for shared, kernel in ((False, "slice"), (True, "winograd_f2k3_o")):
        plan = pkg.Plan(4)
        for n, y, u in ((16, 2, 0), (2, 3, 0 if shared else both)):
            plan.add_conv2d_winograd(d(n), A(0), A(1), none, none, A(y), pkg.Buf.ws(u), both)
        plan.finalize(2 * both)
        assert kernel in plan.node_symbol(1) and ("winograd_f2k3_o" if shared else "winograd_f2k3_bf16x3") in plan.node_symbol(0)
        plan.run(args); torch.cuda.synchronize()
        for y, ref in ((args[2], want), (args[3], want[:2])):
            assert np.linalg.norm(host(y) - ref) <= (9 * c + 16) ** 0.5 * 2.0 ** -23 * np.linalg.norm(ref)
        plan.close()


@pytest.mark.parametrize("xs, o, takes", [
    ((6, 128, 25, 25), 128, True), ((6, 512, 7, 7), 512, True), ((1, 64, 56, 56), 64, True),
    ((1, 256, 14, 14), 256, False),        # the small-launch kernel that stages whole rows
    ((64, 64, 56, 56), 64, False),         # large: Winograd on the bf16 matrix cores
    ((2, 32, 20, 20), 64, False),          # fewer steps of channels than waves
])
def test_which_nodes_take_the_slice_kernel(pkg, monkeypatch, xs, o, takes):
    for name in ("KXC_HIP_CONV_SLICE", "KXC_HIP_CONV_BF16X3", "KXC_HIP_WINOGRAD_BF16X3"):
        monkeypatch.delenv(name, raising=False)
    node = _Node(pkg, xs, o, seed=o)
    assert ("slice" in node.plan.node_symbol(0)) == takes, node.plan.node_symbol(0)
    node.check(node.run())
    node.plan.close()
    for name, value in (("KXC_HIP_CONV_SLICE", "0"), ("KXC_HIP_WINOGRAD_BF16X3", "0"), ("KXC_HIP_CONV_VARIANT", "mfma_k3x3_c4_o1x1_p4x1")):
        monkeypatch.setenv(name, value)
        node = _Node(pkg, xs, o, seed=o)
        assert "slice" not in node.plan.node_symbol(0)
        node.plan.close()
        monkeypatch.delenv(name)


def test_node_without_room_for_the_filter_runs_on_its_weights(pkg, monkeypatch):
    monkeypatch.delenv("KXC_HIP_CONV_SLICE", raising=False)
    node = _Node(pkg, (1, 64, 56, 56), 64, seed=1, room=0)
    assert "_small" in node.plan.node_symbol(0)
    node.check(node.run())
    node.plan.close()


PAIRS = ["mfma_k3x3s2_slice_o1_k%d_ds" % k for k in (4, 8)]


def _pair(pkg, xs, o, seed):
    """A two-output node (3x3 with stride 2, 1x1 with stride 2), its operands and what it should give."""
    rng = np.random.default_rng(seed)
    n, c, h, w = xs
    f32 = lambda s, k=1.0: (rng.standard_normal(s) * k).astype(np.float32)
    x, w1, w2, b1, b2 = f32(xs), f32((o, c, 3, 3), (2 / (9 * c)) ** 0.5), f32((o, c, 1, 1), (2 / c) ** 0.5), f32((o,)), f32((o,))
    t = lambda a: torch.from_numpy(a).double()
    want = [np.maximum(torch.nn.functional.conv2d(t(x), t(w1), t(b1), 2, 1).numpy(), 0), torch.nn.functional.conv2d(t(x), t(w2), t(b2), 2, 0).numpy()]
    desc = pkg.ConvDesc(n, c, h, w, o, 3, 3, 2, 2, 1, 1, 1, 1, pkg.CONV_BIAS | pkg.CONV_RELU)
    size = pkg.conv2d_node_filter_bytes(desc, True)
    args = [dev(a) for a in (x, w1, b1, w2, b2)] + [torch.empty(y.shape, device="cuda") for y in want]
    A, none = pkg.Buf.arg, pkg.Buf.none()
    plan = pkg.Plan(7)
    plan.add_conv2d_packed(desc, A(0), A(1), A(2), none, A(5), A(3), A(4), A(6), pkg.Buf.ws(0), size or 256)
    plan.finalize(size or 256)

    def run(p=plan):
        for y in args[5:]:
            y.fill_(float("nan"))
        p.run(args); torch.cuda.synchronize()
        got = [host(y) for y in args[5:]]
        for y, ref, terms in zip(got, want, (9 * c + 16, c + 16)):
            assert np.isfinite(y).all() and np.linalg.norm(y - ref) <= terms ** 0.5 * 2.0 ** -23 * np.linalg.norm(ref)
        return got
    return plan, size, run


@pytest.mark.parametrize("variant", PAIRS)
@pytest.mark.parametrize("xs, o", [
    ((1, 128, 3, 40), 32), ((3, 128, 13, 13), 40), ((5, 132, 7, 6), 33), ((2, 128, 49, 49), 64), ((1, 144, 9, 203), 64), ((4, 256, 5, 5), 96), ((2, 256, 14, 14), 512)])
def test_slice_kernel_with_a_second_output(pkg, monkeypatch, variant, xs, o):
    monkeypatch.setenv("KXC_HIP_CONV_SLICE", variant)
    plan, size, run = _pair(pkg, xs, o, sum(xs) + o)
    assert size > 0 and variant in plan.node_symbol(0)
    first = run()
    again = pkg.Plan.deserialize(plan.serialize(), 0)
    for p in (plan, again):
        for a, b in zip(run(p), first):
            assert_bit_exact(a, b, "again")
    again.close()
    plan.close()


@pytest.mark.parametrize("xs, o, takes", [((6, 128, 25, 25), 256, True), ((1, 128, 28, 28), 256, False), ((64, 64, 56, 56), 128, False)])
def test_which_two_output_nodes_take_the_slice_kernel(pkg, monkeypatch, xs, o, takes):
    for name in ("KXC_HIP_CONV_SLICE", "KXC_HIP_CONV_BF16X3", "KXC_HIP_WINOGRAD_BF16X3"):
        monkeypatch.delenv(name, raising=False)
    plan, size, run = _pair(pkg, xs, o, o)
    assert ("slice" in plan.node_symbol(0)) == takes, plan.node_symbol(0)
    run()
    plan.close()
