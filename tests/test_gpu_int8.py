"""GPU parity of the int8 matrix-core path (channel-blocked c16 layout) against the CPU int8 operators.

Everything here is integer arithmetic plus one or two individually rounded fp32 operations per output,
so every comparison is bit-exact.  The reference compiler has no int8 operator: the CPU side is this
build's own definition ("parity unpinned" against the reference), pinned by closed forms in
test_oracle_golden.py.
"""
import importlib

import numpy as np
import pytest
import torch

from gpu_util import assert_bit_exact, dev, host
from oracle_lib import Oracle

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def orc():
    return Oracle(fast=True)


def to_c16(pkg, a):
    return pkg.i8_nchw_to_c16(dev(a))


def from_c16(pkg, t, c):
    return host(pkg.i8_c16_to_nchw(t, c))


def np_c16(a):
    """numpy statement of the layout: [N,C,H,W] -> [N,CB,H,W,16], zero padded channels."""
    n, c, h, w = a.shape
    cb = (c + 15) // 16
    p = np.zeros((n, cb * 16, h, w), a.dtype)
    p[:, :c] = a
    return np.ascontiguousarray(p.reshape(n, cb, 16, h, w).transpose(0, 1, 3, 4, 2))


def test_c16_layout_roundtrip(pkg):
    rng = np.random.default_rng(1)
    for shape in [(2, 3, 5, 7), (1, 16, 4, 4), (3, 40, 9, 3), (2, 64, 8, 8)]:
        a = rng.integers(-128, 128, shape, dtype=np.int8)
        t = to_c16(pkg, a)
        assert_bit_exact(host(t), np_c16(a), "nchw->c16 %s" % (shape,))
        assert_bit_exact(from_c16(pkg, t, shape[1]), a, "c16->nchw %s" % (shape,))


def test_quantize_to_c16(pkg, orc, synth):
    x = synth.normal((2, 3, 17, 13), 901, 1.0)
    q = pkg.quantize_to_c16(dev(x), 0.0213)
    assert_bit_exact(host(q), np_c16(orc.quantize(x, 0.0213)), "quantize to c16")
    assert abs(pkg.absmax(dev(x)) - float(np.abs(x).max())) == 0.0


QCONV_SHAPES = [
    # n, c, h, w, o, k, stride, pad
    (2, 64, 56, 56, 64, 3, 1, 1),      # layer1
    (2, 64, 56, 56, 128, 3, 2, 1),     # stride-2 3x3
    (3, 128, 28, 28, 128, 3, 1, 1),
    (5, 256, 14, 14, 256, 3, 1, 1),
    (7, 512, 7, 7, 512, 3, 1, 1),      # tiles cross image boundaries
    (2, 64, 56, 56, 128, 1, 2, 0),     # downsample
    (3, 256, 14, 14, 512, 1, 2, 0),
    (2, 3, 224, 224, 64, 7, 2, 3),     # conv1: one partial channel block, tap pairs
    (1, 3, 64, 64, 64, 7, 2, 3),
    (1, 20, 17, 19, 32, 3, 1, 1),      # channels not a multiple of 16, ragged pixel count
    (2, 48, 9, 33, 96, 3, 2, 1),       # odd number of channel blocks
    (1, 72, 12, 12, 64, 1, 1, 0),      # 5 channel blocks through 4-block chunks
    (2, 10, 11, 13, 32, 3, 1, 1),      # a single partial channel block, 3x3
    (2, 16, 11, 13, 64, 1, 1, 0),      # a single channel block, 1x1
]


@pytest.mark.parametrize("shape", QCONV_SHAPES, ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("residual", [False, True])
def test_qconv_c16_against_cpu(pkg, orc, shape, residual):
    n, c, h, w, o, k, s, p = shape
    rng = np.random.default_rng(hash(shape) % (2 ** 31))
    x = rng.integers(-128, 128, (n, c, h, w), dtype=np.int8)
    wq = rng.integers(-127, 128, (o, c, k, k), dtype=np.int8)
    bias = rng.integers(-20000, 20000, (o,), dtype=np.int32)
    mult = rng.uniform(0.5, 2.0, (o,)).astype(np.float32) * np.float32(1.0 / (8.0 * np.sqrt(c * k * k) * 64))
    oh = (h + 2 * p - k) // s + 1
    ow = (w + 2 * p - k) // s + 1
    res = rng.integers(-128, 128, (n, o, oh, ow), dtype=np.int8) if residual else None
    relu = not residual or (shape[0] % 2 == 0)
    want = orc.qconv(x, wq, bias, mult, s, p, res, 0.37 if residual else 0.0, relu)
    packed = pkg.qconv2d_c16_pack_weights(dev(wq))
    got = pkg.qconv2d_c16(to_c16(pkg, x), c, packed, wq.shape, dev(bias), dev(mult),
                          to_c16(pkg, res) if residual else None, 0.37 if residual else 0.0, s, p, relu)
    assert got.shape == (n, o // 16, oh, ow, 16)
    assert_bit_exact(from_c16(pkg, got, o), want, "qconv c16 %s" % (shape,))
    # the output range must be exercised, not saturated everywhere
    assert len(np.unique(want)) > 20


def test_qconv_c16_row_pitch_kernels_equal_the_general_kernel(pkg, orc, monkeypatch):
    """Stride-1 3x3 layers whose padded rows take 33 to 64 positions run on a compile-time row pitch (kernel names
    qrows_*); with KXC_HIP_QCONV_ROWS=0 the same shapes take the general kernel.  Same bytes either way, and both
    against the CPU: full and ragged tiles, partial channel blocks, tiles that cross image boundaries."""
    rng = np.random.default_rng(31)
    for (n, c, h, w, o, k, s, p, rows_expected) in [(2, 64, 56, 56, 64, 3, 1, 1, True), (3, 40, 5, 62, 32, 3, 1, 1, True),
                                                    (2, 32, 6, 61, 64, 3, 1, 1, True), (5, 64, 9, 33, 96, 3, 1, 1, True),
                                                    (64, 64, 56, 56, 64, 3, 1, 1, True), (2, 64, 56, 56, 128, 3, 2, 1, False),
                                                    (3, 128, 28, 28, 128, 3, 1, 1, False), (2, 32, 6, 63, 64, 3, 1, 1, False)]:
        x = rng.integers(-128, 128, (n, c, h, w), dtype=np.int8)
        wq = rng.integers(-127, 128, (o, c, k, k), dtype=np.int8)
        bias = rng.integers(-20000, 20000, (o,), dtype=np.int32)
        mult = rng.uniform(0.5, 2.0, (o,)).astype(np.float32) * np.float32(1.0 / (8.0 * np.sqrt(c * k * k) * 64))
        oh, ow = (h + 2 * p - k) // s + 1, (w + 2 * p - k) // s + 1
        res = rng.integers(-128, 128, (n, o, oh, ow), dtype=np.int8)
        packed = pkg.qconv2d_c16_pack_weights(dev(wq))
        d = pkg.qconv_desc(n, c, h, w, o, k, k, s, p)
        args = (to_c16(pkg, x), c, packed, wq.shape, dev(bias), dev(mult), to_c16(pkg, res), 0.41, s, p, True)
        monkeypatch.delenv("KXC_HIP_QCONV_ROWS", raising=False)
        name = pkg.qconv2d_c16_variant(d)
        assert name.startswith("qrows_") == rows_expected, (name, w, p)
        rows = pkg.qconv2d_c16(*args)
        monkeypatch.setenv("KXC_HIP_QCONV_ROWS", "0")
        assert pkg.qconv2d_c16_variant(d).startswith("qmfma_")
        general = pkg.qconv2d_c16(*args)
        monkeypatch.delenv("KXC_HIP_QCONV_ROWS")
        assert_bit_exact(host(rows), host(general), "row-pitch kernel against the general kernel %s" % ((n, c, h, w, o, k, s, p),))
        if n <= 5:
            want = orc.qconv(x, wq, bias, mult, s, p, res, 0.41, True)
            assert_bit_exact(from_c16(pkg, rows, o), want, "row-pitch kernel against the CPU %s" % ((n, c, h, w, o, k, s, p),))


def test_qconv_c16_largest_wave_tile_against_cpu(pkg, orc, monkeypatch):
    """The tile the largest stride-1 maps take (64 channels x 128 pixels per wave, four waves), forced by name onto shapes the CPU finishes quickly: whole and ragged tiles, a partial channel block, tiles
    that cross image boundaries, with and without residual, on the row pitch and in the general kernel."""
    rng = np.random.default_rng(77)
    monkeypatch.setenv("KXC_HIP_QCONV_VARIANT", "qmfma_k3x3_cb2_p4x4_o2_d3")
    # (the last flag: the row-pitch kernel holds the shape's patch -- 33-wide rows put 22 rows into a tile, over its 16)
    for (n, c, h, w, o, residual, relu, on_pitch) in [(2, 64, 56, 56, 64, True, True, True), (3, 40, 5, 62, 64, False, True, True),
                                                      (5, 64, 9, 33, 128, True, False, False), (7, 128, 7, 7, 64, False, False, False),
                                                      (1, 20, 17, 19, 64, True, True, False)]:
        x = rng.integers(-128, 128, (n, c, h, w), dtype=np.int8)
        wq = rng.integers(-127, 128, (o, c, 3, 3), dtype=np.int8)
        bias = rng.integers(-20000, 20000, (o,), dtype=np.int32)
        mult = rng.uniform(0.5, 2.0, (o,)).astype(np.float32) * np.float32(1.0 / (8.0 * np.sqrt(c * 9) * 64))
        res = rng.integers(-128, 128, (n, o, h, w), dtype=np.int8) if residual else None
        want = orc.qconv(x, wq, bias, mult, 1, 1, res, 0.29 if residual else 0.0, relu)
        packed = pkg.qconv2d_c16_pack_weights(dev(wq))
        d = pkg.qconv_desc(n, c, h, w, o, 3, 3, 1, 1)
        args = (to_c16(pkg, x), c, packed, wq.shape, dev(bias), dev(mult), to_c16(pkg, res) if residual else None,
                0.29 if residual else 0.0, 1, 1, relu)
        for rows in (None, "0"):
            if rows is None:
                monkeypatch.delenv("KXC_HIP_QCONV_ROWS", raising=False)
            else:
                monkeypatch.setenv("KXC_HIP_QCONV_ROWS", rows)
            name = pkg.qconv2d_c16_variant(d)
            assert "p4x4_o2" in name and name.startswith("qrows_" if rows is None and on_pitch else "qmfma_"), name
            got = pkg.qconv2d_c16(*args)
            assert_bit_exact(from_c16(pkg, got, o), want, "%s %s" % (name, (n, c, h, w, o)))
    monkeypatch.delenv("KXC_HIP_QCONV_ROWS", raising=False)
    monkeypatch.delenv("KXC_HIP_QCONV_VARIANT")
    # the shape rule: 64 -> 64 channels at 56 x 56 takes it where its tiles fill the two workgroup places per compute unit
    variant = lambda n: pkg.qconv2d_c16_variant(pkg.qconv_desc(n, 64, 56, 56, 64, 3, 3, 1, 1))
    assert "p4x4_o2" in variant(64) and "p4x4_o2" in variant(128)
    assert "p4x2_o1" in variant(32) and "p4x2_o1" in variant(96) and "p2x2_o1" in variant(31)


@pytest.mark.parametrize("shape", [
    # n, c, h, w, o, k, stride, tile: one pixel; partial channel blocks and an odd block count; tiles across images; more
    # chunks than waves and fewer; the line between one and two output-channel blocks; the last tile of one pixel
    (1, 17, 1, 1, 32, 3, 1, "o1_p1_ks2"), (3, 80, 13, 9, 96, 3, 2, "o1_p1_ks2"), (5, 512, 7, 7, 512, 3, 1, "o1_p1_ks2"),
    (1, 32, 32, 512, 32, 3, 1, "o1_p1_ks2"), (1, 48, 27, 19, 1088, 3, 1, "o2_p1_ks2"), (21, 512, 7, 7, 512, 3, 1, "o2_p2_ks4"),
    (1, 65, 1, 1, 32, 1, 1, "o1_p1_ks2"), (3, 250, 11, 13, 64, 1, 2, "o1_p1_ks2"), (2, 496, 31, 34, 256, 1, 1, "o2_p1_ks4"),
    # strides and rows whose patch no staged kernel holds
    (2, 40, 44, 143, 64, 3, 3, "o1_p1_ks2"), (1, 20, 9, 200, 32, 3, 2, "o1_p1_ks2"), (1, 33, 10, 301, 32, 1, 3, "o1_p1_ks2"),
], ids=lambda s: "x".join(map(str, s)))
def test_qconv_c16_direct_kernel(pkg, orc, monkeypatch, shape):
    """The kernel of small launches, at the edges of its tiles and of the rule that chooses its tile: the same bytes as the
    CPU operator, or where that would take long as the staged kernel."""
    n, c, h, w, o, k, s, tile = shape
    rng = np.random.default_rng(hash(shape[:-1]) % (2 ** 31))      # (numbers only: the hash of a text differs from run to run)
    x = rng.integers(-128, 128, (n, c, h, w), dtype=np.int8)
    wq = rng.integers(-127, 128, (o, c, k, k), dtype=np.int8)
    bias = rng.integers(-20000, 20000, (o,), dtype=np.int32)
    mult = rng.uniform(0.5, 2.0, (o,)).astype(np.float32) * np.float32(1.0 / (8.0 * np.sqrt(c * k * k) * 64))
    oh, ow = (h + 2 * (k // 2) - k) // s + 1, (w + 2 * (k // 2) - k) // s + 1
    res = rng.integers(-128, 128, (n, o, oh, ow), dtype=np.int8)
    d = pkg.qconv_desc(n, c, h, w, o, k, k, s, k // 2)
    assert pkg.qconv2d_c16_variant(d) == "qmfma_k%dx%d_direct_%s" % (k, k, tile)
    args = (to_c16(pkg, x), c, pkg.qconv2d_c16_pack_weights(dev(wq)), wq.shape, dev(bias), dev(mult), to_c16(pkg, res), 0.37, s, k // 2, True)
    got = pkg.qconv2d_c16(*args)
    if 2 * n * o * oh * ow * c * k * k < 10 ** 9:
        assert_bit_exact(from_c16(pkg, got, o), orc.qconv(x, wq, bias, mult, s, k // 2, res, 0.37, True), "direct %s" % (shape,))
    else:
        monkeypatch.setenv("KXC_HIP_QCONV_VARIANT", "qmfma_k%dx%d_cb%d_p4_o2" % (k, k, 2 if k == 3 else 4))
        assert "direct" not in pkg.qconv2d_c16_variant(d)
        assert torch.equal(got, pkg.qconv2d_c16(*args))


QPAIR_SHAPES = [
    # n, c, h, w, o, stride: the three ResNet-18 blocks, a ragged shape with a partial channel block and an odd block count
    (2, 64, 56, 56, 128, 2), (64, 64, 56, 56, 128, 2), (3, 128, 28, 28, 256, 2), (5, 256, 14, 14, 512, 2),
    (2, 40, 13, 17, 64, 2), (1, 10, 9, 9, 32, 2), (2, 48, 12, 10, 96, 1),
]


@pytest.mark.parametrize("shape", QPAIR_SHAPES, ids=lambda s: "x".join(map(str, s)))
def test_qconv_c16_pair_against_cpu(pkg, orc, shape):
    """A 3x3 convolution (bias, ReLU) and the 1x1 convolution with the same strides and no padding (bias, no ReLU)
    from one launch: both outputs bit-exact against the CPU int8 operators and against the two separate launches."""
    n, c, h, w, o, s = shape
    rng = np.random.default_rng(hash(shape) % (2 ** 31))
    x = rng.integers(-128, 128, (n, c, h, w), dtype=np.int8)
    wq = rng.integers(-127, 128, (o, c, 3, 3), dtype=np.int8)
    w2 = rng.integers(-127, 128, (o, c, 1, 1), dtype=np.int8)
    bias = rng.integers(-20000, 20000, (o,), dtype=np.int32)
    bias2 = rng.integers(-2000, 2000, (o,), dtype=np.int32)
    mult = rng.uniform(0.5, 2.0, (o,)).astype(np.float32) * np.float32(1.0 / (8.0 * np.sqrt(c * 9) * 64))
    mult2 = rng.uniform(0.5, 2.0, (o,)).astype(np.float32) * np.float32(1.0 / (8.0 * np.sqrt(c) * 64))
    assert pkg.qconv2d_c16_pair_supported(n, c, h, w, o, 3, s, 1)
    xc = to_c16(pkg, x)
    packed = pkg.qconv2d_c16_pack_weights(dev(wq))
    packed2 = pkg.qconv2d_c16_pair_pack_weights(dev(w2), 3)
    y, y2 = pkg.qconv2d_c16_pair(xc, c, packed, wq.shape, dev(bias), dev(mult), packed2, dev(bias2), dev(mult2), None, 0.0, s, 1, True)
    if n <= 8:
        assert_bit_exact(from_c16(pkg, y, o), orc.qconv(x, wq, bias, mult, s, 1, None, 0.0, True), "pair, main output %s" % (shape,))
        want2 = orc.qconv(x, w2, bias2, mult2, s, 0, None, 0.0, False)
        assert_bit_exact(from_c16(pkg, y2, o), want2, "pair, second output %s" % (shape,))
        assert len(np.unique(want2)) > 20
    alone = pkg.qconv2d_c16(xc, c, packed, wq.shape, dev(bias), dev(mult), None, 0.0, s, 1, True)
    alone2 = pkg.qconv2d_c16(xc, c, pkg.qconv2d_c16_pack_weights(dev(w2)), w2.shape, dev(bias2), dev(mult2), None, 0.0, s, 0, False)
    assert torch.equal(y, alone) and torch.equal(y2, alone2)
    # no bias on the second output
    _, y2n = pkg.qconv2d_c16_pair(xc, c, packed, wq.shape, dev(bias), dev(mult), packed2, None, dev(mult2), None, 0.0, s, 1, True)
    assert torch.equal(y2n, pkg.qconv2d_c16(xc, c, pkg.qconv2d_c16_pack_weights(dev(w2)), w2.shape, None, dev(mult2), None, 0.0, s, 0, False))


def test_qconv_c16_pair_random_shapes(pkg):
    """Seeded random geometries for the int8 two-output kernel (strides 1-3, padding 1 (0 and 2 are refused: the outputs' extents would differ), ragged channel and pixel
    counts, residual on the main output): both outputs equal the two separate launches byte for byte."""
    rng = np.random.default_rng(20250102)
    ran = 0
    for case in range(40):
        n = int(rng.integers(1, 5)); c = int(rng.choice([3, 10, 16, 24, 40, 64, 100, 128])); o = int(rng.choice([32, 64, 96, 128]))
        h = int(rng.integers(5, 30)); w = int(rng.integers(5, 30)); s = int(rng.integers(1, 4)); p = int(rng.choice([0, 1, 1, 1, 1, 2]))
        if p != 1:
            assert not pkg.qconv2d_c16_pair_supported(n, c, h, w, o, 3, s, p)      # the two outputs would differ in extent
        if h + 2 * p < 3 or w + 2 * p < 3 or not pkg.qconv2d_c16_pair_supported(n, c, h, w, o, 3, s, p):
            continue
        ran += 1
        x = torch.from_numpy(rng.integers(-128, 128, (n, c, h, w), dtype=np.int8)).cuda()
        wq = torch.from_numpy(rng.integers(-127, 128, (o, c, 3, 3), dtype=np.int8)).cuda()
        w2 = torch.from_numpy(rng.integers(-127, 128, (o, c, 1, 1), dtype=np.int8)).cuda()
        bias = torch.from_numpy(rng.integers(-20000, 20000, (o,), dtype=np.int32)).cuda()
        bias2 = torch.from_numpy(rng.integers(-2000, 2000, (o,), dtype=np.int32)).cuda() if case % 2 else None
        mult = torch.from_numpy((rng.uniform(0.5, 2.0, (o,)) / (8.0 * np.sqrt(c * 9) * 64)).astype(np.float32)).cuda()
        mult2 = torch.from_numpy((rng.uniform(0.5, 2.0, (o,)) / (8.0 * np.sqrt(c) * 64)).astype(np.float32)).cuda()
        oh = (h + 2 * p - 3) // s + 1; ow = (w + 2 * p - 3) // s + 1
        xc = pkg.i8_nchw_to_c16(x)
        res = pkg.i8_nchw_to_c16(torch.from_numpy(rng.integers(-128, 128, (n, o, oh, ow), dtype=np.int8)).cuda()) if case % 3 == 0 else None
        relu = case % 4 != 3
        packed = pkg.qconv2d_c16_pack_weights(wq)
        y, y2 = pkg.qconv2d_c16_pair(xc, c, packed, wq.shape, bias, mult, pkg.qconv2d_c16_pair_pack_weights(w2, 3), bias2, mult2,
                                     res, 0.37 if res is not None else 0.0, s, p, relu)
        alone = pkg.qconv2d_c16(xc, c, packed, wq.shape, bias, mult, res, 0.37 if res is not None else 0.0, s, p, relu)
        # the second output: the 1x1 convolution on the tap (p, p) of the window = on x sampled with the stride, unpadded
        xs = pkg.i8_nchw_to_c16(x[:, :, 0:(oh - 1) * s + 1:s, 0:(ow - 1) * s + 1:s].contiguous())
        alone2 = pkg.qconv2d_c16(xs, c, pkg.qconv2d_c16_pack_weights(w2), w2.shape, bias2, mult2, None, 0.0, 1, 0, False)
        assert torch.equal(y, alone), "case %d main" % case
        assert torch.equal(y2, alone2), "case %d second: n=%d c=%d h=%d w=%d o=%d s=%d p=%d" % (case, n, c, h, w, o, s, p)
    assert ran >= 20, ran


@pytest.mark.parametrize("shape", [(2, 3, 224, 224, 64), (1, 3, 64, 64, 64), (3, 4, 20, 36, 32), (2, 1, 9, 8, 96)],
                         ids=lambda s: "x".join(map(str, s)))
def test_qconv_first_layer_c4_against_cpu(pkg, orc, shape):
    """7x7 / stride 2 / padding 3 on the 4-channel input layout: same integers as the NCHW definition."""
    n, c, h, w, o = shape
    rng = np.random.default_rng(hash(shape) % (2 ** 31))
    x = rng.integers(-128, 128, (n, c, h, w), dtype=np.int8)
    wq = rng.integers(-127, 128, (o, c, 7, 7), dtype=np.int8)
    bias = rng.integers(-20000, 20000, (o,), dtype=np.int32)
    mult = rng.uniform(0.5, 2.0, (o,)).astype(np.float32) * np.float32(1.0 / (8.0 * np.sqrt(c * 49) * 64))
    want = orc.qconv(x, wq, bias, mult, 2, 3, None, 0.0, True)
    x4 = np.zeros((n, h, w, 4), np.int8)
    x4[..., :c] = x.transpose(0, 2, 3, 1)
    got = pkg.qconv2d_c4(dev(x4), c, pkg.qconv2d_c4_pack_weights(dev(wq)), wq.shape, dev(bias), dev(mult), True)
    assert_bit_exact(from_c16(pkg, got, o), want, "first layer c4 %s" % (shape,))
    assert len(np.unique(want)) > 20


@pytest.mark.parametrize("shape,relu", [((2, 3, 224, 224, 64), True), ((2, 3, 224, 224, 64), False), ((3, 3, 70, 92, 32), True),
                                        ((1, 4, 64, 64, 96), False), ((2, 3, 33, 240, 64), True), ((2, 1, 9, 8, 32), True),
                                        ((1, 2, 1, 4, 32), False)],
                         ids=lambda v: "x".join(map(str, v)) if isinstance(v, tuple) else str(v))
def test_qconv_first_layer_with_the_max_pool_in_the_kernel(pkg, orc, monkeypatch, shape, relu):
    """First layer (7x7 / 2 / 3 on the 4-channel layout) and the 3x3 / stride 2 / padding 1 max pool behind it as one
    kernel: the CPU int8 convolution followed by the CPU int8 max pool, byte for byte -- full-size maps, odd output
    widths and heights (the last window hangs over the edge), a 60-column pooled map (the widest the four waves
    cover), one-row inputs, with and without ReLU (without it negative values and the -128 pad candidate meet), and
    every number of pooled rows per workgroup."""
    n, c, h, w, o = shape
    rng = np.random.default_rng(hash(shape) % (2 ** 31))
    x = rng.integers(-128, 128, (n, c, h, w), dtype=np.int8)
    wq = rng.integers(-127, 128, (o, c, 7, 7), dtype=np.int8)
    bias = rng.integers(-20000, 20000, (o,), dtype=np.int32)
    mult = rng.uniform(0.5, 2.0, (o,)).astype(np.float32) * np.float32(1.0 / (8.0 * np.sqrt(c * 49) * 64))
    want = orc.qmaxpool(orc.qconv(x, wq, bias, mult, 2, 3, None, 0.0, relu), 3, 2, 1)
    x4 = np.zeros((n, h, w, 4), np.int8)
    x4[..., :c] = x.transpose(0, 2, 3, 1)
    xd, wp = dev(x4), pkg.qconv2d_c4_pack_weights(dev(wq))
    assert pkg.qconv2d_c4_maxpool_supported(x4.shape, o, c, relu)
    for rows in (None, "1", "2", "3", "5", "7"):
        if rows is None:
            monkeypatch.delenv("KXC_HIP_QPOOL_ROWS", raising=False)
        else:
            monkeypatch.setenv("KXC_HIP_QPOOL_ROWS", rows)
        got = pkg.qconv2d_c4_maxpool(xd, c, wp, wq.shape, dev(bias), dev(mult), relu)
        assert_bit_exact(from_c16(pkg, got, o), want, "first layer + max pool %s relu=%s rows=%s" % (shape, relu, rows))
    monkeypatch.delenv("KXC_HIP_QPOOL_ROWS", raising=False)
    # ... and the two launches it replaces
    two = pkg.maxpool2d_c16_i8(pkg.qconv2d_c4(xd, c, wp, wq.shape, dev(bias), dev(mult), relu), o, 3, 2, 1)
    assert torch.equal(got, two)
    if h > 8:
        assert len(np.unique(want)) > 20
    # a map wider than the kernel covers is refused (a 244-pixel row pools to 61 columns)
    assert not pkg.qconv2d_c4_maxpool_supported((1, 8, 244, 4), 32)


@pytest.mark.parametrize("shape", [(2, 3, 12, 16), (2, 3, 7, 9), (1, 4, 8, 8), (3, 1, 5, 4), (1, 2, 3, 3)],
                         ids=["planes-of-4", "odd-planes", "four-channels", "one-channel", "two-channels-odd"])
def test_quantize_to_c4(pkg, orc, synth, shape):
    """Plane sizes that are multiples of four take the kernel with four pixels per thread, others one pixel per
    thread: the same bytes, ties, saturation and NaN included."""
    x = synth.normal(shape, 902 + shape[1] * 10 + shape[3], 1.0)
    x.reshape(-1)[:6] = [0.5 * 0.0171, 1.5 * 0.0171, -2.5 * 0.0171, 1000.0, -1000.0, np.nan]
    q = host(pkg.quantize_to_c4(dev(x), 0.0171))
    want = orc.quantize(x, 0.0171)
    c = shape[1]
    assert_bit_exact(q[..., :c], want.transpose(0, 2, 3, 1), "quantize to c4")
    assert (q[..., c:] == 0).all()


def test_qconv_c16_closed_forms(pkg):
    # all-ones input and weights, unit multiplier: the output counts the taps inside the image times C
    c, o = 32, 32
    x = np.ones((1, c, 6, 6), np.int8)
    wq = np.ones((o, c, 3, 3), np.int8)
    mult = np.full((o,), 1.0 / c, np.float32)          # power of two: exact
    got = pkg.qconv2d_c16(to_c16(pkg, x), c, pkg.qconv2d_c16_pack_weights(dev(wq)), wq.shape, None, dev(mult),
                          None, 0.0, 1, 1, False)
    y = from_c16(pkg, got, o)
    assert y[0, 0, 0, 0] == 4 and y[0, 5, 0, 3] == 6 and y[0, 31, 2, 2] == 9
    # round half to even on exact ties and saturation
    x = np.zeros((1, 16, 1, 1), np.int8); x[0, 0] = 1
    wq = np.zeros((32, 16, 1, 1), np.int8)
    vals = [1, 3, 5, -1, -3, -5, 127, -127]            # * 0.5 -> .5 ties
    for i, v in enumerate(vals):
        wq[i, 0] = v
    mult = np.full((32,), 0.5, np.float32); mult[6] = 4.0; mult[7] = 4.0
    got = from_c16(pkg, pkg.qconv2d_c16(to_c16(pkg, x), 16, pkg.qconv2d_c16_pack_weights(dev(wq)), wq.shape, None,
                                        dev(mult), None, 0.0, 1, 0, False), 32)
    assert got[0, :8, 0, 0].tolist() == [0, 2, 2, 0, -2, -2, 127, -128]


def test_qconv_c16_rejects_unsupported(pkg):
    x = to_c16(pkg, np.zeros((1, 16, 8, 8), np.int8))
    wq = np.zeros((24, 16, 3, 3), np.int8)              # output channels not a multiple of 32
    with pytest.raises(pkg.KxcHipError):
        pkg.qconv2d_c16_pack_weights(dev(wq))
    wq = np.zeros((32, 16, 5, 5), np.int8)              # no 5x5 matrix-core variant
    packed = pkg.qconv2d_c16_pack_weights(dev(wq))
    with pytest.raises(pkg.KxcHipError):
        pkg.qconv2d_c16(x, 16, packed, wq.shape, None, dev(np.ones(32, np.float32)), None, 0.0, 1, 2, False)


def test_pools_c16(pkg, orc):
    rng = np.random.default_rng(5)
    x = rng.integers(-128, 128, (2, 40, 17, 16), dtype=np.int8)
    got = pkg.maxpool2d_c16_i8(to_c16(pkg, x), 40, 3, 2, 1)
    assert_bit_exact(from_c16(pkg, got, 40), orc.qmaxpool(x, 3, 2, 1), "maxpool c16")
    # 3x3 windows take the kernel that loads all nine taps at once (taps outside the input re-read the edge), other
    # windows the general one: strides 1-3, padding 0-2, a one-row input, extreme values at the borders
    for (shape, k, st, pad) in [((1, 16, 9, 11), 3, 1, 1), ((2, 17, 8, 8), 3, 2, 0), ((1, 32, 1, 7), 3, 2, 1), ((1, 16, 12, 5), 3, 3, 2),
                                ((2, 16, 10, 10), 2, 2, 0), ((1, 16, 7, 7), 5, 2, 2)]:
        x = rng.integers(-128, 128, shape, dtype=np.int8)
        x[:, :, 0, :] = -128; x[:, :, -1, -1] = 127
        got = pkg.maxpool2d_c16_i8(to_c16(pkg, x), shape[1], k, st, pad)
        assert_bit_exact(from_c16(pkg, got, shape[1]), orc.qmaxpool(x, k, st, pad), "maxpool c16 %s k%d s%d p%d" % (shape, k, st, pad))
    x = rng.integers(-128, 128, (3, 64, 7, 7), dtype=np.int8)
    got = host(pkg.global_avg_pool2d_c16_i8(to_c16(pkg, x), 64, 0.0173))
    assert_bit_exact(got, orc.qgap(x, 0.0173).reshape(3, 64), "gap c16")


def _quantised_model(pkg, batch, hw, config):
    qr = importlib.import_module("hdkx-aicompiler_amd.qresnet18")
    synth = pkg.synth
    consts = synth.resnet18_consts(config)
    x = synth.resnet18_input(config, batch)
    if hw != 224:
        x = np.ascontiguousarray(x[:, :, :hw, :hw])
    amax = qr.calibrate(dev(x), [dev(c) for c in consts])
    model = qr.prepare(consts, amax)
    return qr, x, model


def test_qresnet18_small_every_layer(pkg, orc):
    """Batch 2, 64x64 input: every quantised tensor of the network through the operator entry points of the C ABI
    (the compiled graph runs the same launches: test_compiled_qresnet18_small_every_layer), bit-exact."""
    qr, x, model = _quantised_model(pkg, 2, 64, 5)
    gap_mult = float(np.float32(model["scale"][model["last"]]) / (np.float32(4) * np.float32(model["gap_scale_out"])))
    want_logits, taps = orc.qresnet18(x, model, gap_mult)
    by = {L["name"]: L for L in model["layers"]}
    q = pkg.quantize_to_c16(dev(x), model["input_scale"])
    assert_bit_exact(from_c16(pkg, q, 3), taps["input"], "quantised input")

    def conv(t, c, name, res=None):
        L = by[name]
        packed = pkg.qconv2d_c16_pack_weights(dev(L["wq"]))
        y = pkg.qconv2d_c16(t, c, packed, L["wq"].shape, dev(L["bias_q"]), dev(L["mult"]), res,
                            L["res_mult"] if res is not None else 0.0, L["stride"], L["pad"], L["relu"])
        assert_bit_exact(from_c16(pkg, y, L["cout"]), taps[name], name)
        return y

    y = conv(q, 3, "conv1")
    cur = pkg.maxpool2d_c16_i8(y, 64, 3, 2, 1)
    assert_bit_exact(from_c16(pkg, cur, 64), taps["maxpool"], "maxpool")
    cin = 64
    for stage, ch in enumerate((64, 128, 256, 512)):
        for blk in range(2):
            first = blk == 0 and stage > 0
            name = "l%d.%d" % (stage + 1, blk)
            a = conv(cur, cin, name + ".conv1")
            idn = conv(cur, cin, name + ".down") if first else cur
            cur = conv(a, ch, name + ".conv2", idn)
            cin = ch
    g = pkg.global_avg_pool2d_c16_i8(cur, 512, gap_mult)
    fc = model["fc"]
    logits = pkg.qdense(g, dev(fc["wq"]), dev(fc["bias_q"]), dev(fc["mult"]))
    assert_bit_exact(host(logits), want_logits, "quantised logits (operator by operator)")
    # the quantisation must be meaningful
    assert np.isfinite(want_logits).all() and np.abs(want_logits).max() > 0


@pytest.mark.parametrize("m,n,k", [(64, 1000, 512), (70, 37, 1056), (33, 65, 32), (70, 37, 1040), (1, 5, 16), (9, 12, 24)])
def test_qdense_shapes(pkg, orc, m, n, k):
    """Matrix-core kernel (k a multiple of 32, ragged rows and columns), wave-per-column kernel (k a multiple
    of 16, more than one 1 KiB slice) and the scalar fallback (k = 24)."""
    rng = np.random.default_rng(m * 1000 + k)
    a = rng.integers(-128, 128, (m, k), dtype=np.int8)
    b = rng.integers(-127, 128, (n, k), dtype=np.int8)
    bias = rng.integers(-5000, 5000, (n,), dtype=np.int32)
    mult = rng.uniform(1e-4, 1e-3, (n,)).astype(np.float32)
    assert_bit_exact(host(pkg.qdense(dev(a), dev(b), dev(bias), dev(mult))), orc.qdense(a, b, bias, mult),
                     "qdense %dx%dx%d" % (m, n, k))


# ---------------------------------------------------------------- the same network compiled from its Relay graph
def _compiled(pkg, model, batch, hw, **kw):
    ha = importlib.import_module("hdkx-aicompiler_amd.hostapi")
    mod = ha.CompiledQResNet18(model, batch, hw, **kw)
    consts = [dev(c) for c in mod.constants(model)]
    return mod, consts


def _run_compiled(mod, x_dev, consts, out):
    mod.run_packed(mod.packed([x_dev] + consts + [out]))
    torch.cuda.synchronize()


def test_compiled_qresnet18_plan_is_the_matrix_core_plan(pkg):
    """Compiler::Compile on the quantised graph chooses the channel-blocked layout itself: 20 launches, the first
    convolution on the 4-channel input layout with the max pool in its kernel, every other one on c16, the three
    downsamples as second outputs, weights packed by the plan from the OIHW constants (20 packs, one per convolution),
    no layout converter anywhere."""
    qr, x, model = _quantised_model(pkg, 2, 64, 5)
    mod, _ = _compiled(pkg, model, 2, 64)
    sym = mod.launches()
    assert len(sym) == 20
    assert sym[0] == "qnn_quantize kxc_quantize_f32_nchw_to_c4_i8"
    assert sym[1] == "qnn_conv2d kxc_qconv2d_c4_i8:qmfma_k7x7s2_c4+relu+maxpool3x3s2"
    assert all(s.startswith("qnn_conv2d kxc_qconv2d_c16_i8:qmfma") for s in sym[2:18])
    assert sum("|qconv1x1+bias" in s for s in sym) == 3
    assert sym[18] == "qnn_global_avg_pool2d kxc_global_avg_pool2d_c16_i8" and sym[19] == "qnn_dense kxc_qdense_i8"
    assert not any("layout_convert" in s for s in sym)
    plan_text = mod.plan_json()
    assert plan_text.count("\\npack ") == 20 and "kxc_hip_plan 3" in plan_text


def test_compiled_qresnet18_small_every_layer(pkg, orc):
    """Batch 2, 64x64 input, through Compiler::Compile: the logits, and every quantised tensor of the network as the
    result of the graph cut at that layer (which also exercises the converter back to NCHW), bit-exact against the
    CPU int8 chain."""
    qr, x, model = _quantised_model(pkg, 2, 64, 5)
    mod, consts = _compiled(pkg, model, 2, 64)
    out = torch.empty((2, 1000), device="cuda")
    _run_compiled(mod, dev(x), consts, out)
    want_logits, taps = orc.qresnet18(x, model, mod.gap_mult)
    assert_bit_exact(host(out), want_logits, "compiled quantised logits")
    # a second run and a run after the weights were updated in place see the current constants
    _run_compiled(mod, dev(x), consts, out)
    assert_bit_exact(host(out), want_logits, "compiled quantised logits, second run")
    for name, want in taps.items():
        cut, cc = _compiled(pkg, model, 2, 64, result=name)
        got = torch.empty(want.shape, dtype=torch.int8, device="cuda")
        _run_compiled(cut, dev(x), cc, got)
        assert_bit_exact(host(got), want, "compiled graph cut at %s" % name)
        cut.close()
    mod.close()


def test_compiled_qresnet18_constants_are_read_on_every_run(pkg, orc):
    """The CPU backend re-reads every constant on every call; so does the compiled module unless its constants are
    frozen: an in-place update of a weight tensor shows in the next run, a frozen module keeps the packed copy until
    it is told."""
    qr, x, model = _quantised_model(pkg, 2, 64, 5)
    mod, consts = _compiled(pkg, model, 2, 64)
    out = torch.empty((2, 1000), device="cuda")
    _run_compiled(mod, dev(x), consts, out)
    before = host(out).copy()
    k = mod.constant_names.index("l3.1.conv1.w")
    saved = consts[k].clone()
    consts[k].neg_()
    changed = dict(model)
    changed["layers"] = [dict(L, wq=-L["wq"]) if L["name"] == "l3.1.conv1" else L for L in model["layers"]]
    want, _ = orc.qresnet18(x, changed, mod.gap_mult)
    _run_compiled(mod, dev(x), consts, out)
    assert_bit_exact(host(out), want, "logits after an in-place weight update")
    assert not np.array_equal(host(out), before)
    mod.freeze_constants(True)
    _run_compiled(mod, dev(x), consts, out)                   # packs what it is given now
    consts[k].copy_(saved)
    _run_compiled(mod, dev(x), consts, out)                   # frozen: still the packed copy of the negated weights
    assert_bit_exact(host(out), want, "frozen module keeps its packed weights")
    mod.invalidate_constants()
    _run_compiled(mod, dev(x), consts, out)
    assert_bit_exact(host(out), before, "after invalidate_constants the restored weights are packed again")
    mod.close()


def test_compiled_qresnet18_batch64_images(pkg, orc):
    """BASELINE configuration 5 through Compiler::Compile: images 0 and 63 of the batch against the CPU int8 chain,
    determinism, graph replay, the launch plan rebuilt from the text inside the module's execution-plan JSON, and two
    shares of the batch side by side."""
    qr, x, model = _quantised_model(pkg, 64, 224, 5)
    mod, consts = _compiled(pkg, model, 64, 224)
    assert len(mod.launches()) == 20
    xd = dev(x)
    out = torch.empty((64, 1000), device="cuda")
    _run_compiled(mod, xd, consts, out)
    first = host(out).copy()
    for n in (0, 63):
        want, _ = orc.qresnet18(x[n:n + 1], model, mod.gap_mult)
        assert_bit_exact(first[n:n + 1], want, "compiled quantised resnet18 batch 64, image %d" % n)
    import json
    again = pkg.Plan.deserialize(json.loads(mod.plan_json())["kxc_hip"]["launch_plan"], 0)
    assert again.num_weight_packs() == 20 and len(again.symbols()) == 20
    out_again = torch.zeros_like(out)
    again.run([xd] + consts + [out_again])
    torch.cuda.synchronize()
    assert_bit_exact(host(out_again), first, "launch plan rebuilt from its text (two-output nodes, weight packs)")
    again.close()
    mod.freeze_constants(True)
    mod.enable_graph_replay(True)
    stream = torch.cuda.Stream()
    args = mod.packed([xd] + consts + [out])
    with torch.cuda.stream(stream):
        for replay in range(4):
            out.zero_()
            mod.run_packed(args, stream.cuda_stream)
            stream.synchronize()
            assert_bit_exact(host(out), first, "frozen module, graph replay %d" % replay)
    two, _ = _compiled(pkg, model, 64, 224, lanes=2)
    assert len(two.launches()) == 40
    out2 = torch.zeros((64, 1000), device="cuda")
    _run_compiled(two, xd, consts, out2)
    assert_bit_exact(host(out2), first, "two shares of the batch")
    two.close()
    mod.close()


def test_plan_weight_pack_and_layout_nodes(pkg, orc):
    """C ABI: a plan that is handed OIHW weights packs them itself at the start of a run (one launch for all packs)
    and converts between NCHW and c16 with layout nodes; its text form round-trips."""
    H = pkg
    rng = np.random.default_rng(17)
    n, c, h, w, o = 2, 40, 13, 17, 64
    x = rng.integers(-128, 128, (n, c, h, w), dtype=np.int8)
    wq = rng.integers(-127, 128, (o, c, 3, 3), dtype=np.int8)
    bias = rng.integers(-20000, 20000, (o,), dtype=np.int32)
    mult = rng.uniform(0.5, 2.0, (o,)).astype(np.float32) * np.float32(1.0 / (8.0 * np.sqrt(c * 9) * 64))
    want = orc.qconv(x, wq, bias, mult, 1, 1, None, 0.0, True)
    d = H.qconv_desc(n, c, h, w, o, 3, 3, 1, 1, H.CONV_BIAS | H.CONV_RELU)
    Buf = H.Buf
    cb, ob = (c + 15) // 16, o // 16
    off_x = 0
    off_y = off_x + (n * cb * h * w * 16 + 255) // 256 * 256
    off_w = off_y + (n * ob * h * w * 16 + 255) // 256 * 256
    plan = H.Plan(5)
    plan.add_i8_layout(True, n, c, h * w, Buf.arg(0), Buf.ws(off_x))
    plan.add_qconv_weight_pack(H.QPACK_C16, d, Buf.arg(1), Buf.ws(off_w))
    plan.add_qconv2d_c16(d, Buf.ws(off_x), Buf.ws(off_w), Buf.arg(2), Buf.arg(3), Buf.none(), Buf.ws(off_y))
    plan.add_i8_layout(False, n, o, h * w, Buf.ws(off_y), Buf.arg(4))
    assert plan.num_weight_packs() == 1
    packed_bytes = int(H.qconv2d_c16_pack_weights(dev(wq)).numel())
    with pytest.raises(H.KxcHipError):
        plan.finalize(off_w + packed_bytes - 1)          # the packed weights must fit the workspace
    plan.finalize(off_w + packed_bytes)
    out = torch.zeros((n, o, h, w), dtype=torch.int8, device="cuda")
    wd = dev(wq)
    plan.run([dev(x), wd, dev(bias), dev(mult), out])
    torch.cuda.synchronize()
    assert_bit_exact(host(out), want, "plan with its own weight pack")
    again = H.Plan.deserialize(plan.serialize(), 0)
    assert again.num_weight_packs() == 1 and again.symbols() == plan.symbols()
    out.zero_()
    again.run([dev(x), wd, dev(bias), dev(mult), out])
    torch.cuda.synchronize()
    assert_bit_exact(host(out), want, "the same plan rebuilt from its text")
    # the weights must be a packed argument, the packed copy a workspace region
    bad = H.Plan(5)
    with pytest.raises(H.KxcHipError):
        bad.add_qconv_weight_pack(H.QPACK_C16, d, Buf.ws(0), Buf.ws(256))
    with pytest.raises(H.KxcHipError):
        bad.add_qconv_weight_pack(H.QPACK_C16, d, Buf.arg(1), Buf.arg(2))
    with pytest.raises(H.KxcHipError):
        bad.add_qconv_weight_pack(9, d, Buf.arg(1), Buf.ws(0))


def test_plan_packs_many_weight_tensors_in_one_launch(pkg):
    """The plan's batched pack (one launch for every weight tensor, rows staged through LDS) writes exactly the bytes
    the per-tensor pack entry points write: full and partial channel blocks, odd block counts, 1x1 / 3x3 / 7x7
    windows, a second-output tensor in its convolution's chunking, the first-layer order, and more tensors than one
    batch holds."""
    import ctypes as C
    H = pkg
    rng = np.random.default_rng(23)
    Buf = H.Buf
    # (kind, o, c, k) ; the pair packs [o, c, 1, 1] weights in the chunking of a 3x3 convolution on c channels
    cases = [(H.QPACK_C16, 64, 40, 3), (H.QPACK_C16, 32, 10, 3), (H.QPACK_C16, 64, 72, 1), (H.QPACK_C16, 64, 3, 7),
             (H.QPACK_C16_PAIR, 128, 64, 3), (H.QPACK_C16_PAIR, 64, 40, 3), (H.QPACK_C4, 64, 3, 7), (H.QPACK_C16, 96, 48, 3),
             (H.QPACK_C16, 64, 16, 1), (H.QPACK_C16, 32, 17, 5)] + [(H.QPACK_C16, 32, 16 * (i + 1), 3) for i in range(18)]
    assert len(cases) > 24
    plan = H.Plan(len(cases))
    weights, expect, offsets = [], [], []
    top = 0
    for i, (kind, o, c, k) in enumerate(cases):
        if kind == H.QPACK_C16_PAIR:
            w = rng.integers(-127, 128, (o, c, 1, 1), dtype=np.int8)
            want = H.qconv2d_c16_pair_pack_weights(dev(w), k)
            d = H.qconv_desc(1, c, 8, 8, o, k, k, 2, 1)
        elif kind == H.QPACK_C4:
            w = rng.integers(-127, 128, (o, c, 7, 7), dtype=np.int8)
            want = H.qconv2d_c4_pack_weights(dev(w))
            d = H.qconv_desc(1, c, 16, 16, o, 7, 7, 2, 3)
        else:
            w = rng.integers(-127, 128, (o, c, k, k), dtype=np.int8)
            want = H.qconv2d_c16_pack_weights(dev(w))
            d = H.qconv_desc(1, c, 8, 8, o, k, k, 1, k // 2)
        plan.add_qconv_weight_pack(kind, d, Buf.arg(i), Buf.ws(top))
        weights.append(dev(w)); expect.append(host(want)); offsets.append(top)
        top += (int(want.numel()) + 255) // 256 * 256
    plan.add_copy(16, Buf.arg(0), Buf.ws(top))          # a plan needs no node to pack, but a run must enqueue something after it
    plan.finalize(top + 256)
    plan.run(weights)
    torch.cuda.synchronize()
    base = plan.workspace_ptr()
    for i, (want, off) in enumerate(zip(expect, offsets)):
        got = np.empty(want.shape, np.int8)
        pkg.lib().kxc_hip_copy(C.c_void_p(base), C.c_size_t(off), got.ctypes.data_as(C.c_void_p), C.c_size_t(0), C.c_size_t(got.nbytes),
                               C.c_int32(1), C.c_int32(0), None)
        torch.cuda.synchronize()
        assert_bit_exact(got, want, "batched pack of tensor %d %s" % (i, cases[i][1:]))
    plan.close()


@pytest.mark.parametrize("shape", [(2, 3, 193, 193, 64), (3, 3, 70, 93, 32), (1, 4, 33, 66, 96), (2, 1, 9, 7, 32), (1, 2, 5, 5, 32), (2, 3, 40, 239, 64)],
                         ids=lambda s: "x".join(map(str, s)))
def test_qconv_first_layer_on_rows_of_any_width(pkg, orc, shape):
    """Rows that are no multiple of four pixels: the last 16-byte piece of a row ends in the next row's pixels (or behind the tensor),
    which must count as padding.  Byte for byte, with the max pool in the kernel and without."""
    n, c, h, w, o = shape
    rng = np.random.default_rng(sum(shape))
    x = rng.integers(-128, 128, (n, c, h, w), dtype=np.int8)
    wq = rng.integers(-127, 128, (o, c, 7, 7), dtype=np.int8)
    bias = rng.integers(-20000, 20000, (o,), dtype=np.int32)
    mult = rng.uniform(0.5, 2.0, (o,)).astype(np.float32) * np.float32(1.0 / (8.0 * np.sqrt(c * 49) * 64))
    want = orc.qconv(x, wq, bias, mult, 2, 3, None, 0.0, True)
    room = torch.full((n * h * w * 4 + 64,), 77, dtype=torch.int8, device="cuda")      # (what lies behind the tensor is not zero)
    x4 = room[:n * h * w * 4].view(n, h, w, 4)
    x4.zero_()
    x4[..., :c] = dev(np.ascontiguousarray(x.transpose(0, 2, 3, 1)))
    wp = pkg.qconv2d_c4_pack_weights(dev(wq))
    got = pkg.qconv2d_c4(x4, c, wp, wq.shape, dev(bias), dev(mult), True)
    assert_bit_exact(from_c16(pkg, got, o), want, "first layer")
    if pkg.qconv2d_c4_maxpool_supported(x4.shape, o, c, True):
        got = pkg.qconv2d_c4_maxpool(x4, c, wp, wq.shape, dev(bias), dev(mult), True)
        assert_bit_exact(from_c16(pkg, got, o), orc.qmaxpool(want, 3, 2, 1), "first layer + max pool")
    assert len(np.unique(want)) > 5
