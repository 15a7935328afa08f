"""Which kernel a convolution takes, asked from the library on the host: no GPU is needed."""
import ctypes
import random
import time

import pytest


def _variant(pkg, xs, o, k, stride=1, pad=None, flags=0):
    return pkg.conv2d_variant(xs, (o, xs[1], k, k), stride, k // 2 if pad is None else pad, flags=flags)


def _node(pkg, xs, o, k, second=False, hpool=False):
    n, c, h, w = xs
    flags = pkg.CONV_BIAS | pkg.CONV_RELU | (pkg.CONV_HPOOL if hpool else 0)
    return pkg.conv2d_node_filter_bytes(pkg.ConvDesc(n, c, h, w, o, k, k, 2, 2, k // 2, k // 2, 1, 1, flags), second)


CALLS = [((8, 64, 27, 27), 96, 5), ((32, 128, 28, 28), 512, 1), ((1, 226, 26, 33), 161, 7), ((17, 370, 9, 8), 363, 3)]
NODES = [((64, 64, 56, 56), 128, 3, True, False), ((64, 64, 56, 56), 128, 3, False, False), ((64, 3, 224, 224), 64, 7, False, True)]


@pytest.mark.parametrize("switches, packed", [
    ({}, True), ({"KXC_HIP_CONV_BF16X3": "0"}, False),
    # the switch that kept every convolution on the fp32 instructions before the packed kernels keeps them out as well
    ({"KXC_HIP_WINOGRAD_BF16X3": "0"}, False), ({"KXC_HIP_WINOGRAD_BF16X3": "0", "KXC_HIP_CONV_BF16X3": "1"}, True)])
def test_switches_of_the_three_part_kernels(pkg, monkeypatch, switches, packed):
    for name in ("KXC_HIP_CONV_BF16X3", "KXC_HIP_WINOGRAD_BF16X3"):
        monkeypatch.delenv(name, raising=False)
    for name, value in switches.items():
        monkeypatch.setenv(name, value)
    for xs, o, k in CALLS:
        assert _variant(pkg, xs, o, k).endswith("_bf16x3") == packed, (xs, o, k)
    for xs, o, k, second, hpool in NODES:
        assert (_node(pkg, xs, o, k, second, hpool) > 0) == packed, (xs, o, k)


def _us(f):
    best = 1e9
    for _ in range(20):
        t = time.perf_counter()
        for _ in range(50):
            f()
        best = min(best, (time.perf_counter() - t) / 50 * 1e6)
    return best


@pytest.mark.parametrize("xs, o, k", [((64, 64, 111, 111), 128, 5), ((16, 64, 87, 87), 128, 5)])
def test_maps_too_wide_for_the_packed_kernel_are_refused_at_once(pkg, monkeypatch, xs, o, k):
    """A call asks for the packed kernel first; where the rows of its map do not fit, that must cost little beside the selection of
    the kernel that takes it (which a plan's node, asked here for comparison, does without the question)."""
    monkeypatch.delenv("KXC_HIP_CONV_BF16X3", raising=False)
    d = pkg.conv_desc(xs, (o, xs[1], k, k), 1, k // 2, 1, 0)
    lib, p = pkg.lib(), ctypes.byref(d)
    assert "bf16x3" not in _variant(pkg, xs, o, k)
    assert _us(lambda: lib.kxc_hip_conv2d_variant(p)) <= 1.5 * _us(lambda: lib.kxc_hip_conv2d_node_variant(p)) + 2


@pytest.mark.parametrize("seed", range(4))
def test_packed_kernel_covers_the_maps_whose_rows_fit(pkg, monkeypatch, seed):
    """Two rows of waves and an LDS plane of 384 positions: the rows that a tile of 64 pixels touches, from a walk over every tile."""
    monkeypatch.setenv("KXC_HIP_CONV_BF16X3", "1")
    monkeypatch.setenv("KXC_HIP_CONV_WINOGRAD", "0")
    rng = random.Random(seed)
    for _ in range(150):
        k, s = rng.choice((3, 5, 7)), rng.choice((1, 2))
        n, h, w, pad = rng.randint(1, 9), rng.randint(k, 60), rng.randint(k, 90), rng.randint(0, 3)
        oh, ow = (h + 2 * pad - k) // s + 1, (w + 2 * pad - k) // s + 1
        at = lambda m: m // (oh * ow) * (oh + (k - 1) // s) + m % (oh * ow) // ow
        rows = max(at(min(m + 64, n * oh * ow) - 1) - at(m) for m in range(0, n * oh * ow, 64)) + 1 + (k - 1) // s
        pitch = 2 * max(ow + (k - 1) // 2, (w - 1 + pad) // 2 + 1) if s == 2 else max(ow + k - 1, w + pad)
        covers = rows * pitch <= 384 and 2 * rows * -(-w // 4) <= 256
        assert _variant(pkg, (n, 16, h, w), 32, k, s, pad).endswith("_bf16x3") == covers, (n, h, w, k, s, pad)


def test_small_calls_are_chosen_without_walking_their_map(pkg):
    """A call of a few microseconds: the kernel that stages whole rows asks how many a tile touches, tile by tile, and is out of the
    question from 257 tiles on.  Compared with the selection of a 1x1 filter, which walks nothing."""
    lib = pkg.lib()
    us = {}
    for k in (1, 3):
        d = pkg.conv_desc((1, 64, 56, 56), (64, 64, k, k), 1, k // 2, 1, 0)
        us[k] = _us(lambda: lib.kxc_hip_conv2d_variant(ctypes.byref(d)))
    assert us[3] <= 1.6 * us[1] + 0.1, us


@pytest.mark.parametrize("xs, o, second, packed", [
    # us, fp32 instructions and packed
    ((64, 64, 56, 56), 128, True, True),        # 97, 61
    ((64, 128, 28, 28), 256, True, True),       # 94, 54
    ((64, 256, 14, 14), 512, True, True),       # 104, 52
    ((21, 96, 26, 16), 512, False, True),       # 37, 21
    ((46, 96, 63, 16), 64, False, True),        # 27, 20: half of a workgroup's output channels
    ((38, 256, 60, 38), 8, False, False),       # 24, 99
    ((43, 384, 32, 31), 16, False, False),      # 34, 61
    ((59, 16, 46, 51), 32, True, False),        # 15, 25
    ((30, 384, 21, 45), 48, False, False),      # 42, 50
    ((18, 384, 13, 56), 64, True, False),       # 26, 34: small-launch kernel
    ((14, 512, 8, 38), 160, False, False),      # 24, 36
    ((2, 64, 56, 56), 128, True, False),        # 12, 16
])
def test_stride_2_nodes_take_the_packed_kernel_where_it_is_the_faster_one(pkg, monkeypatch, xs, o, second, packed):
    for name in ("KXC_HIP_CONV_BF16X3", "KXC_HIP_WINOGRAD_BF16X3"):
        monkeypatch.delenv(name, raising=False)
    assert (_node(pkg, xs, o, 3, second) > 0) == packed


@pytest.mark.parametrize("xs, o, k, stride, packed", [
    # us, fp32 instructions and packed
    ((8, 64, 27, 27), 96, 5, 1, True),          # 38, 25
    ((32, 128, 28, 28), 512, 1, 1, True),       # 74, 50
    ((1, 226, 26, 33), 161, 7, 1, True),        # 72, 44
    ((4, 13, 64, 12), 356, 7, 1, True),         # 32, 25
    ((27, 220, 9, 10), 260, 3, 1, True),        # 48, 35
    ((37, 32, 19, 12), 32, 5, 1, False),        # 16, 21
    ((11, 6, 60, 48), 126, 5, 1, False),        # 18, 27
    ((1, 64, 15, 16), 96, 7, 1, False),         # 18, 25
    ((11, 16, 90, 9), 144, 3, 1, False),        # 12, 17
    ((3, 32, 100, 31), 208, 3, 1, False),       # 18, 22
    ((2, 120, 14, 48), 35, 1, 1, False),        # 6, 11
    ((3, 400, 22, 78), 448, 1, 1, False),       # 27, 31
    ((7, 160, 37, 23), 400, 1, 1, False),       # 18, 30
])
def test_single_calls_take_the_packed_kernel_where_it_is_the_faster_one(pkg, monkeypatch, xs, o, k, stride, packed):
    for name in ("KXC_HIP_CONV_BF16X3", "KXC_HIP_WINOGRAD_BF16X3"):
        monkeypatch.delenv(name, raising=False)
    for flags in (5, 7):
        assert _variant(pkg, xs, o, k, stride, flags=flags).endswith("_bf16x3") == packed


@pytest.mark.parametrize("xs, o, hpool, packed", [
    # us, fp32 instructions and packed
    ((64, 3, 224, 224), 64, True, True),        # 169, 108
    ((2, 3, 224, 224), 8, True, True),          # 31, 17
    ((7, 3, 104, 112), 24, True, True),         # 18, 17: tiles of 13 rows
    ((8, 3, 56, 56), 64, True, True),           # 32, 21: 21 rows, and tiles of 448 pixels on the other side
    ((74, 3, 56, 56), 16, True, True),          # 29, 28
    ((17, 3, 304, 56), 24, True, True),         # 30, 28
    ((24, 3, 30, 56), 64, True, False),         # 19, 21
    ((2, 3, 168, 56), 256, True, False),        # 19, 21
    ((20, 3, 21, 224), 32, True, False),        # 19, 20: images meet inside a tile
    ((18, 3, 224, 224), 64, False, True),       # 58, 35
    ((24, 3, 224, 224), 48, False, True),       # 82, 53
    ((33, 3, 224, 224), 32, False, True),       # 64, 62
    ((78, 3, 224, 224), 24, False, True),       # 124, 116
    ((57, 3, 144, 112), 32, False, False),      # 37, 44
    ((42, 3, 112, 224), 24, False, False),      # 41, 43
    ((4, 3, 224, 224), 64, False, False),       # 21, 22
])
def test_first_layers_take_the_packed_kernel_where_it_is_the_faster_one(pkg, monkeypatch, xs, o, hpool, packed):
    for name in ("KXC_HIP_CONV_BF16X3", "KXC_HIP_WINOGRAD_BF16X3"):
        monkeypatch.delenv(name, raising=False)
    assert (_node(pkg, xs, o, 7, hpool=hpool) > 0) == packed


@pytest.mark.parametrize("name, value", [("KXC_HIP_CONV_VARIANT", "direct"), ("KXC_HIP_CONV_GSPLIT", "2"), ("KXC_HIP_CONV_HPOOL_VARIANT", "mfma_k7x7_t1_o1x2_p7x1")])
def test_switches_that_force_another_kernel_s_shape(pkg, monkeypatch, name, value):
    """A workgroup shape or a split that the environment names is that of the kernels on the fp32 instructions."""
    monkeypatch.delenv("KXC_HIP_CONV_BF16X3", raising=False)
    monkeypatch.setenv(name, value)
    assert not any(_variant(pkg, xs, o, k).startswith("mfma_") and _variant(pkg, xs, o, k).endswith("_bf16x3") for xs, o, k in CALLS)
    assert not any(_node(pkg, *n) for n in NODES)


@pytest.mark.parametrize("xs, o, three_part", [
    # us, fp32 instructions and bf16 matrix cores
    ((6, 128, 28, 28), 128, True),              # 21.1, 17.8
    ((6, 256, 14, 14), 256, True),              # 23.0, 20.7
    ((12, 256, 10, 10), 256, True),             # 23.6, 20.8
    ((13, 384, 65, 16), 16, True),              # 45, 23: fp32 workgroups a quarter full
    ((9, 512, 20, 24), 64, True),               # 35, 20
    ((16, 32, 16, 58), 300, False),             # 24.8, 29.6: a nearly empty second round of workgroups
    ((4, 512, 10, 60), 64, False),              # 20.4, 23.4
    ((12, 128, 43, 14), 128, False),            # 20.3, 24.6
    ((3, 200, 9, 70), 192, False),              # 19.3, 20.8
])
def test_winograd_nodes_take_the_bf16_matrix_cores_where_they_are_faster(pkg, monkeypatch, xs, o, three_part):
    """18 to 36 million (tile, output channel, input channel) triples."""
    for name in ("KXC_HIP_WINOGRAD_BF16X3", "KXC_HIP_WINOGRAD_VARIANT"):
        monkeypatch.delenv(name, raising=False)
    assert pkg.conv2d_winograd_variant(xs, (o, xs[1], 3, 3)).endswith("_bf16x3") == three_part
