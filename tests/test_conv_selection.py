"""Which kernel a convolution takes, asked from the library on the host: no GPU is needed."""
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
