"""Small products (16x16 or 32x32 tiles, the K loop split over the waves of a workgroup)
against the oracle at the edges of its tiles, K steps and ways of reading rows, on
both sides of the line to the kernels for larger problems; and those kernels'
partial last K step."""
import numpy as np
import pytest

from glow_amd import capi
from oracle import glow_oracle as go
from tests import cases

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _device():
    capi.init(0)
    yield
    capi.sync()


def _fc(M, K, N):
    for seed, sym, b8 in ((1, True, False), (2, False, True)):
        print("fc", M, K, N, sym, flush=True)
        c = cases.rwq_fc_case(seed + K, M, K, N, symmetric=sym, bias_i8=b8)
        args = cases.rwq_fc_args(c)
        want = go.rwq_fc_i8(*args)
        np.testing.assert_array_equal(capi.rwq_fc_i8(*args), want)
        np.testing.assert_array_equal(capi.rwq_fc_i8(*args, precomputed_sums=False), want)


# a row shorter than one load, its end in either half of a step, whole chunks; more
# steps than one round of every wave
@pytest.mark.parametrize("K", [1, 13, 15, 16, 17, 31, 32, 33, 48, 63, 64, 65, 127, 255, 272, 415,
                               1023, 1024, 1025, 2080])
def test_row_lengths(K):
    _fc(45, K, 70)


# 32x32 tiles (1.6 16x16 tiles per unit and more): a wave's steps below, at and past the
# eight it asks for ahead, and past twice as many
@pytest.mark.parametrize("K", [1, 17, 32, 33, 130, 480, 1023, 1024, 1056, 2047, 2080, 3105])
def test_row_lengths_32x32_tiles(K):
    _fc(300, K, 800)


# the same for the six steps of 64 bytes of 16x16 tiles
@pytest.mark.parametrize("K", [1472, 1536, 1600, 3071, 3072, 3150, 4681])
def test_long_rows_16x16_tiles(K):
    _fc(18, K, 50)


# the line between the tiles (410 16x16 tiles on 256 units; 1024 of a single column), and
# the lines to the larger kernels, which lie further out for short rows
@pytest.mark.parametrize("M,K,N", [(656, 96, 160), (657, 96, 160), (16384, 80, 16), (16385, 80, 16),
                                   (1024, 64, 1024), (1025, 64, 1024), (512, 512, 1024),
                                   (513, 512, 1024), (512, 415, 1024), (513, 415, 1024),
                                   (700, 1088, 700)])
def test_lines_between_kernels(M, K, N):
    _fc(M, K, N)


@pytest.mark.parametrize("M,N", [(1, 1), (31, 3), (32, 32), (33, 30), (1, 1029), (700, 5),
                                 (512, 512), (513, 512), (544, 481)])
@pytest.mark.parametrize("K", [64, 80, 77])
def test_tile_edges(M, N, K):
    _fc(M, K, N)


@pytest.mark.parametrize("M,N", [(5, 65536), (32, 32 * 2049), (33, 8200)])
def test_few_rows_many_columns(M, N):
    _fc(M, 1024, N)


@pytest.mark.parametrize("M,N", [(4100, 70), (1030, 1100), (2070, 1030)])
@pytest.mark.parametrize("K", [16, 48, 80, 208])
def test_partial_last_step_of_the_larger_tiles(M, N, K):
    _fc(M, K, N)


@pytest.mark.parametrize("geom", [
    dict(N=1, H=9, W=11, IC=4, OC=7),                                   # words, K 36
    dict(N=2, H=12, W=7, IC=20, OC=33, stride=(2, 2)),                  # words over taps
    dict(N=1, H=10, W=10, IC=8, OC=6, group=2, kernel=(2, 3)),          # groups of four channels
    dict(N=1, H=9, W=9, IC=16, OC=40, kernel=(5, 5), pads=(2, 2, 2, 2)),  # half steps
    dict(N=3, H=8, W=9, IC=48, OC=36, dilation=(2, 2)),                 # steps across taps
    dict(N=1, H=7, W=7, IC=96, OC=66, group=3),                         # whole steps per tap
    dict(N=1, H=7, W=7, IC=512, OC=32),                                 # many rounds
    dict(N=2, H=6, W=5, IC=3, OC=9),                                    # not readable in words
    dict(N=1, H=3, W=3, IC=1024 + 16, OC=20, kernel=(1, 1), pads=(0, 0, 0, 0)),
    dict(N=1, H=4, W=4, IC=1824, OC=8),                                 # K past the locator's range
    dict(N=7, H=62, W=38, IC=16, OC=64),                                # 4 tiles per unit, and more
    dict(N=4, H=56, W=38, IC=16, OC=128),
    dict(N=2, H=64, W=64, IC=64, OC=64),                                # 2 tiles per unit, and more
    dict(N=2, H=65, W=64, IC=64, OC=64),
    dict(N=1, H=33, W=31, IC=64, OC=48, stride=(2, 2), kernel=(1, 1), pads=(0, 0, 0, 0)),  # strided pixels
    dict(N=9, H=36, W=36, IC=24, OC=40),                                # words, 4 tiles per unit
], ids=lambda g: "-".join(str(v) for v in g.values()))
@pytest.mark.parametrize("symmetric", [True, False])
def test_windows(geom, symmetric):
    print("conv", geom, symmetric, flush=True)
    c = cases.cwq_conv_case(5, symmetric=symmetric, in_offset=-7, **geom)
    args = cases.cwq_conv_args(c)
    want = go.cwq_conv2d_i8(*args)
    np.testing.assert_array_equal(capi.cwq_conv2d_i8(*args), want)
    np.testing.assert_array_equal(capi.cwq_conv2d_i8(*args, precomputed_sums=False), want)
    rng = np.random.default_rng(6)
    res = rng.integers(-128, 128, want.shape).astype(np.int8)
    cp, rp, dp = (2, 9, 300), (1, 8, 200), (0, 7, 140)
    add = capi.fused_add(11, -20, cp, rp, True, -128, dp)
    summed = go.relu_i8(go.add_i8(want, res, 11, c["out_offset"], -20, cp, rp), 11, -128, dp)
    np.testing.assert_array_equal(capi.cwq_conv2d_add_i8(*args, res, add), summed)


# the same product as a pointwise convolution and as a FullyConnected layer at the lines
# between the kernels for small products, tiles and streamed rows (4, and 2 and 3 tiles per
# unit), which one rule draws for both
@pytest.mark.parametrize("H,W,K,N", [(64, 128, 128, 128), (64, 129, 128, 128), (128, 128, 64, 64),
                                     (64, 64, 256, 128), (64, 65, 256, 128), (64, 96, 256, 128),
                                     (64, 97, 256, 128), (128, 193, 256, 32)])
def test_lines_of_pointwise_convolutions(H, W, K, N):
    c = cases.cwq_conv_case(7 + K, 1, H, W, K, N, kernel=(1, 1), pads=(0, 0, 0, 0), act=go.ACT_RELU,
                            in_offset=-128, out_offset=-3)
    print("pointwise", H, W, K, N, flush=True)
    np.testing.assert_array_equal(capi.cwq_conv2d_i8(*cases.cwq_conv_args(c)),
                                  go.cwq_conv2d_i8(*cases.cwq_conv_args(c)))
    c = cases.rwq_fc_case(8 + K, H * W, K, N)
    c["w_offsets"][:] = 0
    np.testing.assert_array_equal(capi.rwq_fc_i8(*cases.rwq_fc_args(c)),
                                  go.rwq_fc_i8(*cases.rwq_fc_args(c)))
