"""The streaming kernel for short K and many rows (tile 8): FullyConnected and
pointwise convolutions over 64, 128 or 256 inputs, against the oracle and the
tiled kernels, with column slices, row tails, strides, the fused residual add
and Relu, and the requantisation hints.

Run on the GPU box:  python -u -m pytest tests -m gpu -x -v --timeout 120
"""
import numpy as np
import pytest

from glow_amd import capi
from oracle import glow_oracle as go
from tests import cases, tiles

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _device():
    capi.init(0)
    yield
    capi.sync()


def say(*a):
    print(*a, flush=True)


class forced_tile:
    def __init__(self, tile):
        self.tile = tile

    def __enter__(self):
        capi.check(capi.lib().mi355x_gemm_tile_override(self.tile))

    def __exit__(self, *exc):
        capi.check(capi.lib().mi355x_gemm_tile_override(-1))
        return False


FC_SHAPES = [
    # M, K, N: row tails, one and several column slices, more tiles than waves
    (1, 64, 32), (33, 64, 64), (1000, 64, 256), (257, 128, 512), (4096, 256, 64),
    (70, 256, 384), (20000, 64, 96), (129, 128, 1024),
]


@pytest.mark.parametrize("shape", FC_SHAPES)
def test_stream_fc_vs_oracle(shape):
    M, K, N = shape
    c = cases.rwq_fc_case(800 + M + K, M, K, N)
    c["w_offsets"][:] = 0          # what the kernel takes: symmetric weights
    want = go.rwq_fc_i8(*cases.rwq_fc_args(c))
    say("stream fc", shape)
    with forced_tile(8):
        got = capi.rwq_fc_i8(*cases.rwq_fc_args(c))
    np.testing.assert_array_equal(got, want)
    assert want.std() > 5
    # with the requantisation hint the backend derives for these constants
    hint = capi.gemm_requant_hint_host(K, c["in_offset"], c["out_offset"], c["w_offsets"],
                                       c["bias"], c["bias_offset"], c["bias_pre"], c["bias_post"],
                                       c["bias_scale"], c["out_pre"], c["out_post"], c["out_scale"])
    with forced_tile(8), capi.requant_hint(hint):
        np.testing.assert_array_equal(capi.rwq_fc_i8(*cases.rwq_fc_args(c)), want)
    # no input offset (no use of the weight row sums), int8 bias
    c2 = cases.rwq_fc_case(801 + M, M, K, N, in_offset=0, bias_i8=True, bias_scale=0.01,
                           bias_offset=3)
    c2["w_offsets"][:] = 0
    with forced_tile(8):
        np.testing.assert_array_equal(capi.rwq_fc_i8(*cases.rwq_fc_args(c2)),
                                      go.rwq_fc_i8(*cases.rwq_fc_args(c2)))


def test_stream_refuses_what_it_cannot_run():
    """Weight offsets (row sums of A would be needed), other K, sums not
    precomputed: asked for by number (tile 8) the kernel refuses the launch,
    and the shape rule runs the tiled kernels."""
    for K, kw, sums in ((64, dict(symmetric=False), True), (192, dict(), True),
                        (64, dict(in_offset=5), False),   # an input offset needs the row sums
                        (320, dict(), True)):
        c = cases.rwq_fc_case(850 + K, 100, K, 64, **kw)
        if kw.get("symmetric", True):
            c["w_offsets"][:] = 0
        want = go.rwq_fc_i8(*cases.rwq_fc_args(c))
        assert tiles.refused(8, lambda: capi.rwq_fc_i8(*cases.rwq_fc_args(c),
                                                       precomputed_sums=sums))
        got = capi.rwq_fc_i8(*cases.rwq_fc_args(c), precomputed_sums=sums)
        np.testing.assert_array_equal(got, want)


CONV_CASES = [
    dict(N=2, H=56, W=56, IC=64, OC=256),                              # ResNet stage 1
    dict(N=1, H=28, W=28, IC=128, OC=512, in_offset=-128),
    dict(N=3, H=9, W=7, IC=256, OC=96, act=go.ACT_CLIP, in_offset=3),
    dict(N=2, H=56, W=56, IC=256, OC=512, stride=(2, 2)),              # strided shortcut
    dict(N=1, H=15, W=13, IC=64, OC=64, stride=(2, 3), act=go.ACT_LEAKY_RELU, out_offset=10),
    dict(N=1, H=5, W=5, IC=128, OC=32, bias_i8=True, act=go.ACT_NONE, in_offset=-5),
]


@pytest.mark.parametrize("kw", CONV_CASES)
def test_stream_pointwise_conv_vs_oracle(kw):
    kw = dict(kw)
    kw.setdefault("in_offset", -128)
    c = cases.cwq_conv_case(61, kernel=(1, 1), pads=(0, 0, 0, 0), **kw)
    g = c["geom"]
    say("stream conv", kw, "output", g.OH, "x", g.OW)
    want = go.cwq_conv2d_i8(*cases.cwq_conv_args(c))
    with forced_tile(8):
        got = capi.cwq_conv2d_i8(*cases.cwq_conv_args(c))
    np.testing.assert_array_equal(got, want)
    with forced_tile(1):
        np.testing.assert_array_equal(capi.cwq_conv2d_i8(*cases.cwq_conv_args(c)), want)
    hint = capi.gemm_requant_hint_host(g.IC, c["in_offset"], c["out_offset"], c["f_offsets"],
                                       c["bias"], 0, c["bias_pre"], c["bias_post"], c["bias_scale"],
                                       c["out_pre"], c["out_post"], c["out_scale"],
                                       bias_offsets=c["b_offsets"])
    with forced_tile(8), capi.requant_hint(hint):
        np.testing.assert_array_equal(capi.cwq_conv2d_i8(*cases.cwq_conv_args(c)), want)
    assert want.std() > 1


WINDOW_CASES = [
    # the stem of an image network after space-to-depth: 4x4 over 16 channels
    dict(N=2, H=115, W=115, IC=16, OC=64, kernel=(4, 4)),
    dict(N=1, H=9, W=11, IC=16, OC=32, kernel=(2, 2), act=go.ACT_CLIP),             # K 64
    dict(N=3, H=8, W=8, IC=32, OC=96, kernel=(2, 2), stride=(2, 2), in_offset=4),   # K 128
    dict(N=1, H=10, W=7, IC=64, OC=64, kernel=(2, 2), stride=(1, 2)),               # K 256
    dict(N=2, H=6, W=12, IC=16, OC=256, kernel=(2, 8), act=go.ACT_LEAKY_RELU),      # rows of 128 bytes
    dict(N=1, H=7, W=7, IC=32, OC=64, kernel=(4, 1), bias_i8=True),                 # rows of 32 bytes
]


@pytest.mark.parametrize("kw", WINDOW_CASES)
def test_stream_window_conv_vs_oracle(kw):
    """Windows without padding whose rows are whole 32-byte chunks run on the
    streaming kernel as rows of several segments."""
    kw = dict(kw)
    kw.setdefault("in_offset", -128)
    c = cases.cwq_conv_case(63, pads=(0, 0, 0, 0), **kw)
    g = c["geom"]
    say("stream window conv", kw, "output", g.OH, "x", g.OW)
    want = go.cwq_conv2d_i8(*cases.cwq_conv_args(c))
    with forced_tile(8):
        got = capi.cwq_conv2d_i8(*cases.cwq_conv_args(c))
    np.testing.assert_array_equal(got, want)
    with forced_tile(2):
        np.testing.assert_array_equal(capi.cwq_conv2d_i8(*cases.cwq_conv_args(c)), want)
    assert want.std() > 1


@pytest.mark.parametrize("relu", [False, True])
@pytest.mark.parametrize("IC,OC", [(64, 256), (128, 512), (256, 1024)])
def test_stream_conv_with_fused_residual_add(IC, OC, relu):
    c = cases.cwq_conv_case(71 + IC, 2, 14, 14, IC, OC, kernel=(1, 1), pads=(0, 0, 0, 0),
                            act=go.ACT_NONE, in_offset=-128, out_offset=6)
    conv = go.cwq_conv2d_i8(*cases.cwq_conv_args(c))
    rng = np.random.default_rng(72)
    res = rng.integers(-128, 128, conv.shape).astype(np.int8)
    p = lambda r: go.quantize_scale_offset_32to8(float(np.float32(r)), 0)[:3]
    cs, rs, ss, ds = np.float32(c["out_scale_f"]), np.float32(0.09), np.float32(0.13), np.float32(0.2)
    cp, rp, dp = p(cs / ss), p(rs / ss), p(ss / ds)
    want = go.add_i8(conv, res, 11, c["out_offset"], -20, cp, rp)
    if relu:
        want = go.relu_i8(want, 11, -128, dp)
    add = capi.fused_add(11, -20, cp, rp, relu, -128, dp)
    with forced_tile(8):
        got = capi.cwq_conv2d_add_i8(*cases.cwq_conv_args(c), res, add)
    np.testing.assert_array_equal(got, want)


def test_stream_conv_full_batch():
    """The first ResNet stage's pointwise layer with the residual at batch 64:
    two images on the oracle, the rest through batch independence."""
    c = cases.cwq_conv_case(91, 64, 56, 56, 64, 256, kernel=(1, 1), pads=(0, 0, 0, 0),
                            in_offset=-128)
    c["x"][2::2] = c["x"][0]
    c["x"][3::2] = c["x"][1]
    with forced_tile(8):
        got = capi.cwq_conv2d_i8(*cases.cwq_conv_args(c))
    c2 = dict(c, x=c["x"][:2], geom=go.conv_geom(2, 56, 56, 64, 256, (1, 1), (1, 1), (0, 0, 0, 0)))
    want = go.cwq_conv2d_i8(*cases.cwq_conv_args(c2))
    np.testing.assert_array_equal(got[:2], want)
    for i in range(2, 64):
        np.testing.assert_array_equal(got[i], want[i % 2])


@pytest.mark.parametrize("IC,OC,slow", [(64, 64, False), (128, 96, False), (64, 32, True),
                                        (128, 256, True), (64, 128, False)])
def test_stream_add_narrow_slices_and_general_scales(IC, OC, slow):
    """Slices of 32, 64 and 96 columns (two and four passes of the copy-out,
    lanes past the tile's rows) with the residual, and add parameters outside
    the short form (a pre-shift, a scale beyond 23 bits)."""
    c = cases.cwq_conv_case(75 + IC + OC, 3, 11, 13, IC, OC, kernel=(1, 1), pads=(0, 0, 0, 0),
                            act=go.ACT_NONE, in_offset=-128, out_offset=-3)
    conv = go.cwq_conv2d_i8(*cases.cwq_conv_args(c))
    rng = np.random.default_rng(76)
    res = rng.integers(-128, 128, conv.shape).astype(np.int8)
    p = lambda r: go.quantize_scale_offset_32to8(float(np.float32(r)), 0)[:3]
    cp, rp, dp = p(0.8), p(0.61), p(0.7)
    if slow:
        cp = (1, cp[1], cp[2] * 2)                 # the same ratio through a pre-shift
        rp = (0, 24, int(round(0.61 * (1 << 24))))
    want = go.relu_i8(go.add_i8(conv, res, 7, c["out_offset"], -9, cp, rp), 7, -128, dp)
    add = capi.fused_add(7, -9, cp, rp, True, -128, dp)
    say("stream add", IC, OC, "slow" if slow else "short form", cp, rp)
    with forced_tile(8):
        got = capi.cwq_conv2d_add_i8(*cases.cwq_conv_args(c), res, add)
    np.testing.assert_array_equal(got, want)
    with forced_tile(2):
        np.testing.assert_array_equal(capi.cwq_conv2d_add_i8(*cases.cwq_conv_args(c), res, add), want)
    assert len(np.unique(want)) > 20


def test_stream_add_several_tiles_per_wave():
    """More 32-row tiles than the launch has waves, with the residual: a wave's
    next rows and residual bytes are asked for while it works on a tile. Two
    images and two residual images on the oracle, the rest through batch
    independence."""
    n = 44                                           # 137984 rows = 4312 tiles
    c = cases.cwq_conv_case(93, n, 56, 56, 64, 64, kernel=(1, 1), pads=(0, 0, 0, 0),
                            act=go.ACT_NONE, in_offset=-128)
    c["x"][2::2] = c["x"][0]
    c["x"][3::2] = c["x"][1]
    rng = np.random.default_rng(94)
    res = np.empty((n, 56, 56, 64), np.int8)
    res[0::2] = rng.integers(-128, 128, (56, 56, 64)).astype(np.int8)
    res[1::2] = rng.integers(-128, 128, (56, 56, 64)).astype(np.int8)
    p = lambda r: go.quantize_scale_offset_32to8(float(np.float32(r)), 0)[:3]
    cp, rp, dp = p(0.9), p(0.5), p(0.66)
    add = capi.fused_add(2, 5, cp, rp, True, -128, dp)
    with forced_tile(8):
        got = capi.cwq_conv2d_add_i8(*cases.cwq_conv_args(c), res, add)
    c2 = dict(c, x=c["x"][:2], geom=go.conv_geom(2, 56, 56, 64, 64, (1, 1), (1, 1), (0, 0, 0, 0)))
    conv = go.cwq_conv2d_i8(*cases.cwq_conv_args(c2))
    want = go.relu_i8(go.add_i8(conv, res[:2], 2, c["out_offset"], 5, cp, rp), 2, -128, dp)
    for i in range(n):
        np.testing.assert_array_equal(got[i], want[i % 2])
    assert len(np.unique(want)) > 20


# rescale triples (pre, post, scale) at the lines of the add in words: a post-shift of 16
# and one beyond, the largest scale that a post-shift of 16, 9 and 0 leaves room for (2^22
# scaled up) and one beyond, negative scales
ADD_LINES = [(0, 16, 40000), (0, 17, 80000), (0, 16, 1 << 22), (0, 16, (1 << 22) + 1),
             (0, 9, 1 << 15), (0, 9, (1 << 15) + 1), (0, 9, 300), (0, 0, 64), (0, 0, 65), (0, 0, 1),
             (0, 16, -(1 << 22)), (0, 9, -300), (0, 31, 1 << 22)]


@pytest.mark.parametrize("line", ADD_LINES)
@pytest.mark.parametrize("swap", [False, True])
def test_add_in_words_at_its_lines(line, swap):
    """The fused add and the separate instructions, with each operand's rescale at the
    lines of the add in words, and offsets at the ends of their range and outside."""
    c = cases.cwq_conv_case(61, 1, 65, 64, 64, 64, kernel=(1, 1), pads=(0, 0, 0, 0),
                            act=go.ACT_NONE, in_offset=-128, out_offset=-128 if swap else 127)
    conv = go.cwq_conv2d_i8(*cases.cwq_conv_args(c))
    res = np.random.default_rng(62).integers(-128, 128, conv.shape).astype(np.int8)
    cp, rp, dp = line, (0, 9, 411), (0, 8, 282)
    if swap:
        cp, rp = rp, cp
    say("add in words", cp, rp)
    for sum_off, res_off, relu in ((127, -128, True), (-128, 127, True), (11, 200, True), (300, 5, False)):
        want = go.add_i8(conv, res, sum_off, c["out_offset"], res_off, cp, rp)
        if relu:
            want = go.relu_i8(want, sum_off, -128, dp)
        add = capi.fused_add(sum_off, res_off, cp, rp, relu, -128, dp)
        for tile in (8, 2, 5):
            with forced_tile(tile):
                got = capi.cwq_conv2d_add_i8(*cases.cwq_conv_args(c), res, add)
            np.testing.assert_array_equal(got, want)


@pytest.mark.parametrize("OC", [32, 64, 96, 256])
@pytest.mark.parametrize("IC", [64, 128, 256])
def test_every_variant_of_the_kernel(IC, OC):
    """A kernel per number of copy-out passes, residual and requantisation variant, on rows
    that do not fill their last tile and on as many tiles as leave some waves without one."""
    p = lambda r: go.quantize_scale_offset_32to8(float(np.float32(r)), 0)[:3]
    for act, H, W in ((go.ACT_RELU, 13, 11), (go.ACT_LEAKY_RELU, 1, 1), (go.ACT_NONE, 13, 41)):
        c = cases.cwq_conv_case(81 + IC + OC, 1, H, W, IC, OC, kernel=(1, 1), pads=(0, 0, 0, 0),
                                act=act, in_offset=-128, out_offset=-3)
        conv = go.cwq_conv2d_i8(*cases.cwq_conv_args(c))
        res = np.random.default_rng(82).integers(-128, 128, conv.shape).astype(np.int8)
        cp, rp, dp = p(0.8), p(0.61), p(0.7)
        want = go.relu_i8(go.add_i8(conv, res, 7, c["out_offset"], -9, cp, rp), 7, -128, dp)
        add = capi.fused_add(7, -9, cp, rp, True, -128, dp)
        derived = capi.gemm_requant_hint_host(IC, c["in_offset"], c["out_offset"], c["f_offsets"],
                                              c["bias"], 0, c["bias_pre"], c["bias_post"],
                                              c["bias_scale"], c["out_pre"], c["out_post"],
                                              c["out_scale"], bias_offsets=c["b_offsets"])
        say("stream variants", IC, OC, "act", act, H, "x", W, "hint", derived)
        for hint in sorted({0, derived & 1, derived}):
            with forced_tile(8), capi.requant_hint(hint):
                np.testing.assert_array_equal(capi.cwq_conv2d_i8(*cases.cwq_conv_args(c)), conv)
                np.testing.assert_array_equal(
                    capi.cwq_conv2d_add_i8(*cases.cwq_conv_args(c), res, add), want)


@pytest.mark.parametrize("M", [5119, 5120, 5151])
@pytest.mark.parametrize("K", [32, 96])
def test_line_of_short_rows(K, M):
    """K of 32 and 96 runs here by the shape rule alone, from 5 x 2^19 results on."""
    c = cases.rwq_fc_case(870 + K + M, M, K, 512)
    c["w_offsets"][:] = 0
    want = go.rwq_fc_i8(*cases.rwq_fc_args(c))
    say("short rows", K, M)
    np.testing.assert_array_equal(capi.rwq_fc_i8(*cases.rwq_fc_args(c)), want)
    assert tiles.refused(8, lambda: capi.rwq_fc_i8(*cases.rwq_fc_args(c)))


SHORT_CONVS = [
    dict(H=149, W=331, IC=32, OC=32, kernel=(1, 1)),                    # 49 319 rows, narrow
    dict(H=101, W=67, IC=96, OC=512, kernel=(1, 1)),
    dict(H=301, W=202, IC=32, OC=96, kernel=(1, 1), stride=(2, 1)),
    dict(H=150, W=150, IC=16, OC=128, kernel=(3, 2)),                   # K 96 as rows of 32 bytes
]


@pytest.mark.parametrize("kw", SHORT_CONVS)
def test_short_rows_with_the_residual(kw):
    c = cases.cwq_conv_case(64, N=1, pads=(0, 0, 0, 0), act=go.ACT_NONE, in_offset=-128,
                            out_offset=-3, **kw)
    g = c["geom"]
    conv = go.cwq_conv2d_i8(*cases.cwq_conv_args(c))
    res = np.random.default_rng(83).integers(-128, 128, conv.shape).astype(np.int8)
    p = lambda r: go.quantize_scale_offset_32to8(float(np.float32(r)), 0)[:3]
    cp, rp, dp = p(0.8), p(0.61), p(0.7)
    want = go.relu_i8(go.add_i8(conv, res, 7, c["out_offset"], -9, cp, rp), 7, -128, dp)
    add = capi.fused_add(7, -9, cp, rp, True, -128, dp)
    K = g.KH * g.KW * g.IC
    hint = capi.gemm_requant_hint_host(K, c["in_offset"], c["out_offset"], c["f_offsets"],
                                       c["bias"], 0, c["bias_pre"], c["bias_post"], c["bias_scale"],
                                       c["out_pre"], c["out_post"], c["out_scale"],
                                       bias_offsets=c["b_offsets"])
    say("short rows", kw, "rows", g.OH * g.OW, "hint", hint)
    for h in sorted({0, hint}):
        with capi.requant_hint(h):
            np.testing.assert_array_equal(capi.cwq_conv2d_i8(*cases.cwq_conv_args(c)), conv)
            np.testing.assert_array_equal(
                capi.cwq_conv2d_add_i8(*cases.cwq_conv_args(c), res, add), want)


@pytest.mark.parametrize("IC,OC", [(32, 32), (32, 96), (96, 64), (96, 512)])
def test_short_rows_leaky_relu(IC, OC):
    """The variant of K 32 and 96 that test_every_variant_of_the_kernel, which asks for the
    kernel by number, cannot reach; with and without the residual."""
    c = cases.cwq_conv_case(91 + IC + OC, N=1, H=149, W=331, IC=IC, OC=OC, kernel=(1, 1),
                            pads=(0, 0, 0, 0), act=go.ACT_LEAKY_RELU, in_offset=-128, out_offset=-3)
    say("short rows, leaky", IC, OC)
    conv = go.cwq_conv2d_i8(*cases.cwq_conv_args(c))
    np.testing.assert_array_equal(capi.cwq_conv2d_i8(*cases.cwq_conv_args(c)), conv)
    res = np.random.default_rng(84).integers(-128, 128, conv.shape).astype(np.int8)
    p = lambda r: go.quantize_scale_offset_32to8(float(np.float32(r)), 0)[:3]
    cp, rp, dp = p(0.8), p(0.61), p(0.7)
    want = go.relu_i8(go.add_i8(conv, res, 7, c["out_offset"], -9, cp, rp), 7, -128, dp)
    add = capi.fused_add(7, -9, cp, rp, True, -128, dp)
    np.testing.assert_array_equal(capi.cwq_conv2d_add_i8(*cases.cwq_conv_args(c), res, add), want)


# windows with K of 256 around two and three 32x32 tiles per unit: up to 64 columns the
# streaming kernel follows on the one for small products, wider ones the tiled kernels do
@pytest.mark.parametrize("H,W,IC,k,OC", [(64, 128, 16, 4, 64), (65, 128, 16, 4, 64), (96, 128, 64, 2, 64),
                                         (97, 128, 64, 2, 64), (129, 128, 16, 4, 32),
                                         (65, 64, 64, 2, 128), (97, 64, 64, 2, 128)])
def test_lines_of_windows_over_256_bytes(H, W, IC, k, OC):
    c = cases.cwq_conv_case(17 + H + OC, 1, H + k - 1, W + k - 1, IC, OC, kernel=(k, k),
                            pads=(0, 0, 0, 0), act=go.ACT_RELU, in_offset=-128, out_offset=-3)
    say("windows of 256 bytes", H, W, IC, k, OC)
    np.testing.assert_array_equal(capi.cwq_conv2d_i8(*cases.cwq_conv_args(c)),
                                  go.cwq_conv2d_i8(*cases.cwq_conv_args(c)))
