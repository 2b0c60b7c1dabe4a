"""The tiles that the estimates of gemm_i8.h choose: products on either side of where the choice
changes (the row counts around it are a tile's edges as well), every column count with
remainders, with and without row sums to form, against the oracle."""
import numpy as np
import pytest

from glow_amd import capi
from oracle import glow_oracle as go
from tests import cases


@pytest.mark.gpu
@pytest.mark.parametrize("M,K,N", [
    (2049, 1088, 64), (8543, 192, 64), (2560, 512, 200), (4097, 80, 300), (1500, 448, 1030),
    (16385, 64, 130), (2421, 28, 2111), (1270, 65, 1023), (4800, 99, 470), (2600, 1030, 500),
    (66001, 64, 200), (70001, 128, 100)])
@pytest.mark.parametrize("symmetric", [True, False])
def test_dense_rows(M, K, N, symmetric):
    c = cases.rwq_fc_case(M + K, M, K, N, symmetric=symmetric)
    args = cases.rwq_fc_args(c)
    rows = np.unique(np.r_[0:70, M // 2:M // 2 + 70, M - 140:M])
    want = go.rwq_fc_i8(np.ascontiguousarray(args[0][rows]), *args[1:])
    np.testing.assert_array_equal(capi.rwq_fc_i8(*args)[rows], want)


@pytest.mark.gpu
@pytest.mark.parametrize("N,H,W,IC,OC,k,stride,group", [
    (4, 33, 30, 256, 100, 3, 2, 2), (1, 26, 27, 512, 100, 5, 1, 1), (6, 35, 35, 64, 100, 3, 1, 1),
    (3, 31, 33, 48, 72, 3, 1, 1), (12, 21, 17, 24, 130, 1, 1, 1), (9, 33, 31, 16, 128, 1, 1, 2)])
@pytest.mark.parametrize("symmetric", [True, False])
def test_windows(N, H, W, IC, OC, k, stride, group, symmetric):
    c = cases.cwq_conv_case(N + H, N, H, W, IC, OC, (k, k), (stride, stride), (k // 2,) * 4, group,
                            symmetric=symmetric, in_offset=-3)
    args = cases.cwq_conv_args(c)
    np.testing.assert_array_equal(capi.cwq_conv2d_i8(*args), go.cwq_conv2d_i8(*args))


# Either side of where the streaming kernel takes over, by rows and by results.
@pytest.mark.gpu
@pytest.mark.parametrize("K,N,line", [
    (64, 32, 28000), (64, 128, 28000), (64, 512, 9180), (128, 64, 80000), (128, 96, 60000),
    (128, 256, 39063), (256, 64, 90000), (256, 128, 60000), (256, 384, 42969), (256, 512, 4096)])
@pytest.mark.parametrize("past", [-1, 0])
def test_lines_of_the_streaming_kernel(K, N, line, past):
    M = line + past
    c = cases.rwq_fc_case(K + N, M, K, N, symmetric=True)
    c["w_offsets"][:] = 0
    args = cases.rwq_fc_args(c)
    rows = np.unique(np.r_[0:70, M // 2:M // 2 + 70, M - 140:M])
    want = go.rwq_fc_i8(np.ascontiguousarray(args[0][rows]), *args[1:])
    np.testing.assert_array_equal(capi.rwq_fc_i8(*args)[rows], want)


# Pixels apart, with the residual's kernels of the same lines: 88 x 57 of every second pixel and
# a few images less or more.
@pytest.mark.gpu
@pytest.mark.parametrize("IC,OC,images", [(64, 96, 4), (64, 256, 3), (128, 256, 3), (256, 64, 5)])
@pytest.mark.parametrize("more", [0, 1])
def test_lines_of_the_streaming_kernel_for_pixels_apart(IC, OC, images, more):
    c = cases.cwq_conv_case(IC + OC, images + more, 175, 113, IC, OC, (1, 1), (2, 2), (0,) * 4, 1,
                            symmetric=True, in_offset=-3)
    args = cases.cwq_conv_args(c)
    np.testing.assert_array_equal(capi.cwq_conv2d_i8(*args), go.cwq_conv2d_i8(*args))


# Either side of where the lines stay whatever the estimates say: few columns, many results with sums
# to form, short K.
@pytest.mark.gpu
@pytest.mark.parametrize("M,K,N", [(19073, 1408, 10), (30000, 1024, 63), (30000, 1024, 64), (62500, 192, 200),
                                   (62501, 192, 200), (121186, 64, 242), (2707, 320, 1740), (4109, 1008, 1526)])
@pytest.mark.parametrize("symmetric", [True, False])
def test_dense_rows_past_the_estimates(M, K, N, symmetric):
    test_dense_rows(M, K, N, symmetric)


@pytest.mark.gpu
@pytest.mark.parametrize("N,H,W,IC,OC,k,group", [
    (26, 49, 49, 16, 246, 2, 1), (9, 49, 49, 32, 492, 2, 2), (5, 40, 40, 112, 300, 3, 1), (5, 40, 40, 96, 300, 3, 1)])
@pytest.mark.parametrize("symmetric", [True, False])
def test_windows_past_the_estimates(N, H, W, IC, OC, k, group, symmetric):
    test_windows(N, H, W, IC, OC, k, 1, group, symmetric)


@pytest.mark.gpu
def test_windows_past_the_estimates_with_the_residual():
    """2x2 over 26x49x49, 16 -> 246: the wide tiles that the estimates ask for are not taken."""
    c = cases.cwq_conv_case(7, 26, 49, 49, 16, 246, (2, 2), (1, 1), (1, 1, 1, 1), 1, symmetric=True, in_offset=-3)
    args = cases.cwq_conv_args(c)
    conv = go.cwq_conv2d_i8(*args)
    res = np.random.default_rng(7).integers(-128, 128, conv.shape).astype(np.int8)
    cp, rp = (2, 9, 300), (1, 8, 200)
    want = go.add_i8(conv, res, 11, c["out_offset"], -20, cp, rp)
    np.testing.assert_array_equal(capi.cwq_conv2d_add_i8(*args, res, capi.fused_add(11, -20, cp, rp)), want)


# Windows whose channels are no multiple of sixteen, and rows off sixteen bytes below a step of 64:
# either side of where 128x128 tiles take them (with and without sums to form, a quarter of the
# columns past N over a long K).
@pytest.mark.gpu
@pytest.mark.parametrize("N,H,W,IC,OC,k", [
    (24, 37, 37, 24, 238, 2), (24, 37, 37, 102, 238, 2), (13, 49, 49, 149, 150, 2), (13, 49, 49, 151, 150, 2)])
@pytest.mark.parametrize("symmetric", [True, False])
def test_ragged_windows(N, H, W, IC, OC, k, symmetric):
    test_windows(N, H, W, IC, OC, k, 1, 1, symmetric)


@pytest.mark.gpu
@pytest.mark.parametrize("M,K,N", [(1007, 13, 1208), (5088, 30, 902), (9000, 63, 1100), (9000, 65, 1100), (2563, 15, 2100)])
@pytest.mark.parametrize("symmetric", [True, False])
def test_rows_around_a_step(M, K, N, symmetric):
    test_dense_rows(M, K, N, symmetric)
