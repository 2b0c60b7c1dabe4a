"""Products over rows that start at any byte: pointers off a word by every number of bytes, row
lengths around a load and a K step, both sides of the lines between the kernels that read
them, against the oracle. The bytes around the operands differ between two runs of a launch,
which must give the same results."""
import numpy as np
import pytest

from glow_amd import capi
from oracle import glow_oracle as go
from tests import cases
from tests.tiles import forced_tile

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _device():
    capi.init(0)
    yield
    capi.sync()


def _at(a, off, fill):
    """The device address of `a`, `off` bytes into a buffer of `fill`."""
    buf = np.full(a.nbytes + 64, fill, np.int8)
    buf[16 + off:16 + off + a.nbytes] = a.reshape(-1)
    d = capi.to_device(buf)
    return d, d.ptr + 16 + off


def _run(M, K, N, off_x=0, off_w=0, symmetric=True, sums=True):
    print("fc", M, K, N, off_x, off_w, symmetric, sums, flush=True)
    c = cases.rwq_fc_case(M + K, M, K, N, symmetric=symmetric, bias_i8=False)
    x, w, bias, w_offs, *params, out_off, in_off, bias_off = cases.rwq_fc_args(c)
    want = go.rwq_fc_i8(*cases.rwq_fc_args(c))
    vectors = [capi.to_device(np.ascontiguousarray(v, np.int32)) for v in (w_offs, *params)]
    d_bias = capi.to_device(np.ascontiguousarray(bias, np.int32))
    d_sums = capi.to_device(w.astype(np.int32).sum(1).astype(np.int32)) if sums else None
    for fill in (-128, 127):
        dx, px = _at(np.ascontiguousarray(x, np.int8), off_x, fill)
        dw, pw = _at(np.ascontiguousarray(w, np.int8), off_w, fill)
        out = capi.DeviceBuffer.empty((M, N), np.int8)
        capi.launch_rwq_fc_i8(out, px, pw, d_bias, 0, *vectors, M, K, N, out_off, in_off, bias_off,
                              w_offsets_all_zero=symmetric, w_row_sums=d_sums)
        np.testing.assert_array_equal(out.numpy(), want)
        del dx, dw


# 16x16 and 32x32 tiles: every offset of either operand within a word, rows of whole words
# (two ways of reading) and of any length
@pytest.mark.parametrize("M,N", [(33, 50), (300, 400)])
@pytest.mark.parametrize("K", [31, 64, 77, 100, 130, 1026])
def test_offsets_of_small_products(M, N, K):
    for off_x, off_w in ((0, 0), (1, 0), (0, 3), (2, 1), (3, 2), (4, 8)):
        _run(M, K, N, off_x, off_w)
    _run(M, K, N, 1, 2, symmetric=False)
    _run(M, K, N, 3, 0, symmetric=False, sums=False)


# the tiles behind them: rows below one step, whole steps, one byte to 63 past them, at any
# offset
@pytest.mark.parametrize("tile", [1, 2, 3])
@pytest.mark.parametrize("K", [5, 16, 47, 63, 64, 65, 79, 80, 127, 129, 200, 447, 833])
def test_last_step_of_the_tiles(tile, K):
    with forced_tile(tile):
        for off_x, off_w in ((1, 0), (0, 3), (3, 1)):
            _run(150, K, 140, off_x, off_w)
        _run(70, K, 130, 2, 1, symmetric=False)
        _run(70, K, 130, 2, 1, sums=False)


# the lines of the rules: 3 and 2 small tiles per unit at any byte, 4 and 3 in words; 512 tiles
# of 64x64, 256 of 128x128, of which a last column would be half empty or not
@pytest.mark.parametrize("M,K,N", [(1536, 203, 512), (1537, 203, 512), (1024, 415, 512),
                                   (1025, 415, 512), (512, 801, 512), (513, 801, 512),
                                   (2048, 300, 512), (2049, 300, 512), (1536, 1028, 512),
                                   (1537, 1028, 512), (2048, 130, 1024), (2049, 131, 1024),
                                   (4096, 67, 1024), (4096, 67, 1090), (8192, 41, 500)])
def test_lines_between_kernels(M, K, N):
    _run(M, K, N)


# rows short enough for loads of sixteen bytes off a word, and the first that come by words: 16x16
# tiles up to one per unit and more, 32x32 tiles one, two and three per unit, lengths around a
# multiple of 128
@pytest.mark.parametrize("M,N,line", [(40, 70, 640), (300, 300, 240), (400, 450, 350), (600, 600, 120),
                                      (600, 600, 180), (1000, 600, 120), (40, 70, 256), (40, 70, 384)])
def test_line_of_the_byte_shift(M, N, line):
    for K in (line - 6, line - 5, line - 2, line - 1, line + 1, line + 2, line + 5, line + 6):
        _run(M, K, N)
    _run(M, line - 1, N, 1, 2, symmetric=False)
    _run(M, line + 1, N, 2, 1, symmetric=False)
    _run(M, line, N, 3, 1)
    _run(M, line - 4, N, 0, 3)
