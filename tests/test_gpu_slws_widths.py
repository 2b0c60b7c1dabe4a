"""Pooled lookups at the edges of the dispatch: row widths around each lane
count (a lane reads one or four bytes of a row), bag counts around each change of
kernel, rows that do and do not start on a word."""
import numpy as np
import pytest

from glow_amd import capi
from oracle import glow_oracle as go
from tests import cases
from tests.test_gpu_slws_fused import bag_magnitude, check

pytestmark = [pytest.mark.gpu, pytest.mark.fused_math]


@pytest.fixture(scope="module", autouse=True)
def _device():
    capi.init(0)
    yield
    capi.sync()


def _batch(kind, cols, bags, mean, seed):
    rng = np.random.default_rng(seed)
    table = cases.random_fused_table(rng, 500, cols, kind)
    lengths, idx, w = cases.slws_batch(seed, 500, bags, mean, 1.05, np.int64)
    lengths[bags // 2] = 0
    total = int(lengths.sum())
    return table, lengths, idx[:total], w[:total]


def _run(kind, cols, bags, mean, seed):
    print("lookup", kind, cols, bags, flush=True)
    table, lengths, idx, w = _batch(kind, cols, bags, mean, seed)
    f16 = kind in (capi.FUSED_U8_F16, capi.FUSED_U4_F16)
    want = go.frwq_slws_generic(table, kind, w, idx, lengths, f16, False)
    strict = capi.frwq_slws(table, kind, w, idx, lengths, f16,
                            opts=capi.LaunchOpts(slws_math=capi.SLWS_MATH_STRICT))
    assert np.array_equal(strict.view(np.uint8), want.view(np.uint8))
    for offsets in (False, True):
        got = capi.frwq_slws(table, kind, w, idx, lengths, f16, bag_offsets=offsets)
        check(got.astype(np.float32), want.astype(np.float32),
              bag_magnitude(table, kind, w, idx, lengths), f16, what=f"offsets={offsets}")


@pytest.mark.parametrize("cols", [4, 12, 16, 20, 28, 32, 36, 60, 64, 68, 100, 124, 128, 132, 200,
                                  252, 256, 260, 30])
@pytest.mark.parametrize("kind", [capi.FUSED_U8_F32, capi.FUSED_U4_F16])
def test_row_widths(kind, cols):
    _run(kind, cols * 2 if kind == capi.FUSED_U4_F16 else cols, 37, 25, cols)


@pytest.mark.parametrize("bags", [1, 1023, 2047, 2048, 4097, 12288, 12289, 16383, 16384, 16385])
@pytest.mark.parametrize("kind,cols", [(capi.FUSED_U8_F32, 16), (capi.FUSED_U8_F16, 48),
                                       (capi.FUSED_U4_F32, 96), (capi.FUSED_U8_F32, 100)])
def test_bag_counts(kind, cols, bags):
    _run(kind, cols, bags, 3, bags)


def test_one_huge_length_among_short_rows():
    """Lengths past what the index list holds empty the bags behind them."""
    table, lengths, idx, w = _batch(capi.FUSED_U8_F32, 64, 12500, 2, 3)
    lengths = lengths.copy()
    lengths[6000] = 2 ** 31 - 1
    got = capi.frwq_slws(table, capi.FUSED_U8_F32, w, idx, lengths)
    assert np.all(got[6001:] == 0)
    ref = lengths.copy()
    ref[6000] = len(idx) - int(lengths[:6000].sum())
    ref[6001:] = 0
    want = go.frwq_slws_f32(table, w, idx, ref)
    check(got, want, bag_magnitude(table, 0, w, idx, ref), what="huge length")


@pytest.mark.parametrize("cols,bags", [(128, 1500), (128, 9000), (128, 16383), (128, 20000), (64, 9000),
                                       (64, 12500), (64, 20000), (16, 5000), (300, 9000)])
@pytest.mark.parametrize("long", [2 ** 31 - 1, 140_000])
@pytest.mark.parametrize("shift", [0, 1])
def test_positions_behind_long_bags(cols, bags, long, shift):
    """Lengths that no 32-bit sum holds, in one block, one wave's share and different
    chunks of the bags: a bag starts where the lengths in front of it say, which behind
    them is past the list. And bags too long for a 32-bit sum of many, all in the list.
    Lengths at a 16-byte boundary and off it; the fused kernels and the strict ones.
    Small whole numbers (sums below 2^24), so that every order of a sum is exact."""
    rng = np.random.default_rng(bags + cols)
    table = np.zeros((500, cols + 8), np.uint8)
    table[:, :cols] = rng.integers(0, 8, (500, cols))
    table[:, cols:].view(np.float32)[:] = [1.0, -2.0]
    lengths = rng.integers(0, 4, bags).astype(np.int32)
    at = [bags // 3, bags // 3 + 1, 2 * bags // 3, bags - 5]
    lengths[at] = long
    n = int(lengths.sum(dtype=np.int64)) if long < 10 ** 6 else 2 * bags
    idx = rng.integers(0, 500, n).astype(np.int64)
    w = rng.integers(1, 4, n).astype(np.float32)
    ends = np.minimum(np.cumsum(lengths.astype(np.int64)), n)
    ref = np.diff(np.r_[0, ends]).astype(np.int32)
    want = go.frwq_slws_f32(table, w, idx, ref)
    dt, dw, di = capi.to_device(table), capi.to_device(w), capi.to_device(idx)
    dl = capi.to_device(np.r_[np.full(shift, 9, np.int32), lengths])
    out = capi.DeviceBuffer.empty((bags, cols), np.float32)
    for math in (capi.SLWS_MATH_STRICT, capi.SLWS_MATH_ELEMENT):
        print("long bags", cols, bags, long, shift, math, flush=True)
        capi.launch_frwq_slws(out, False, dt, 500, 0, dw, False, di, True, n, dl.ptr + 4 * shift, bags,
                              table.shape[1], cols, opts=capi.LaunchOpts(slws_math=math))
        assert np.array_equal(out.numpy(), want), math


@pytest.mark.parametrize("cols,bags", [(128, 1900), (128, 16383), (128, 20000), (64, 20000)])
def test_positions_in_a_list_of_more_than_2_to_26_lookups(cols, bags):
    """Lists as long as that are summed in 64 bits. Every lookup of a bag names the same
    row, so that a bag's sum says whether it began in the right place."""
    rng = np.random.default_rng(bags)
    mean = 2 ** 26 // bags + 1
    lengths = rng.integers(mean, mean + 9, bags).astype(np.int32)
    rows = (np.arange(bags) * 7 % 500).astype(np.int32)
    idx = np.repeat(rows, lengths)
    assert len(idx) >= 2 ** 26
    table = np.zeros((500, cols + 8), np.uint8)
    table[:, :cols] = rng.integers(0, 8, (500, cols))
    table[:, cols:].view(np.float32)[:] = [1.0, 0.0]
    want = table[rows, :cols].astype(np.float32) * lengths[:, None]
    lengths[-4:] = 2 ** 31 - 1             # the first of them takes what is left
    rest = len(idx) - int(lengths[:-4].sum(dtype=np.int64))
    want[-4] = np.bincount(idx[-rest:], minlength=500).astype(np.float64) @ table[:, :cols]
    want[-3:] = 0
    dt, di, dl = capi.to_device(table), capi.to_device(idx), capi.to_device(lengths)
    out = capi.DeviceBuffer.empty((bags, cols), np.float32)
    for math in (capi.SLWS_MATH_STRICT, capi.SLWS_MATH_ELEMENT):
        print("long list", cols, bags, math, flush=True)
        capi.launch_frwq_slws(out, False, dt, 500, 0, None, False, di, False, len(idx), dl, bags,
                              table.shape[1], cols, opts=capi.LaunchOpts(slws_math=math))
        assert np.array_equal(out.numpy(), want), math
