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
