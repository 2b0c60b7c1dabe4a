"""Pooled lookups of many bags with sixteen bytes of a row to a lane: row widths around
what a lane and a row's lanes hold, rows at any byte, bag lengths around a round, against
the oracle and, bit for bit, against the kernels for fewer bags."""
import numpy as np
import pytest

from glow_amd import capi
from oracle import glow_oracle as go
from tests import cases
from tests.test_gpu_slws_fused import bag_magnitude, check

pytestmark = [pytest.mark.gpu, pytest.mark.fused_math]

BAGS = 12400          # past the line where this kernel starts


@pytest.fixture(scope="module", autouse=True)
def _device():
    capi.init(0)
    yield
    capi.sync()


def _run(kind, cols, mean, seed, bags=BAGS, half_w=False, idx32=False):
    print("lookup", kind, cols, bags, mean, flush=True)
    rng = np.random.default_rng(seed)
    rows = 300
    table = cases.random_fused_table(rng, rows, cols, kind)
    lengths, idx, w = cases.slws_batch(seed, rows, bags, mean, 1.05, np.int64)
    lengths[::7] = 0
    lengths[[1, 500, bags - 1]] = [1, 203, 65]       # more than one round; one past it
    total = int(lengths.sum())
    idx = np.resize(idx, total).astype(np.int32 if idx32 else np.int64)
    idx[::11] = [rows, -1][seed % 2]                 # skipped lookups
    w = np.resize(w, total).astype(np.float16 if half_w else np.float32)
    f16 = kind in (capi.FUSED_U8_F16, capi.FUSED_U4_F16)
    got = capi.frwq_slws(table, kind, w, idx, lengths, f16)
    # the same bags in launches below the line: bit for bit
    cut = bags // 2
    n = int(lengths[:cut].sum())
    parts = [capi.frwq_slws(table, kind, w[:n], idx[:n], lengths[:cut], f16),
             capi.frwq_slws(table, kind, w[n:], idx[n:], lengths[cut:], f16)]
    np.testing.assert_array_equal(got.view(np.uint8), np.concatenate(parts).view(np.uint8))
    ok = (idx >= 0) & (idx < rows)
    wz, iz = np.where(ok, w.astype(np.float32), 0).astype(np.float32), np.where(ok, idx, 0)
    want = go.frwq_slws_generic(table, kind, wz, iz.astype(np.int64), lengths, f16, False)
    check(got.astype(np.float32), want.astype(np.float32),
          bag_magnitude(table, kind, wz, iz, lengths), f16, what=f"{cols} columns")
    offsets = capi.frwq_slws(table, kind, w, idx, lengths, f16, bag_offsets=True)
    np.testing.assert_array_equal(offsets.view(np.uint8), got.view(np.uint8))


@pytest.mark.parametrize("cols", [68, 100, 124, 128, 132, 200, 252, 256])
@pytest.mark.parametrize("kind", [capi.FUSED_U8_F32, capi.FUSED_U8_F16])
def test_words(kind, cols):
    _run(kind, cols, 4, cols)


@pytest.mark.parametrize("cols", [136, 200, 256])
def test_four_bits(cols):
    _run(capi.FUSED_U4_F16, cols, 3, cols)
    _run(capi.FUSED_U4_F32, cols, 3, cols + 1)


# rows that start at any byte, in the arithmetic of the CPU loop
@pytest.mark.parametrize("kind,cols", [(capi.FUSED_U8_F32, 33), (capi.FUSED_U8_F32, 63),
                                       (capi.FUSED_U8_F16, 65), (capi.FUSED_U8_F32, 101),
                                       (capi.FUSED_U8_F16, 127), (capi.FUSED_U8_F32, 129),
                                       (capi.FUSED_U8_F32, 255), (capi.FUSED_U4_F16, 100),
                                       (capi.FUSED_U4_F32, 130), (capi.FUSED_U4_F32, 258)])
def test_any_byte(kind, cols):
    _run(kind, cols, 3, cols, idx32=True)
    _run(kind, cols, 3, cols + 1, half_w=True)


def test_lines_of_the_rule():
    for bags, mean, kind, cols in ((12288, 3, 0, 100), (12289, 3, 0, 100), (12300, 42, 0, 100),
                                   (12300, 38, 0, 100), (12300, 29, 0, 100),
                                   (12300, 23, 0, 128), (12300, 24, 0, 128), (12300, 3, 2, 256), (12300, 9, 3, 256), (24000, 17, 3, 100),
                                   (23999, 18, 3, 100)):
        _run(kind, cols, mean, bags, bags=bags)


# bags around the length from which one gets a wavefront of its own (32, or four times the
# average), many in one block and at the edges of a round, next to empty ones and the ends
@pytest.mark.parametrize("kind,cols", [(capi.FUSED_U8_F32, 68), (capi.FUSED_U8_F16, 128),
                                       (capi.FUSED_U8_F32, 132), (capi.FUSED_U8_F32, 256),
                                       (capi.FUSED_U8_F32, 33), (capi.FUSED_U8_F16, 54),
                                       (capi.FUSED_U8_F32, 101), (capi.FUSED_U8_F16, 255)])
@pytest.mark.parametrize("bags", [12400, 20010])
def test_long_bags(kind, cols, bags):
    print("long bags", kind, cols, bags, flush=True)
    rng = np.random.default_rng(cols)
    rows = 500
    table = cases.random_fused_table(rng, rows, cols, kind)
    lengths = rng.poisson(3, bags).astype(np.int32)
    lengths[:70] = np.arange(70)
    lengths[6000:6064] = 40
    lengths[[199, 201, 9000, bags - 1]] = [1030, 0, 64, 129]
    total = int(lengths.sum())
    idx = rng.integers(0, rows, total)
    idx[::13] = rows
    w = rng.random(total).astype(np.float32)
    f16 = kind == capi.FUSED_U8_F16
    got = capi.frwq_slws(table, kind, w, idx, lengths, f16)
    cut, n = bags // 2, int(lengths[:bags // 2].sum())
    parts = [capi.frwq_slws(table, kind, w[:n], idx[:n], lengths[:cut], f16),
             capi.frwq_slws(table, kind, w[n:], idx[n:], lengths[cut:], f16)]
    np.testing.assert_array_equal(got.view(np.uint8), np.concatenate(parts).view(np.uint8))
    offsets = capi.frwq_slws(table, kind, w, idx, lengths, f16, bag_offsets=True)
    np.testing.assert_array_equal(offsets.view(np.uint8), got.view(np.uint8))


@pytest.mark.parametrize("cols", [66, 101, 128, 256])
def test_separate_scales_and_offsets(cols):
    """Rows without a scale and offset behind them, which lie in arrays of their own."""
    bags, rows = 20010, 400
    print("separate scales", cols, flush=True)
    rng = np.random.default_rng(cols)
    data = rng.integers(0, 256, (rows, cols), dtype=np.uint8)
    scales = rng.uniform(0.001, 0.1, rows).astype(np.float32)
    offs = rng.normal(0, 1, rows).astype(np.float32)
    lengths = rng.poisson(3, bags).astype(np.int32)
    lengths[[5, 777, bags - 1]] = [90, 400, 33]
    total = int(lengths.sum())
    idx = rng.integers(0, rows, total).astype(np.int64)
    w = rng.random(total).astype(np.float32)
    got = capi.rwq_slws(data, scales, offs, w, idx, lengths)
    cut, n = bags // 2, int(lengths[:bags // 2].sum())
    parts = [capi.rwq_slws(data, scales, offs, w[:n], idx[:n], lengths[:cut]),
             capi.rwq_slws(data, scales, offs, w[n:], idx[n:], lengths[cut:])]
    np.testing.assert_array_equal(got, np.concatenate(parts))
    want = go.rwq_slws_f32(data, scales, offs, w, idx, lengths)
    # two roundings a term and one a sum, of 400 terms at most, on either side
    adds_up = go.rwq_slws_f32(data, scales, np.abs(offs), w, idx, lengths)
    assert np.all(np.abs(got - want) <= 2 * 403 * 2.0 ** -24 * adds_up)
    if cols % 4:
        np.testing.assert_array_equal(got, want)       # rows at any byte: the CPU loop's arithmetic
