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
