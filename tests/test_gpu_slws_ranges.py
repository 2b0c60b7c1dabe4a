"""Pooled lookups of more bags than there are wavefronts, each wavefront taking bags in turns:
bag counts around the lines and blocks of that kernel, bag lengths around a round, empty and
long bags, against the oracle and, bit for bit, against launches with a bag per wavefront."""
import numpy as np
import pytest

from glow_amd import capi
from oracle import glow_oracle as go
from tests import cases
from tests.test_gpu_slws_fused import bag_magnitude, check

pytestmark = [pytest.mark.gpu, pytest.mark.fused_math]

HALF = (capi.FUSED_U8_F16, capi.FUSED_U4_F16)


@pytest.fixture(scope="module", autouse=True)
def _device():
    capi.init(0)
    yield
    capi.sync()


def _pieces(table, kind, w, idx, lengths, at_most=4000):
    """The same bags in launches below the line."""
    out, n = [], 0
    for lo in range(0, len(lengths), at_most):
        part = lengths[lo:lo + at_most]
        m = n + int(np.maximum(part, 0).sum())
        out.append(capi.frwq_slws(table, kind, None if w is None else w[n:m], idx[n:m], part, kind in HALF))
        n = m
    return np.concatenate(out)


def _run(kind, cols, bags, mean, seed, idx=np.int64, weights=np.float32):
    print("lookup", kind, cols, bags, mean, flush=True)
    rng = np.random.default_rng(seed)
    rows = 300
    table = cases.random_fused_table(rng, rows, cols, kind)
    lengths = rng.poisson(mean, bags).astype(np.int32)
    lengths[::9] = 0
    lengths[:4] = [0, 32, 33, 64]                     # rounds of 32 and 64 lookups
    lengths[[7, 8, 63, 64, bags - 2, bags - 1]] = [65, 0, 129, 31, 0, 1]
    total = int(lengths.sum())
    index = rng.integers(0, rows, total).astype(idx)
    index[::11] = [rows, -1][seed % 2]                # skipped lookups
    w = None if weights is None else rng.random(total).astype(weights)
    got = capi.frwq_slws(table, kind, w, index, lengths, kind in HALF)
    np.testing.assert_array_equal(got.view(np.uint8),
                                  _pieces(table, kind, w, index, lengths).view(np.uint8))
    ok = (index >= 0) & (index < rows)
    wz = np.where(ok, 1 if w is None else w.astype(np.float32), 0).astype(np.float32)
    iz = np.where(ok, index, 0).astype(np.int64)
    want = go.frwq_slws_generic(table, kind, wz, iz, lengths, kind in HALF, False)
    check(got.astype(np.float32), want.astype(np.float32), bag_magnitude(table, kind, wz, iz, lengths),
          kind in HALF, what=f"{cols} columns")
    offsets = capi.frwq_slws(table, kind, w, index, lengths, kind in HALF, bag_offsets=True)
    np.testing.assert_array_equal(offsets.view(np.uint8), got.view(np.uint8))


# the lines of the rule and the edges of its blocks
@pytest.mark.parametrize("bags", [4096, 4097, 4104, 6144, 6145, 8192, 8193, 16384, 16385, 20479])
@pytest.mark.parametrize("cols", [128, 256])
def test_lines(bags, cols):
    _run(capi.FUSED_U8_F32, cols, bags, 10, bags)


# rows around what 32 and 64 lanes hold
@pytest.mark.parametrize("kind,cols", [(capi.FUSED_U8_F32, 68), (capi.FUSED_U8_F16, 100),
                                       (capi.FUSED_U8_F16, 128), (capi.FUSED_U8_F32, 132),
                                       (capi.FUSED_U8_F16, 252), (capi.FUSED_U4_F16, 136),
                                       (capi.FUSED_U4_F32, 256), (capi.FUSED_U4_F16, 264),
                                       (capi.FUSED_U4_F32, 512)])
def test_widths(kind, cols):
    _run(kind, cols, 9001, 12, cols, idx=np.int32)
    _run(kind, cols, 4500, 40, cols + 1, weights=np.float16)
    _run(kind, cols, 8200, 5, cols + 3, weights=None)


# either side of the mean length from which bags keep a wavefront each (every ninth is empty)
@pytest.mark.parametrize("kind,cols,bags,means", [(capi.FUSED_U4_F32, 200, 4200, (68, 76)),
                                                  (capi.FUSED_U8_F32, 100, 8200, (120, 132))])
def test_long_means(kind, cols, bags, means):
    for mean in means:
        _run(kind, cols, bags, mean, mean)


def test_full_blocks_and_more_rounds():
    """More bags than resident blocks of 64 hold, and a last block of one bag."""
    _run(capi.FUSED_U8_F32, 72, 49152, 10, 3)
    _run(capi.FUSED_U8_F32, 72, 49153, 10, 4)
    _run(capi.FUSED_U4_F16, 136, 32769, 10, 5)


@pytest.mark.parametrize("cols", [128, 200])
def test_long_and_negative_bags(cols):
    """One very long bag, neighbours that are negative (empty), lengths past the list."""
    bags, rows = 5000, 200
    print("long bags", cols, flush=True)
    rng = np.random.default_rng(cols)
    table = cases.random_fused_table(rng, rows, cols, capi.FUSED_U8_F32)
    lengths = rng.poisson(4, bags).astype(np.int32)
    lengths[[3, 11, 4999]] = [3000, 700, 1500]
    lengths[[4, 12, 100]] = [-5, -1, -2 ** 31]
    idx = rng.integers(0, rows, int(np.maximum(lengths, 0).sum())).astype(np.int64)
    w = rng.random(len(idx)).astype(np.float32)
    got = capi.frwq_slws(table, capi.FUSED_U8_F32, w, idx, lengths)
    np.testing.assert_array_equal(got, _pieces(table, capi.FUSED_U8_F32, w, idx, lengths))
    # a list that ends early: the bags behind its end are short or empty
    cut = len(idx) // 2
    short = capi.frwq_slws(table, capi.FUSED_U8_F32, w[:cut], idx[:cut], lengths)
    ends = np.cumsum(np.maximum(lengths, 0))
    np.testing.assert_array_equal(short[ends <= cut], got[ends <= cut])
    assert not short[ends - np.maximum(lengths, 0) >= cut].any()
    # nothing to look up at all
    assert not capi.frwq_slws(table, capi.FUSED_U8_F32, w[:0], idx[:0], lengths).any()


def test_separate_scales_and_offsets():
    """Rows without a scale and offset behind them, which lie in arrays of their own."""
    bags, rows, cols = 9000, 400, 128
    print("separate scales", flush=True)
    rng = np.random.default_rng(7)
    data = rng.integers(0, 256, (rows, cols), dtype=np.uint8)
    scales = rng.uniform(0.001, 0.1, rows).astype(np.float32)
    offs = rng.normal(0, 1, rows).astype(np.float32)
    lengths = rng.poisson(12, bags).astype(np.int32)
    idx = rng.integers(0, rows, int(lengths.sum())).astype(np.int64)
    w = rng.random(len(idx)).astype(np.float32)
    got = capi.rwq_slws(data, scales, offs, w, idx, lengths)
    want, n = [], 0
    for lo in range(0, bags, 4000):
        m = n + int(lengths[lo:lo + 4000].sum())
        want.append(capi.rwq_slws(data, scales, offs, w[n:m], idx[n:m], lengths[lo:lo + 4000]))
        n = m
    np.testing.assert_array_equal(got, np.concatenate(want))


# the lengths in front of a block summed by itself: a trip of them, two, three; then by chunks
@pytest.mark.parametrize("bags", [16385, 16392, 32768, 32800, 40953, 40960, 40961])
@pytest.mark.parametrize("kind,cols", [(capi.FUSED_U8_F32, 72), (capi.FUSED_U4_F16, 264)])
def test_sums_over_many_bags(bags, kind, cols):
    _run(kind, cols, bags, 14, bags)


@pytest.mark.parametrize("first", [0, 1])
def test_long_lengths_in_front_of_many_bags(first):
    """Lengths that start on and off sixteen bytes; sums far past the list stop at its end."""
    bags, rows, cols = 40001, 500, 72
    print("lengths from", first, flush=True)
    rng = np.random.default_rng(first)
    table = cases.random_fused_table(rng, rows, cols, capi.FUSED_U8_F32)
    lengths = rng.poisson(24, bags).astype(np.int32)
    total = int(lengths.sum())
    idx = rng.integers(0, rows, total).astype(np.int64)
    w = rng.random(total).astype(np.float32)
    want = _pieces(table, capi.FUSED_U8_F32, w, idx, lengths)
    d_table, d_idx, d_w = (capi.to_device(v) for v in (table, idx, w))
    for end in (bags, 20000):
        some = lengths.copy()
        some[end:] = 2 ** 31 - 1
        d_len = capi.to_device(np.concatenate([np.full(first, 9, np.int32), some]))
        out = capi.to_device(np.full((bags, cols), 7, np.float32))
        n = int(lengths[:end].sum())
        capi.launch_frwq_slws(out.ptr, False, d_table.ptr, rows, capi.FUSED_U8_F32,
                              d_w.ptr, False, d_idx.ptr, True, n,
                              d_len.ptr + 4 * first, bags, table.shape[1], cols)
        got = out.numpy()
        np.testing.assert_array_equal(got[:end], want[:end])
        assert not got[end:].any()


# the lengths in front of a block by fours, wherever they start, in every kernel that sums them:
# few and many bags, several to a wavefront, in turns, behind sums of chunks
@pytest.mark.parametrize("cols,bags", [(128, 1001), (32, 3000), (128, 4096), (200, 4500), (72, 13001), (64, 17000),
                                       (200, 17001), (100, 41001)])
def test_lengths_that_start_anywhere(cols, bags):
    rows = 300
    print("lengths", cols, bags, flush=True)
    rng = np.random.default_rng(cols + bags)
    table = cases.random_fused_table(rng, rows, cols, capi.FUSED_U8_F32)
    lengths = rng.poisson(11, bags).astype(np.int32)
    lengths[::7] = [-3, 0][bags % 2]
    total = int(np.maximum(lengths, 0).sum())
    idx = rng.integers(0, rows, total).astype(np.int32)
    d_table, d_idx = capi.to_device(table), capi.to_device(idx)
    got = []
    for first in (0, 1, 2, 3):
        d_len = capi.to_device(np.concatenate([np.full(first, 9, np.int32), lengths, [9]]).astype(np.int32))
        out = capi.to_device(np.full((bags, cols), 7, np.float32))
        capi.launch_frwq_slws(out.ptr, False, d_table.ptr, rows, capi.FUSED_U8_F32, None, False, d_idx.ptr,
                              False, total, d_len.ptr + 4 * first, bags, table.shape[1], cols)
        got.append(out.numpy())
        np.testing.assert_array_equal(got[-1], got[0])
    ones, positive = np.ones(total, np.float32), np.maximum(lengths, 0)
    idx = idx.astype(np.int64)
    want = go.frwq_slws_generic(table, capi.FUSED_U8_F32, ones, idx, positive, False, False)
    check(got[0], want.astype(np.float32), bag_magnitude(table, capi.FUSED_U8_F32, ones, idx, positive), False,
          what=f"{cols} columns")


@pytest.mark.parametrize("first", [0, 3])
def test_positions_in_lists_past_32_bits(first):
    """An index list of more than 2^26 entries, whose positions are summed in 64 bits, bags in turns."""
    bags, rows, cols = 20001, 300, 200
    print("long list", first, flush=True)
    rng = np.random.default_rng(first)
    table = cases.random_fused_table(rng, rows, cols, capi.FUSED_U8_F32)
    lengths = rng.poisson(6, bags).astype(np.int32)
    total = int(lengths.sum())
    idx = np.zeros(2 ** 26 + 3, np.int32)
    idx[:total] = rng.integers(0, rows, total)
    d_table, d_idx = capi.to_device(table), capi.to_device(idx)
    d_len = capi.to_device(np.concatenate([np.full(first, 9, np.int32), lengths]).astype(np.int32))
    out = capi.to_device(np.full((bags, cols), 7, np.float32))
    capi.launch_frwq_slws(out.ptr, False, d_table.ptr, rows, capi.FUSED_U8_F32, None, False, d_idx.ptr,
                          False, len(idx), d_len.ptr + 4 * first, bags, table.shape[1], cols)
    np.testing.assert_array_equal(out.numpy(), _pieces(table, capi.FUSED_U8_F32, None, idx[:total], lengths))


# either side of where each kind of row is taken in turns, and blocks of four-bit rows, which are
# rounded to four bags: twelve and twenty of them, the last block with one bag
@pytest.mark.parametrize("kind,cols,bags", [
    (capi.FUSED_U8_F16, 128, (4111, 4112)), (capi.FUSED_U8_F32, 256, (4096, 4097, 4111, 4112)),
    (capi.FUSED_U8_F32, 100, (4159, 4160, 6144, 6145, 8223, 8224)),
    (capi.FUSED_U4_F32, 200, (4159, 4160, 6145, 8223, 8224, 8301)),
    (capi.FUSED_U4_F16, 200, (4159, 4160, 6144, 6145, 8223, 8224, 8245)),
    (capi.FUSED_U4_F16, 400, (4111, 4112, 4159, 4160, 5005, 6146))])
@pytest.mark.parametrize("mean", [6, 17])            # (every ninth is empty)
def test_lines_by_kind(kind, cols, bags, mean):
    for n in bags:
        _run(kind, cols, n, mean, n)


def _takes_turns(lengths, data_bytes):
    """Eight-bit rows of 65 to 128 bytes whose bags are too long for the kernel that works on several
    side by side (nine lookups or 900 bytes on the average), and not so long that each keeps a
    wavefront."""
    mean = int(lengths.sum()) // len(lengths)
    return mean < 112 and (mean > 9 or mean * data_bytes > 900)


# blocks of 64 bags, then two rounds of resident blocks (and sums of chunks in front of them), and last
# blocks of one bag: 1229 blocks of 40 and one, 911 of 36 and one of four-bit rows
@pytest.mark.parametrize("kind,cols,bags,per_block", [
    (capi.FUSED_U8_F32, 72, 49152, 64), (capi.FUSED_U8_F32, 72, 49153, 40), (capi.FUSED_U8_F32, 72, 49161, 40),
    (capi.FUSED_U8_F16, 200, 49152, 64), (capi.FUSED_U8_F32, 256, 49161, 40),
    (capi.FUSED_U4_F32, 136, 32768, 64), (capi.FUSED_U4_F32, 136, 32797, 36)])
def test_blocks_of_64_bags_and_more_rounds(kind, cols, bags, per_block):
    rng = np.random.default_rng(bags)                 # as _run draws them
    cases.random_fused_table(rng, 300, cols, kind)
    lengths = rng.poisson(14, bags).astype(np.int32)
    lengths[::9] = 0
    four = kind in (capi.FUSED_U4_F16, capi.FUSED_U4_F32)
    assert four or _takes_turns(lengths, cols)
    resident, whole = (512, 4) if four else (768, 8)
    rounds = -(-bags // (64 * resident))
    assert -(-(-(-bags // (resident * rounds))) // whole) * whole == per_block
    _run(kind, cols, bags, 14, bags)
