"""Transfers of a request: mi355x_copy_segments at the edges of its workgroups, and
a device manager's inputs and outputs at the edges of the pieces they are staged
in (128 KiB), whatever memory the caller's arrays lie in."""
import ctypes as C

import numpy as np
import pytest

from glow_amd import capi
from glow_amd import host as H
from oracle import glow_oracle as go
from tests import cases

pytestmark = pytest.mark.gpu


class Segment(C.Structure):
    _fields_ = [("dst", C.c_void_p), ("src", C.c_void_p), ("bytes", C.c_uint64),
                ("positions", C.c_void_p), ("bags", C.c_uint32), ("op", C.c_int32)]


@pytest.fixture(scope="module", autouse=True)
def _device():
    capi.init(0)
    yield
    capi.sync()


def _send(segs):
    arr = (Segment * len(segs))(*segs)
    done = capi.pinned_empty((1,), np.uint32)
    done[0] = 0
    arrived = capi.to_device(np.zeros(1, np.uint32))
    capi.sync()
    capi.check(capi.lib().mi355x_copy_segments(arr, C.c_size_t(len(segs)), capi._vp(done),
                                               C.c_uint32(7), capi._vp(arrived), None))
    capi.sync()
    assert done[0] == 7 and arrived.numpy().view(np.uint32)[0] == 0


@pytest.mark.parametrize("shift", [0, 1])
def test_copies_of_every_size_in_one_call(shift):
    rng = np.random.default_rng(5)
    sizes = [1, 15, 16, 17, 4095, 16383, 16384, 16385, 40000] + [64] * 60   # over one launch's worth
    src = [capi.pinned_copy(rng.integers(0, 256, n + shift, dtype=np.uint8)) for n in sizes]
    dst = [capi.to_device(np.full(n + 2, 0xEE, np.uint8)) for n in sizes]
    print("copies", len(sizes), shift, flush=True)
    _send([Segment(d.ptr, s.ctypes.data + shift, n, None, 0, 0) for d, s, n in zip(dst, src, sizes)])
    for d, s, n in zip(dst, src, sizes):
        got = d.numpy()
        assert np.array_equal(got[:n], s[shift:shift + n]) and np.all(got[n:] == 0xEE), n


@pytest.mark.parametrize("n", [1, 3, 4, 5, 4095, 4096, 4097, 20001])
def test_indices_travel_as_32_bits(n):
    v = np.random.default_rng(n).integers(-2 ** 31, 2 ** 31, n).astype(np.int32)
    src, dst = capi.pinned_copy(v), capi.to_device(np.full(n + 1, -9, np.int64))
    print("widen", n, flush=True)
    _send([Segment(dst.ptr, src.ctypes.data, 4 * n, None, 0, 1)])
    assert np.array_equal(dst.numpy(), np.r_[v.astype(np.int64), -9])


@pytest.mark.parametrize("n", [1, 7, 8, 9, 8191, 8192, 8193, 40001])
@pytest.mark.parametrize("bits", [16, 24])
def test_indices_travel_as_two_or_three_bytes(n, bits):
    v = np.random.default_rng(n).integers(0, 2 ** bits, n)
    v[-1] = 2 ** bits - 1
    room = (2 * n + 15) // 16 * 16
    wire = np.zeros(room + n, np.uint8)
    wire[:2 * n] = (v & 0xffff).astype(np.uint16).view(np.uint8)
    wire[room:] = v >> 16
    src, dst = capi.pinned_copy(wire), capi.to_device(np.full(n + 1, -9, np.int64))
    print("widen", n, bits, flush=True)
    _send([Segment(dst.ptr, src.ctypes.data, 2 * n, None, 0, 3 if bits == 16 else 4)])
    assert np.array_equal(dst.numpy(), np.r_[v, -9])


@pytest.mark.parametrize("n", [1, 2, 7, 8, 31, 33, 8190, 8191, 8192, 8193, 16385, 40001])
def test_indices_travel_as_two_and_a_half_bytes(n):
    v = np.random.default_rng(n).integers(0, 2 ** 20, n)
    v[-1] = 2 ** 20 - 1
    room = (2 * n + 15) // 16 * 16
    high = np.r_[v >> 16, 0][:(n + 1) // 2 * 2]
    wire = np.zeros(room + len(high) // 2, np.uint8)
    wire[:2 * n] = (v & 0xffff).astype(np.uint16).view(np.uint8)
    wire[room:] = high[::2] | high[1::2] << 4
    src, dst = capi.pinned_copy(wire), capi.to_device(np.full(n + 1, -9, np.int64))
    print("widen", n, 20, flush=True)
    _send([Segment(dst.ptr, src.ctypes.data, 2 * n, None, 0, 5)])
    assert np.array_equal(dst.numpy(), np.r_[v, -9])


@pytest.mark.parametrize("given,bags", [(0, 5), (1, 1), (15, 16), (17, 17), (4096, 4096), (4097, 4100),
                                        (9000, 9001)])
def test_bag_positions_from_lengths_of_a_byte(given, bags):
    v = np.random.default_rng(bags).integers(0, 256, given).astype(np.int32)
    full = np.r_[v, np.zeros(bags - given, np.int32)]
    src = capi.pinned_copy(np.r_[v, 0].astype(np.uint8))
    dst = capi.to_device(np.full(bags, 77, np.int32))
    pos = capi.to_device(np.full(bags + 1, 77, np.int32))
    print("positions", given, bags, "bytes", flush=True)
    _send([Segment(dst.ptr, src.ctypes.data, given, pos.ptr, bags, 6)])
    assert np.array_equal(dst.numpy(), full)
    assert np.array_equal(pos.numpy(), np.r_[0, np.cumsum(full)].astype(np.int32))


@pytest.mark.parametrize("given,bags", [(0, 5), (1, 1), (15, 16), (17, 17), (4096, 4096), (4097, 4100),
                                        (9000, 9001)])
@pytest.mark.parametrize("huge", [False, True])
def test_bag_positions(given, bags, huge):
    rng = np.random.default_rng(bags)
    v = rng.integers(-2, 9, given).astype(np.int32)
    if huge and given:
        v[given // 2:] = 2 ** 31 - 1
    full = np.r_[v, np.zeros(bags - given, np.int32)]
    want = np.minimum(np.r_[0, np.cumsum(np.maximum(full, 0).astype(np.int64))], 2 ** 31 - 1)
    src = capi.pinned_copy(np.r_[v, 0].astype(np.int32))
    dst = capi.to_device(np.full(bags, 77, np.int32))
    pos = capi.to_device(np.full(bags + 1, 77, np.int32))
    print("positions", given, bags, huge, flush=True)
    _send([Segment(dst.ptr, src.ctypes.data, 4 * given, pos.ptr, bags, 2)])
    assert np.array_equal(dst.numpy(), full)
    assert np.array_equal(pos.numpy(), want.astype(np.int32))


def _manager(build):
    m = H.Module("transfers")
    f = m.function("main")
    build(m, f)
    m.compile(f)
    dm = H.DeviceManager().init()
    dm.add_network(m)
    return dm


@pytest.mark.parametrize("n", [1, 32767, 32768, 32769, 262144, 300001])
@pytest.mark.parametrize("pinned", [False, True])
def test_request_copies(n, pinned):
    """A float tensor through a request, from aligned, shifted and pinned arrays."""
    def build(m, f):
        a = m.placeholder("in", (n,), H.FLOAT, np.float32)
        b = m.placeholder("out", (n,), H.FLOAT, np.float32)
        m.instruction(f, H.COPY, "copy", [b, a])
    dm = _manager(build)
    rng = np.random.default_rng(n)
    try:
        for shift in (0, 1):
            x = rng.normal(size=n + shift).astype(np.float32)
            x = (capi.pinned_copy(x) if pinned else x)[shift:]
            out = np.zeros(n + shift, np.float32)[shift:]
            print("request", n, pinned, shift, flush=True)
            dm.run("main", {"in": x, "out": out})
            assert np.array_equal(x, out)
    finally:
        dm.stop()


@pytest.mark.parametrize("wide", [False, True])
def test_request_with_indices_past_32_bits(wide):
    """int64 indices that do not fit 32 bits are out of range, not truncated."""
    rows, cols, bags, n = 500, 16, 40, 40000
    rng = np.random.default_rng(4)
    table = cases.random_fused_table(rng, rows, cols)

    def build(m, f):
        t = m.constant("table", table, H.UINT8_FUSED)
        i = m.placeholder("idx", (n,), H.INT64I, np.int64)
        ln = m.placeholder("len", (bags,), H.INT32I, np.int32)
        o = m.placeholder("out", (bags, cols), H.FLOAT, np.float32)
        m.instruction(f, H.FRWQ_SLS, "sls", [o, t, i, ln], [0])
    dm = _manager(build)
    lengths = np.full(bags, n // bags, np.int32)
    idx = rng.integers(0, rows, n).astype(np.int64)
    keep = np.ones(n, bool)
    if wide:
        keep[::777] = False
        idx[~keep] += 1 << 32
    out = np.zeros((bags, cols), np.float32)
    try:
        dm.run("main", {"idx": idx, "len": lengths, "out": out})
    finally:
        dm.stop()
    w = keep.astype(np.float32)
    want = go.frwq_slws_f32(table, w, np.where(keep, idx, 0), lengths)
    np.testing.assert_allclose(out, want, rtol=1e-5, atol=1e-3)


@pytest.mark.parametrize("top", [0xffff, 0x10000, 0xffffff, 0x1000000, -1])
@pytest.mark.parametrize("n", [15, 16, 16384, 40001])
def test_request_with_indices_of_every_width(top, n):
    """The largest index decides how many bytes each travels as; those past the
    table count as out of range whatever they travelled as."""
    rows, cols, bags = 70000, 16, 5
    rng = np.random.default_rng(n)
    table = cases.random_fused_table(rng, rows, cols)

    def build(m, f):
        t = m.constant("table", table, H.UINT8_FUSED)
        i = m.placeholder("idx", (n,), H.INT64I, np.int64)
        ln = m.placeholder("len", (bags,), H.INT32I, np.int32)
        o = m.placeholder("out", (bags, cols), H.FLOAT, np.float32)
        m.instruction(f, H.FRWQ_SLS, "sls", [o, t, i, ln], [0])
    dm = _manager(build)
    lengths = np.full(bags, n // bags, np.int32)
    idx = rng.integers(0, min(rows, max(1, top + 1)), n).astype(np.int64)
    idx[n // 2] = top
    out = np.zeros((bags, cols), np.float32)
    print("request", n, top, flush=True)
    try:
        dm.run("main", {"idx": idx, "len": lengths, "out": out})
    finally:
        dm.stop()
    ok = (idx >= 0) & (idx < rows)
    want = go.frwq_slws_f32(table, ok.astype(np.float32), np.where(ok, idx, 0), lengths)
    np.testing.assert_allclose(out, want, rtol=1e-5, atol=2e-3)


@pytest.mark.parametrize("top", [0xfffff, 0x100000])
@pytest.mark.parametrize("n", [17, 31, 16384 + 33])
@pytest.mark.parametrize("longest", [255, 256, -1])
def test_request_with_indices_and_lengths_at_the_edges_of_their_forms(top, n, longest):
    """Indices in half bytes up to 2^20 - 1 and lengths in a byte up to 255, past those
    the next form; a negative length is an empty bag."""
    rows, cols, bags = 70000, 16, 300
    rng = np.random.default_rng(n)
    table = cases.random_fused_table(rng, rows, cols)

    def build(m, f):
        t = m.constant("table", table, H.UINT8_FUSED)
        i = m.placeholder("idx", (n,), H.INT64I, np.int64)
        ln = m.placeholder("len", (bags,), H.INT32I, np.int32)
        o = m.placeholder("out", (bags, cols), H.FLOAT, np.float32)
        m.instruction(f, H.FRWQ_SLS, "sls", [o, t, i, ln], [0])
    dm = _manager(build)
    lengths = np.zeros(bags, np.int32)
    lengths[[3, 41, 299]] = [min(n // 2, 200), longest, 1]
    idx = rng.integers(0, rows, n).astype(np.int64)
    idx[[0, n - 1]] = [top, 65536]
    out = np.zeros((bags, cols), np.float32)
    print("request", n, top, longest, flush=True)
    try:
        dm.run("main", {"idx": idx, "len": lengths, "out": out})
    finally:
        dm.stop()
    ok = (idx >= 0) & (idx < rows)
    ends = np.minimum(np.cumsum(np.maximum(lengths, 0)), n)
    ref = np.diff(np.r_[0, ends]).astype(np.int32)
    want = go.frwq_slws_f32(table, ok.astype(np.float32), np.where(ok, idx, 0), ref)
    np.testing.assert_allclose(out, want, rtol=1e-5, atol=2e-3)


@pytest.mark.parametrize("n", [1, 5])
def test_float_images_quantized_on_the_way(n):
    """A stem's float input, which the device manager quantizes while it stages it:
    values on the rounding ties, past int8 and int32, infinite and not a number give
    the bytes the Quantize kernel gives, through a request, a partial request and a
    static placeholder."""
    size, scale, offset = 96, 0.05, 3
    rng = np.random.default_rng(n)
    filt = rng.integers(-127, 128, (16, 3, 3, 3)).astype(np.int8)
    m = H.Module("stem")
    x = m.placeholder("x", (n, size, size, 3), H.FLOAT, np.float32)
    out = m.placeholder("out", (n, size // 2, size // 2, 16), H.INT8Q, np.int8, 2.0, -3)
    ops = [m.constant("f", filt, H.INT8Q), m.constant("b", np.zeros(16, np.int32), H.INT32Q),
           m.constant("fs", np.full(16, 0.01, np.float32), H.FLOAT),
           m.constant("fo", np.zeros(16, np.int32), H.INT32I),
           m.constant("bs", np.full(16, 0.01 * scale, np.float32), H.FLOAT),
           m.constant("bo", np.zeros(16, np.int32), H.INT32I)]
    f = m.function("main")
    q = m.activation(f, "q", (n, size, size, 3), H.INT8Q, scale, offset)
    m.instruction(f, H.QUANTIZE, "quantize", [q, x])
    m.instruction(f, H.CHANNELWISE_QUANTIZED_CONV, "stem", [out, q, *ops],
                  H.conv_attrs((3, 3), (2, 2), (1, 1, 1, 1)))
    m.compile(f)
    v = (rng.integers(-3000, 3000, (n, size, size, 3)) * (scale / 8)).astype(np.float32)
    v.reshape(-1)[:7] = [np.inf, -np.inf, np.nan, 1e30, -1e30, 3e9, -0.0]

    def want(vals):
        return capi.conv2d_i8(capi.quantize_i8(vals, scale, offset), filt, np.zeros(16, np.int32),
                              geom, -3, offset, 0, 0, (0, 0, 1),
                              capi.quantize_scale_offset_32to8(scale * 0.01 / 2.0, 0)[:3])
    from glow_amd import workloads
    geom = workloads.default_host().conv_geom(n, size, size, 3, 16, (3, 3), (2, 2), (1, 1, 1, 1))
    dm = H.DeviceManager().init()
    try:
        dm.add_network(m)
        got = np.zeros((n, size // 2, size // 2, 16), np.int8)
        print("stem", n, flush=True)
        dm.run("main", {"x": v, "out": got})
        assert np.array_equal(got, want(v))
        w = v.copy()
        w.reshape(-1)[:5001] += 4 * scale          # a shorter tensor replaces the front
        dm.run("main", {"x": np.ascontiguousarray(w.reshape(-1)[:5001]), "out": got})
        assert np.array_equal(got, want(w))
        dm.transfer_static_placeholder(m, "x", v)
        dm.run("main", {"out": got})
        assert np.array_equal(got, want(v))
    finally:
        dm.stop()


@pytest.mark.parametrize("n", [1, 64])
@pytest.mark.parametrize("pinned", [False, True])
def test_float_values_follow_an_image_that_travels_quantized(n, pinned):
    """The slot of an image that the launches take quantized holds its float values
    when the request is over: from a function loaded only then, piece by piece and by
    one copy out of pinned memory, while recordings are compared and afterwards."""
    size = 96
    m = H.Module("late")
    x = m.placeholder("x", (n, size, size, 3), H.FLOAT, np.float32)
    out = m.placeholder("out", (n, size // 2, size // 2, 16), H.INT8Q, np.int8, 2.0, -3)
    ops = [m.constant("f", np.ones((16, 3, 3, 3), np.int8), H.INT8Q),
           m.constant("b", np.zeros(16, np.int32), H.INT32Q),
           m.constant("fs", np.full(16, 0.01, np.float32), H.FLOAT),
           m.constant("fo", np.zeros(16, np.int32), H.INT32I),
           m.constant("bs", np.full(16, 0.0005, np.float32), H.FLOAT),
           m.constant("bo", np.zeros(16, np.int32), H.INT32I)]
    f = m.function("reader")
    q = m.activation(f, "q", (n, size, size, 3), H.INT8Q, 0.05, 3)
    m.instruction(f, H.QUANTIZE, "quantize", [q, x])
    m.instruction(f, H.CHANNELWISE_QUANTIZED_CONV, "stem", [out, q, *ops],
                  H.conv_attrs((3, 3), (2, 2), (1, 1, 1, 1)))
    m.compile(f)
    g = m.function("copy")
    m.instruction(g, H.COPY, "copy", [m.placeholder("y", (n, size, size, 3), H.FLOAT, np.float32), x])
    m.compile(g)
    rng = np.random.default_rng(n)
    got = np.zeros((n, size // 2, size // 2, 16), np.int8)
    y = np.zeros((n, size, size, 3), np.float32)
    dm = H.DeviceManager().init()
    try:
        dm.add_network(m, [f])
        for requests in (1, 14):
            for _ in range(requests):
                v = rng.normal(size=y.shape).astype(np.float32)
                v = capi.pinned_copy(v) if pinned else v
                print("image", n, pinned, flush=True)
                dm.run("reader", {"x": v, "out": got})
            dm.add_network(m, [g])
            dm.run("copy", {"y": y})
            assert np.array_equal(y, v)
            dm.evict_network("copy")
    finally:
        dm.stop()


def test_bag_positions_follow_lengths_that_came_through_a_view():
    rows, cols, bags, n = 500, 16, 40, 400
    rng = np.random.default_rng(6)
    table = cases.random_fused_table(rng, rows, cols)
    m = H.Module("views")
    t = m.constant("table", table, H.UINT8_FUSED)
    i = m.placeholder("idx", (n,), H.INT64I, np.int64)
    ln = m.placeholder("len", (bags,), H.INT32I, np.int32)
    front = m.view("front", ln, (10,), H.INT32I)
    o = m.placeholder("out", (bags, cols), H.FLOAT, np.float32)
    f = m.function("main")
    m.instruction(f, H.FRWQ_SLS, "sls", [o, t, i, ln], [0])
    m.compile(f)
    g = m.function("second")
    m.instruction(g, H.COPY, "copy", [m.placeholder("copy", (10,), H.INT32I, np.int32), front])
    m.compile(g)
    idx = rng.integers(0, rows, n).astype(np.int64)
    lengths = rng.integers(0, 8, bags).astype(np.int32)
    out, copy = np.zeros((bags, cols), np.float32), np.zeros(10, np.int32)
    w = np.ones(n, np.float32)
    print("lengths through a view", flush=True)
    dm = H.DeviceManager().init()
    try:
        dm.add_network(m)
        dm.run("main", {"idx": idx, "len": lengths, "out": out})
        for how in ("request", "static"):
            lengths[:10] = rng.integers(0, 8, 10)
            if how == "request":
                dm.run("second", {"front": lengths[:10].copy(), "copy": copy})
                assert np.array_equal(copy, lengths[:10])
            else:
                dm.transfer_static_placeholder(m, "front", lengths[:10].copy())
            dm.run("main", {"out": out})
            np.testing.assert_allclose(out, go.frwq_slws_f32(table, w, idx, lengths), rtol=1e-5, atol=1e-4)
    finally:
        dm.stop()
