"""Chains of FullyConnected layers in one kernel (fc_chain.hip): the bytes of the layers one
by one, at the edges of its tiles (16 rows, 16 outputs, steps of 64 inputs, eight steps asked
for at once, sixteen waves); and which towers of a network the backend runs that way."""
import ctypes as C

import numpy as np
import pytest

from glow_amd import capi
from glow_amd import host as H
from glow_amd.harness import dlrm
from glow_amd.harness import net as netlib
from oracle import glow_oracle as go
from tests import cases


def _layers(seed, K, widths):
    """Layer parameters; every second layer has no Relu, every third an int8 bias."""
    out = []
    for i, n in enumerate(widths):
        c = cases.rwq_fc_case(seed + i, 1, K, n, bias_i8=i % 3 == 2, out_offset=(3 * i) % 11 - 5,
                              out_scale=0.1 * max(1.0, np.sqrt(K / 64)), bias_offset=i % 2)
        c["relu"] = None if i % 2 else (capi.quantize_scale_offset_32to8(0.9 + 0.3 * i)[:3], -100 + 7 * i)
        out.append(c)
        K = n
    return out


def _oracle(x, layers):
    for c in layers:
        a = cases.rwq_fc_args(c)
        x = go.rwq_fc_i8(x, *a[1:])
        if c["relu"]:
            x = go.relu_i8(x, c["out_offset"], c["relu"][1], c["relu"][0])
    return x


def _chain(layers, M, keep):
    ch = capi.FcChain()
    ch.n_layers, ch.M = len(layers), M
    for d, c in zip(ch.layers, layers):
        packed, cols = capi.fc_chain_pack(c["w"], c["bias"], c["bias_pre"], c["bias_post"], c["bias_scale"],
                                          c["out_pre"], c["out_post"], c["out_scale"], c["in_offset"],
                                          c["bias_offset"])
        keep += [capi.to_device(packed), capi.to_device(cols)]
        d.weights, d.columns = keep[-2].ptr, keep[-1].ptr
        d.N, d.K = c["w"].shape
        d.fc_offset = c["out_offset"]
        if c["relu"]:
            d.relu, d.relu_offset = 1, c["relu"][1]
            d.relu_pre, d.relu_post, d.relu_scale = c["relu"][0]
    return ch


@pytest.mark.gpu
@pytest.mark.parametrize("M", [1, 15, 16, 17, 259])
@pytest.mark.parametrize("K,widths", [
    (13, (512, 256, 64)), (415, (512, 256, 1)), (1, (1, 1)), (3, (5, 2)), (63, (16, 17)), (64, (15, 33)),
    (65, (1024, 7)), (1024, (257, 1000)), (577, (1024, 1024, 64, 3, 300, 31)), (512, (513, 513))])
def test_chain_equals_its_layers(M, K, widths):
    rng = np.random.default_rng(K + M)
    x = rng.integers(-128, 128, (M, K)).astype(np.int8)
    layers = _layers(K, K, widths)
    want = _oracle(x, layers)
    N = widths[-1]
    keep = []
    ch = _chain(layers, M, keep)
    # the result itself, between bytes that nobody may touch
    guard = np.full(M * N + 128, 77, np.int8)
    out = capi.to_device(guard)
    ch.out = out.ptr + 64
    # its rescale into rows of a wider tensor, at any byte
    pitch = N + 5
    wide = capi.to_device(np.full((M, pitch), 77, np.int8))
    p = capi.quantize_scale_offset_32to8(0.7)[:3]
    ch.n_slices = 2
    for s, off in zip(ch.slices, (0, 5)):
        s.dst_row_stride, s.out_offset, s.in_offset = pitch, 4 + off, -3
        s.pre, s.post, s.scale = p
    second = capi.to_device(np.full((M, pitch), 77, np.int8))
    ch.slices[0].dst, ch.slices[1].dst = wide.ptr + 3, second.ptr + 5
    prob = capi.DeviceBuffer.empty((M, N), np.float32)
    ch.sigmoid, ch.sigmoid_scale, ch.sigmoid_offset = prob.ptr, 0.03, 2
    # from a float input, quantized on the way, and from the same bytes
    xf = (x.astype(np.float32) + rng.uniform(-0.4, 0.4, x.shape).astype(np.float32)) * np.float32(0.25)
    xq = go.quantize_i8(xf, np.float32(0.25), 1)
    for floats in (False, True):
        d_in = capi.to_device(xf if floats else x)
        ch.inp, ch.in_f32 = (None, d_in.ptr) if floats else (d_in.ptr, None)
        ch.in_scale, ch.in_offset = 0.25, 1
        capi.launch_rwq_fc_chain_i8(ch)
        if floats:
            want = _oracle(xq, layers)
        got = out.numpy()
        np.testing.assert_array_equal(got[64:64 + M * N].reshape(M, N), want)
        assert np.all(got[:64] == 77) and np.all(got[64 + M * N:] == 77)
        for buf, at, off in ((wide, 3, 0), (second, 5, 5)):
            w = buf.numpy()
            np.testing.assert_array_equal(w[:, at:at + N], go.rescale_i8(want, 4 + off, -3, *p))
            assert np.all(w[:, :at] == 77) and np.all(w[:, at + N:] == 77)
        np.testing.assert_allclose(prob.numpy(), go.sigmoid_f32(go.dequantize_i8(want, np.float32(0.03), 2)),
                                   rtol=1e-5)


def _run_net(net, bindings, outputs, **opts):
    m, f = netlib.to_module(net)
    m.compile(f, **opts)
    dm = H.DeviceManager().init()
    try:
        dm.add_network(m)
        got = []
        for _ in range(14):           # past the comparison of recordings
            o = {k: np.zeros_like(v) for k, v in outputs.items()}
            dm.run("main", dict(bindings, **o))
            got.append(o)
        return got
    finally:
        dm.stop()


@pytest.mark.gpu
@pytest.mark.parametrize("batch,bottom,top", [(1, (32, 16), (32, 1)), (33, (512, 256, 64), (512, 256, 1)),
                                              (300, (64, 64), (70, 1))])
def test_ranking_net_with_and_without_chains(batch, bottom, top):
    net, max_idx = dlrm.make(seed=5, tables=3, rows=500, dim=bottom[-1], batch=batch, mean_len=4,
                             bottom=bottom, top=top)
    b = dlrm.bindings(net, dlrm.Inputs(9, 3, 500, batch, 4, 1.1, 13), max_idx)
    out = dict(logit_q=np.zeros((batch, 1), np.int8), prob=np.zeros((batch, 1), np.float32))
    a = _run_net(net, b, out)
    c = _run_net(net, b, out, fuse_fc_chains=False)
    for o in a + c:
        for k in out:
            np.testing.assert_array_equal(o[k], c[0][k])


def _listing(net, **opts):
    m, f = netlib.to_module(net)
    m.compile(f, **opts)
    return [r for r in H.parse_listing(m.describe(f)) if r["phase"] == "launch"]


def test_which_launches_a_chain_covers():
    net, _ = dlrm.make(seed=2, tables=3, rows=200, dim=16, batch=64, mean_len=5, bottom=(32, 16), top=(32, 1))
    rows = _listing(net)
    covered = {r["inst"]: r.get("covered_by") for r in rows}
    head = {r["inst"]: r.get("chain") for r in rows if "chain" in r}
    # the Quantize in front, both layers, both slices of their result; both layers, the sigmoid
    assert head == {"quantize_dense": 5, "top0": 3}
    assert [k for k, v in covered.items() if v == "quantize_dense"] == \
        ["bot0", "bot1", "bot_to_feat+insert_bot", "bot_to_top+insert_dense"]
    assert [k for k, v in covered.items() if v == "top0"] == ["top1", "dequantize+sigmoid"]
    rows = _listing(net, fuse_fc_chains=False)
    assert not any("chain" in r or "covered_by" in r for r in rows)


def _tower(extra=None, symmetric=True, last_width=8):
    """Two FullyConnected layers of 4 rows; `extra` adds instructions behind them."""
    rng = np.random.default_rng(1)
    net = netlib.Net("tower")
    net.placeholder("x", (4, 24), H.INT8Q, 0.05, 1)
    cur, k = "x", 24
    for i, n in enumerate((16, last_width)):
        net.constant(f"w{i}", rng.integers(-100, 100, (n, k)).astype(np.int8), H.INT8Q)
        net.constant(f"b{i}", rng.integers(-100, 100, n).astype(np.int32), H.INT32Q, 0.001, 0)
        net.constant(f"s{i}", np.full(n, 0.01, np.float32), H.FLOAT)
        net.constant(f"o{i}", np.full(n, 0 if symmetric else 3, np.int32), H.INT32I)
        dst = f"y{i}"
        (net.placeholder if i else net.activation)(dst, (4, n), H.INT8Q, 0.1, -1)
        net.op(H.ROWWISE_QUANTIZED_FC, f"fc{i}", [dst, cur, f"w{i}", f"b{i}", f"s{i}", f"o{i}"])
        cur, k = dst, n
    if extra:
        extra(net)
    return net


def _second_reader(net):
    net.placeholder("r", (4, 16), H.INT8Q, 0.2, 0)
    net.op(H.RESCALE_QUANTIZED, "again", ["r", "y0"])


def _through_a_view(net):
    net.view("v", "y0", (64,))
    net.placeholder("r", (64,), H.INT8Q, 0.2, 0)
    net.op(H.RESCALE_QUANTIZED, "again", ["r", "v"])


@pytest.mark.parametrize("extra,symmetric,width,chain", [
    (None, True, 8, True), (_second_reader, True, 8, False), (_through_a_view, True, 8, False),
    (None, False, 8, False), (None, True, 1025, False)])
def test_what_stays_a_launch_of_its_own(extra, symmetric, width, chain):
    rows = _listing(_tower(extra, symmetric, width))
    assert [r["inst"] for r in rows if "covered_by" in r] == (["fc1"] if chain else [])


def test_arguments_are_checked_before_the_device():
    ch = capi.FcChain()
    call = capi.lib().mi355x_rwq_fc_chain_i8
    ch.n_layers, ch.M = 1, 1
    assert call(C.byref(ch), None) == -1                                   # no input
    ch.inp = 4096
    for field, bad in (("K", 0), ("K", 1025), ("N", 0), ("N", 1025), ("weights", None), ("columns", 4100)):
        d = ch.layers[0]
        d.weights, d.columns, d.K, d.N = 4096, 4096, 8, 8
        setattr(d, field, bad)
        assert call(C.byref(ch), None) == -1, field
    ch.n_layers = 7
    assert call(C.byref(ch), None) == -1
    ch.n_layers, ch.M = 2, 0
    assert call(C.byref(ch), None) == 0                                    # nothing to do
    ch.struct_size -= 8
    assert call(C.byref(ch), None) == -1
    with pytest.raises(Exception):
        capi.fc_chain_pack(np.zeros((4, 1025), np.int8), np.zeros(4, np.int32), *[np.zeros(4, np.int32)] * 6, 0, 0)


def _nameless(net):
    for o in net.ops:
        o.name = ""
    return net


def test_launches_without_names_are_covered_too():
    """An instruction's name may be empty: what a chain covers does not hang on it."""
    rows = _listing(_nameless(_tower()))
    assert [r["chain"] for r in rows if "chain" in r] == [2]
    assert ["covered_by" in r for r in rows] == [False, True]
    net, _ = dlrm.make(seed=2, tables=3, rows=200, dim=16, batch=64, mean_len=5, bottom=(32, 16), top=(32, 1))
    named = _listing(net)
    rows = _listing(_nameless(net))
    assert [r.get("chain") for r in rows] == [r.get("chain") for r in named]
    assert ["covered_by" in r for r in rows] == ["covered_by" in r for r in named]


@pytest.mark.gpu
def test_nameless_net_with_and_without_chains():
    net, max_idx = dlrm.make(seed=6, tables=3, rows=500, dim=16, batch=33, mean_len=4, bottom=(32, 16),
                             top=(32, 1))
    b = dlrm.bindings(net, dlrm.Inputs(9, 3, 500, 33, 4, 1.1, 13), max_idx)
    out = dict(logit_q=np.zeros((33, 1), np.int8), prob=np.zeros((33, 1), np.float32))
    c = _run_net(net, b, out, fuse_fc_chains=False)
    for o in _run_net(_nameless(net), b, out):
        for k in out:
            np.testing.assert_array_equal(o[k], c[0][k])


def test_destinations_are_checked_before_the_device():
    """Rows of a slice that overlap each other, and destinations that touch the input of a chain of
    more than one workgroup, are refused."""
    call = capi.lib().mi355x_rwq_fc_chain_i8
    M, K, N, base = 40, 24, 8, 1 << 20

    def refused(m=M, stride=None, **dst):
        ch = capi.FcChain()
        ch.n_layers, ch.M, ch.inp = 1, m, base
        d = ch.layers[0]
        d.weights, d.columns, d.K, d.N = 4096, 4096, K, N
        if dst.pop("floats", False):
            ch.inp, ch.in_f32 = None, base
        if stride is not None:
            ch.n_slices = 1
            ch.slices[0].dst, ch.slices[0].dst_row_stride = dst.pop("at"), stride
        for k, v in dst.items():
            setattr(ch, k, v)
        rc = call(C.byref(ch), None)
        return rc == -1 and ("overlap" in capi.lib().mi355x_last_error().decode())

    size = M * K
    assert refused(stride=N - 1, at=1 << 24) and refused(m=1, stride=0, at=1 << 24)
    for first in (base, base + 1, base + size - 1, base - M * N + 1, base - 1):
        assert refused(out=first), first
    for first in (base + size - 1, base - 4 * M * N + 1):
        assert refused(sigmoid=first), first
    assert refused(floats=True, out=base + 4 * size - 1)
    # rows 64 apart that reach into the input from below, and that start in it
    for first in (base - 39 * 64 - N + 1, base - 7, base + size - 1, base - 128 + 63):
        assert refused(stride=64, at=first), first


def _overlap_oracle(first, pitch, rows, n, at, size):
    return any(first + r * pitch < at + size and first + r * pitch + n > at for r in range(rows))


@pytest.mark.gpu
def test_destinations_next_to_the_input():
    """Every place of a strided destination around the input, against the check row by row; those that
    do not touch it run and leave it alone."""
    M, K, widths = 20, 3, (5, 2)
    layers = _layers(3, K, widths)
    rng = np.random.default_rng(0)
    x = rng.integers(-128, 128, (M, K)).astype(np.int8)
    want = _oracle(x, layers)
    p = capi.quantize_scale_offset_32to8(0.7)[:3]
    keep, pitch, n = [], 70, widths[-1]
    ch = _chain(layers, M, keep)
    ch.n_slices = 1
    s = ch.slices[0]
    s.dst_row_stride, s.out_offset, s.in_offset = pitch, 4, -3
    s.pre, s.post, s.scale = p
    room, at = 2 * M * pitch + 200, M * pitch + 64
    ran = 0
    for first in range(at - M * pitch - 3, at + M * K + 3):
        host = np.full(room, 77, np.int8)
        host[at:at + M * K] = x.reshape(-1)
        touches = _overlap_oracle(first, pitch, M, n, at, M * K)
        buf = capi.to_device(host)
        ch.inp, s.dst = buf.ptr + at, buf.ptr + first
        if touches:
            with pytest.raises(capi.MI355XError):
                capi.launch_rwq_fc_chain_i8(ch)
            continue
        capi.launch_rwq_fc_chain_i8(ch)
        got = buf.numpy()
        for r in range(M):
            host[first + r * pitch:first + r * pitch + n] = go.rescale_i8(want, 4, -3, *p)[r]
        np.testing.assert_array_equal(got, host)
        ran += 1
    assert ran >= 9 * M                # of each pitch, what is left beside the input


@pytest.mark.gpu
def test_one_workgroup_may_write_over_its_input():
    """Sixteen rows are read before any is stored: accepted, as one layer after the other is."""
    layers = _layers(5, 24, (40, 8))
    x = np.random.default_rng(5).integers(-128, 128, (16, 24)).astype(np.int8)
    keep = []
    ch = _chain(layers, 16, keep)
    buf = capi.to_device(x)
    ch.inp, ch.out = buf.ptr, buf.ptr + 3
    capi.launch_rwq_fc_chain_i8(ch)
    got = buf.numpy().reshape(-1)
    np.testing.assert_array_equal(got[3:3 + 16 * 8].reshape(16, 8), _oracle(x, layers))
    np.testing.assert_array_equal(got[3 + 16 * 8:], x.reshape(-1)[3 + 16 * 8:])


def test_issued_launches_of_a_listing():
    net, _ = dlrm.make(seed=2, tables=3, rows=200, dim=16, batch=64, mean_len=5, bottom=(32, 16), top=(32, 1))
    m, f = netlib.to_module(net)
    m.compile(f)
    rows = [r for r in H.parse_listing(m.describe(f)) if r["phase"] == "launch"]
    # the two chains (of five and three launches), the lookups and the interaction
    assert H.issued_launches(m.describe(f)) == len(rows) - (5 - 1) - (3 - 1)
    m, f = netlib.to_module(_nameless(net))
    m.compile(f)
    assert H.issued_launches(m.describe(f)) == len(rows) - 6


def _plain_tower(rows, K, widths):
    rng = np.random.default_rng(2)
    net = netlib.Net("plain")
    net.placeholder("x", (rows, K), H.INT8Q, 0.05, 1)
    cur, k = "x", K
    for i, n in enumerate(widths):
        net.constant(f"w{i}", rng.integers(-100, 100, (n, k)).astype(np.int8), H.INT8Q)
        net.constant(f"b{i}", rng.integers(-100, 100, n).astype(np.int32), H.INT32Q, 0.001, 0)
        net.constant(f"s{i}", np.full(n, 0.01, np.float32), H.FLOAT)
        net.constant(f"o{i}", np.zeros(n, np.int32), H.INT32I)
        (net.activation if i + 1 < len(widths) else net.placeholder)(f"y{i}", (rows, n), H.INT8Q, 0.1, -1)
        net.op(H.ROWWISE_QUANTIZED_FC, f"fc{i}", [f"y{i}", cur, f"w{i}", f"b{i}", f"s{i}", f"o{i}"])
        cur, k = f"y{i}", n
    return net


# a result too wide for the launches saved, with one round of rows on a unit and with two
@pytest.mark.parametrize("rows,widths,chain", [
    (4, (16, 768), True), (4, (16, 769), False), (4096, (16, 768), True), (4097, (16, 400), True),
    (4097, (16, 401), False), (4097, (16, 16, 800), True), (4097, (16, 16, 801), False), (8193, (16, 16), False)])
def test_towers_with_wide_results(rows, widths, chain):
    listed = _listing(_plain_tower(rows, 24, widths))
    assert [r["inst"] for r in listed if "covered_by" in r] == \
        ([f"fc{i}" for i in range(1, len(widths))] if chain else [])
