"""Requests of a device manager on a device made of host memory (fake_device.cpp; no
GPU needed): what the launches of an image stem read, whoever else is loaded. Every
scenario runs in a process of its own, where the host library binds to that device."""
import ctypes as C
import os
import subprocess
import sys

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SCALE, OFFSET = 0.05, 3


@pytest.fixture(scope="module")
def fake_device(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("fake") / "libfake_device.so")
    subprocess.check_call(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-I",
                           os.path.join(ROOT, "include"),
                           os.path.join(ROOT, "tests", "fake_device.cpp"), "-o", so])
    return so


def _in_child(fake_device, scenario, *args):
    r = subprocess.run([sys.executable, "-c",
                        f"from tests import test_host_requests as t; t.bind({fake_device!r}); "
                        f"t.{scenario}(*{args!r})"], cwd=ROOT, capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, r.stderr[-3000:]


def bind(so):
    global FAKE
    FAKE = C.CDLL(so, C.RTLD_GLOBAL)
    FAKE.fake_graph_launches.restype = C.c_long


# ---- in the child ------------------------------------------------------------------

def _image_module(size=16):
    """out = the convolution of quantize(x); the fake kernels hand quantize(x) through."""
    from glow_amd import host as H
    m = H.Module("images")
    x = m.placeholder("x", (1, size, size, 3), H.FLOAT, np.float32)
    f = m.function("reader")
    out = m.placeholder("out", (1, size // 2, size // 2, 16), H.INT8Q, np.int8, 2.0, -3)
    ops = [m.constant("f", np.ones((16, 3, 3, 3), np.int8), H.INT8Q),
           m.constant("b", np.zeros(16, np.int32), H.INT32Q),
           m.constant("fs", np.full(16, 0.01, np.float32), H.FLOAT),
           m.constant("fo", np.zeros(16, np.int32), H.INT32I),
           m.constant("bs", np.full(16, 0.01 * SCALE, np.float32), H.FLOAT),
           m.constant("bo", np.zeros(16, np.int32), H.INT32I)]
    q = m.activation(f, "q", (1, size, size, 3), H.INT8Q, SCALE, OFFSET)
    m.instruction(f, H.QUANTIZE, "quantize", [q, x])
    m.instruction(f, H.CHANNELWISE_QUANTIZED_CONV, "stem", [out, q, *ops],
                  H.conv_attrs((3, 3), (2, 2), (1, 1, 1, 1)))
    return m, f, x


def _image(seed, size=16):
    return np.random.default_rng(seed).normal(0, 2, (1, size, size, 3)).astype(np.float32)


def _codes(x):
    return np.clip(np.rint(x / np.float32(SCALE) + np.float32(OFFSET)), -128, 127).astype(np.int8).reshape(-1)


def _run(dm, x=None, size=16):
    out = np.zeros((1, size // 2, size // 2, 16), np.int8)
    dm.run("reader", {"out": out} if x is None else {"x": x, "out": out})
    return out.reshape(-1)[:3 * size * size]


def one_function_on_two_managers():
    from glow_amd import host as H
    m, f, _ = _image_module()
    m.compile(f)
    for graphs in (False, True):
        first = H.DeviceManager(use_launch_graphs=graphs).init()
        second = H.DeviceManager(use_launch_graphs=graphs).init()
        first.add_network(m)
        second.add_network(m)
        images = [_image(i) for i in range(4)]
        for i in range(12):            # past the comparison of recordings
            a, b = images[i % 4], images[(i + 1) % 4]
            assert np.array_equal(_run(second, b), _codes(b)), (graphs, i)
            assert np.array_equal(_run(first, a), _codes(a)), (graphs, i)
            assert np.array_equal(_run(second), _codes(b)), (graphs, i)
        second.stop()
        for a in images:
            assert np.array_equal(_run(first, a), _codes(a)), graphs
        first.stop()


def function_loaded_behind_a_request(size):
    from glow_amd import host as H
    m, f, x = _image_module(size)
    m.compile(f)
    g = m.function("second")
    m.instruction(g, H.COPY, "copy", [m.placeholder("y", (1, size, size, 3), H.FLOAT, np.float32), x])
    m.compile(g)
    dm = H.DeviceManager(use_launch_graphs=size < 1000).init()   # (the large one untuned)
    dm.add_network(m, [f])
    a, y = _image(1, size), np.zeros((1, size, size, 3), np.float32)
    assert np.array_equal(_run(dm, a, size), _codes(a))
    dm.add_network(m, [g])
    dm.run("second", {"y": y})           # on the image of the request before
    assert np.array_equal(y, a)
    # a tensor that ends inside a value: the rest of the value is the old one's
    dm.evict_network("second")
    _run(dm, a, size)
    cut = _image(2, size).reshape(-1).view(np.uint8)[:10]
    a.reshape(-1).view(np.uint8)[:10] = cut
    assert np.array_equal(_run(dm, cut.copy(), size), _codes(a))
    dm.stop()


def writer_of_the_image(writer_first, requests):
    from glow_amd import host as H
    m, f, x = _image_module()
    m.compile(f)
    w = m.function("writer")             # the reader was compiled without knowing of it
    m.instruction(w, H.COPY, "copy", [x, m.placeholder("z", (1, 16, 16, 3), H.FLOAT, np.float32)])
    m.compile(w)
    for graphs in (False, True):
        dm = H.DeviceManager(use_launch_graphs=graphs).init()
        if writer_first:
            dm.add_network(m, [w])
        dm.add_network(m, [f])
        for i in range(requests):
            a = _image(i)
            assert np.array_equal(_run(dm, a), _codes(a))
        if not writer_first:
            dm.add_network(m, [w])
        for i in range(12):
            z = _image(100 + i)
            dm.run("writer", {"z": z})
            assert np.array_equal(_run(dm), _codes(z)), (graphs, i)
        dm.evict_network("writer")
        assert np.array_equal(_run(dm), _codes(z))
        assert np.array_equal(_run(dm, a), _codes(a))
        dm.stop()


def values_bound_through_a_view():
    from glow_amd import host as H
    m, f, x = _image_module()
    half = m.view("half", x, (1, 8, 16, 3), H.FLOAT, byte_offset=8 * 16 * 3 * 4)   # the lower half
    m.compile(f)
    g = m.function("second")
    m.instruction(g, H.COPY, "copy", [m.placeholder("y", (1, 8, 16, 3), H.FLOAT, np.float32), half])
    m.compile(g)
    dm = H.DeviceManager().init()
    dm.add_network(m)
    a, b, y = _image(1), _image(2), np.zeros((1, 8, 16, 3), np.float32)
    assert np.array_equal(_run(dm, a), _codes(a))
    low = np.ascontiguousarray(b[:, 8:])
    dm.run("second", {"half": low, "y": y})
    a[:, 8:] = low
    assert np.array_equal(y, low) and np.array_equal(_run(dm), _codes(a))
    low = np.ascontiguousarray(b[:, :8])
    dm.transfer_static_placeholder(m, "half", low)
    a[:, 8:] = low
    assert np.array_equal(_run(dm), _codes(a))
    dm.stop()


def little_pinned_memory():
    from glow_amd import host as H
    os.environ["FAKE_DEVICE_PINNED_MOST"] = str(5 << 20)
    dm = H.DeviceManager(use_launch_graphs=False).init()
    small, f, _ = _image_module(100)
    small.compile(f)
    large, g, _ = _image_module(1100)        # 14.5 MB
    large.compile(g)
    dm.add_network(small)
    a = _image(1, 100)
    assert np.array_equal(_run(dm, a, 100), _codes(a))
    dm.evict_network("reader")
    dm.add_network(large)
    a = _image(2, 1100)
    assert np.array_equal(_run(dm, a, 1100), _codes(a))
    dm.evict_network("reader")
    dm.add_network(small)
    a = _image(3, 100)
    assert np.array_equal(_run(dm, a, 100), _codes(a))
    dm.stop()


def managers_side_by_side():
    import threading
    from glow_amd import host as H
    m, f, _ = _image_module()
    m.compile(f)
    dms = [H.DeviceManager().init() for _ in range(3)]
    wrong = []

    def serve(k, dm, loads):
        for load in range(loads):          # tuned and recorded anew each time
            dm.add_network(m)
            for i in range(15):
                a = _image(100 * k + i)
                if not np.array_equal(_run(dm, a), _codes(a)):
                    wrong.append((k, load, i))
            dm.evict_network("reader")
    threads = [threading.Thread(target=serve, args=(k, dm, 40)) for k, dm in enumerate(dms)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong, wrong[:5]
    for dm in dms:
        dm.stop()


def recordings_where_they_are_asked_for():
    from glow_amd import host as H
    m, f, _ = _image_module()
    m.compile(f)
    # launches one by one 0.98 of the recordings' time are no reason to leave them
    for graphs, direct_ms, recorded in ((-1, "0.1", True), (-4, "0.1", True), (True, "1", True),
                                        (3, "0.98", True), (True, "0.9", False), (2, "0.5", False),
                                        (False, "1", False)):
        os.environ["FAKE_DEVICE_DIRECT_MS"] = direct_ms
        dm = H.DeviceManager(use_launch_graphs=graphs).init()
        dm.add_network(m)
        for i in range(12):
            a = _image(i)
            assert np.array_equal(_run(dm, a), _codes(a)), (graphs, i)
        for i in range(3):
            before = FAKE.fake_graph_launches()
            a = _image(i)
            assert np.array_equal(_run(dm, a), _codes(a)), (graphs, i)
            assert FAKE.fake_graph_launches() - before == recorded, (graphs, direct_ms)
        assert (dm.recorded_branches("reader") > 0) == recorded, (graphs, direct_ms)
        dm.stop()


def launches_side_by_side():
    import threading
    from glow_amd import host as H
    m, f, _ = _image_module()
    m.compile(f)
    dms = [H.DeviceManager(use_launch_graphs=False).init() for _ in range(2)]
    for dm in dms:
        dm.add_network(m)
    os.environ["FAKE_DEVICE_MEET"] = "2"      # a launch waits for the other manager's
    right = [False, False]

    def serve(k):
        a = _image(k)
        right[k] = np.array_equal(_run(dms[k], a), _codes(a))
    threads = [threading.Thread(target=serve, args=(k,)) for k in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert all(right)
    for dm in dms:
        dm.stop()


# ---- in the parent -----------------------------------------------------------------

def test_each_manager_computes_from_its_own_image(fake_device):
    _in_child(fake_device, "one_function_on_two_managers")


def test_managers_load_and_run_one_function_side_by_side(fake_device):
    _in_child(fake_device, "managers_side_by_side")


@pytest.mark.parametrize("size", [16, 250, 2432])      # 2432: past the staging buffer
def test_a_function_loaded_behind_a_request_runs_on_its_image(fake_device, size):
    _in_child(fake_device, "function_loaded_behind_a_request", size)


@pytest.mark.parametrize("writer_first", [False, True])
@pytest.mark.parametrize("requests", [1, 4, 12])       # within and past the comparison of recordings
def test_a_reader_sees_what_another_function_wrote(fake_device, writer_first, requests):
    _in_child(fake_device, "writer_of_the_image", writer_first, requests)


def test_a_reader_sees_what_came_through_a_view(fake_device):
    _in_child(fake_device, "values_bound_through_a_view")


def test_networks_larger_than_the_pinned_memory_there_is(fake_device):
    _in_child(fake_device, "little_pinned_memory")


def test_recordings_serve_where_they_are_asked_for(fake_device):
    _in_child(fake_device, "recordings_where_they_are_asked_for")


def test_managers_issue_the_launches_of_one_function_side_by_side(fake_device):
    _in_child(fake_device, "launches_side_by_side")
