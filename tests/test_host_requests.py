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
SIZE, SCALE, OFFSET = 16, 0.05, 3
ELEMENTS = SIZE * SIZE * 3


@pytest.fixture(scope="module")
def fake_device(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("fake") / "libfake_device.so")
    subprocess.check_call(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-I",
                           os.path.join(ROOT, "include"),
                           os.path.join(ROOT, "tests", "fake_device.cpp"), "-o", so])
    return so


def _in_child(fake_device, scenario):
    r = subprocess.run([sys.executable, "-c",
                        f"from tests import test_host_requests as t; t.bind({fake_device!r}); "
                        f"t.{scenario}()"], cwd=ROOT, capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, r.stderr[-3000:]


def bind(so):
    C.CDLL(so, C.RTLD_GLOBAL)


# ---- in the child ------------------------------------------------------------------

def _stem(m, f, x):
    """out = the convolution of quantize(x); the fake kernels hand quantize(x) through."""
    from glow_amd import host as H
    out = m.placeholder("out", (1, SIZE // 2, SIZE // 2, 16), H.INT8Q, np.int8, 2.0, -3)
    ops = [m.constant("f", np.ones((16, 3, 3, 3), np.int8), H.INT8Q),
           m.constant("b", np.zeros(16, np.int32), H.INT32Q),
           m.constant("fs", np.full(16, 0.01, np.float32), H.FLOAT),
           m.constant("fo", np.zeros(16, np.int32), H.INT32I),
           m.constant("bs", np.full(16, 0.01 * SCALE, np.float32), H.FLOAT),
           m.constant("bo", np.zeros(16, np.int32), H.INT32I)]
    q = m.activation(f, "q", (1, SIZE, SIZE, 3), H.INT8Q, SCALE, OFFSET)
    m.instruction(f, H.QUANTIZE, "quantize", [q, x])
    m.instruction(f, H.CHANNELWISE_QUANTIZED_CONV, "stem", [out, q, *ops],
                  H.conv_attrs((3, 3), (2, 2), (1, 1, 1, 1)))


def _image_module():
    from glow_amd import host as H
    m = H.Module("images")
    x = m.placeholder("x", (1, SIZE, SIZE, 3), H.FLOAT, np.float32)
    f = m.function("reader")
    _stem(m, f, x)
    return m, f, x


def _image(seed):
    return np.random.default_rng(seed).normal(0, 2, (1, SIZE, SIZE, 3)).astype(np.float32)


def _codes(x):
    return np.clip(np.rint(x / np.float32(SCALE) + np.float32(OFFSET)), -128, 127).astype(np.int8)


def _run(dm, x=None):
    out = np.zeros((1, SIZE // 2, SIZE // 2, 16), np.int8)
    dm.run("reader", {"out": out} if x is None else {"x": x, "out": out})
    return out.reshape(-1)[:ELEMENTS]


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
            assert np.array_equal(_run(second, b), _codes(b).reshape(-1)), (graphs, i)
            assert np.array_equal(_run(first, a), _codes(a).reshape(-1)), (graphs, i)
            assert np.array_equal(_run(second), _codes(b).reshape(-1)), (graphs, i)
        second.stop()
        for a in images:
            assert np.array_equal(_run(first, a), _codes(a).reshape(-1)), graphs
        first.stop()


# ---- in the parent -----------------------------------------------------------------

def test_each_manager_computes_from_its_own_image(fake_device):
    _in_child(fake_device, "one_function_on_two_managers")
