"""What the host library enqueues and when it waits, on a device made of host memory (fakedevice.cpp), in child processes."""
import os
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

COMMON = r'''
import ctypes as C, os, sys
import numpy as np
from ncnn_amd import host, modelwriter as mw
fake = C.CDLL(os.environ["LD_PRELOAD"])
L = host.lib()
F = np.float32
source = np.arange(-4, 8, dtype=F).reshape(3, 4)  # what the layer without inputs makes, on the host

def net_with(lines):
    """Net with the device path on and a host layer type "Source" that has no input."""
    keep = []
    def creator():
        layer = L.ncnn_layer_create()
        L.ncnn_layer_set_one_blob_only(layer, 0)
        def forward_n(self, bottoms, n, tops, n2, opt):
            m = host.Mat.from_numpy(source)
            tops[0] = m.h_
            m.h_ = None
            return 0
        fn = host.LayerTable._fields_[6][1](forward_n)
        keep.append(fn)
        layer.contents.forward_n = fn
        return layer
    net = host.Net()
    net.set_use_hip_compute(True)
    net.register_custom_layer("Source", creator, lambda layer: L.ncnn_layer_destroy(layer))
    assert net.load_param_mem(mw.assemble_param(lines)) == 0 and net.load_model_mem(b"") == 0
    net.keep = keep
    return net
'''


@pytest.fixture(scope="module")
def child(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("fakedevice") / "libfakedevice.so")
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-fPIC", "-shared", "-Wall", os.path.join(ROOT, "tests", "fakedevice.cpp"), "-o", so])

    def run(code):
        p = subprocess.run([sys.executable, "-c", COMMON + code + "\nprint('DONE')"], capture_output=True, text=True, timeout=120, cwd=ROOT,
                           env=dict(os.environ, LD_PRELOAD=so, PYTHONPATH=ROOT))
        assert p.returncode == 0 and p.stdout.strip().endswith("DONE"), (p.returncode, p.stdout[-800:], p.stderr[-2000:])
    return run


def test_a_recorded_pass_replays_on_new_inputs(child):
    child(r'''
net = net_with(["Input in0 0 1 data", "ReLU r 1 1 data out"])
x = np.linspace(-1, 1, 12, dtype=F).reshape(3, 4)
g = net.record("data", net.upload(x), "out")
for k in range(4):
    g.update_input(x + F(0.1 * k)); g.launch(); g.synchronize()
    assert np.array_equal(g.output().to_numpy(), np.maximum(x + F(0.1 * k), 0)), k
''')


@pytest.mark.parametrize("output", ["out", "src"])
def test_a_pass_that_takes_a_blob_from_a_host_layer_cannot_be_recorded(child, output):
    """Its upload would be replayed from a staging buffer that holds other bytes by then."""
    child(r'''
net = net_with(["Input in0 0 1 data", "Source s 0 1 src", "ReLU r 1 1 src out"])
x = np.ones((3, 4), F)
blob = net.upload(x)
for _ in range(4):  # eagerly it runs (and the command that record takes up has all its staging buffers)
    assert np.array_equal(net.create_extractor().extract("%(output)s"), np.maximum(source, 0) if "%(output)s" == "out" else source)
    net.create_extractor().extract_resident("%(output)s")
try:
    g = net.record("data", blob, "%(output)s")
except RuntimeError:
    g = None
if g is not None:
    for _ in range(4):  # uploads through the same staging buffers
        g.update_input(x * 7)
    g.launch(); g.synchronize()
    print("recorded; a replay gives", g.output().to_numpy())
assert g is None, "recorded"
assert np.array_equal(net.upload(x).to_numpy(), x)  # and the net still works
ex = net.create_extractor()
assert np.array_equal(ex.extract("out"), np.maximum(source, 0))
''' % {"output": output})


def test_a_resident_blob_that_came_from_the_host_is_ready_on_return(child):
    """Another Extractor may read it at once, on its own stream: a host layer's blob, and an input handed back.  A device
    layer's result is handed back without waiting, as ever."""
    child(r'''
net = net_with(["Input in0 0 1 data", "ReLU r0 1 1 data out0", "Source s 0 1 src", "Split sp 1 2 src a b", "ReLU r1 1 1 a out1"])
for name in ("src", "data", "b"):
    ex = net.create_extractor()
    ex.input("data", np.ones((8, 6, 6), F))
    blob = ex.extract_resident(name)
    assert fake.fake_pending() == 0, name
ex = net.create_extractor()
ex.input("data", np.ones((8, 6, 6), F))
out = ex.extract_resident("out0")
assert fake.fake_pending() > 0
''')
