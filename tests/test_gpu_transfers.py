"""Blobs on their way to the device and back, bit for bit: the staging pieces of an upload (whole samples, pixel ranges of a
sample larger than a 2 MB piece, odd planes, padded and dense strides) and the one-launch and chunked downloads."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(7,), (1, 3), (5, 700001), (3, 2, 5), (3, 193, 257), (2, 3, 193, 257), (40, 3, 64, 64), (1, 4, 900, 901), (2, 3, 600, 601),
                                   (5, 17, 33, 31), (2, 96, 90, 91), (3, 1, 1, 1)], ids=str)
@pytest.mark.parametrize("dtype", [np.float32, np.int8], ids=["fp32", "int8"])
def test_upload_and_download_return_the_same_bits(shape, dtype):
    from ncnn_amd import host
    print(shape, dtype, flush=True)
    rng = np.random.default_rng(1)
    x = rng.integers(-127, 128, shape).astype(dtype)
    if dtype == np.float32:
        x += rng.random(shape, dtype=np.float32)
    net = host.Net()
    net.set_use_hip_compute(True)
    want = x[0] if x.ndim == 4 and x.shape[0] == 1 else x
    assert np.array_equal(net.upload(x).to_numpy(), want)                        # read where it lies
    assert np.array_equal(net.upload(host.Mat.from_numpy(x)).to_numpy(), want)   # ncnn's own layout (padded planes and samples)


def test_a_host_array_may_be_reused_once_it_was_fed():
    from ncnn_amd import host, zoo
    g, param, blob, _ = zoo.build("tiny", seed=21)
    net = host.Net()
    net.set_use_hip_compute(True)
    assert net.register_int8_layers() == 0 and net.load_param_mem(param) == 0 and net.load_model_mem(blob) == 0
    a, b = np.random.default_rng(3).random((2, 5) + tuple(g.input_shape), dtype=np.float32)

    def scores(x):
        ex = net.create_extractor()
        ex.input("data", x)
        return ex.extract("fc")
    want_a, want_b = scores(a.copy()), scores(b.copy())
    x = a.copy()
    first = net.create_extractor()
    first.input("data", x)
    x[:] = b
    second = net.create_extractor()
    second.input("data", x)
    x[:] = 0
    assert np.array_equal(first.extract("fc"), want_a) and np.array_equal(second.extract("fc"), want_b)


def test_a_pass_with_a_host_source_layer_cannot_be_recorded():
    """A blob made on the host has to be uploaded in the middle of the pass: run eagerly, refused by a recording, and the
    net works on afterwards (what a replay would do to it: tests/test_device_queue.py)."""
    from ncnn_amd import host, modelwriter as mw
    L = host.lib()
    source = np.arange(-4, 8, dtype=np.float32).reshape(3, 4)
    keep = []

    def creator():
        layer = L.ncnn_layer_create()
        L.ncnn_layer_set_one_blob_only(layer, 0)

        def forward_n(self, bottoms, n, tops, n2, opt):
            m = host.Mat.from_numpy(source)
            tops[0] = m.h_
            m.h_ = None
            return 0
        keep.append(host.LayerTable._fields_[6][1](forward_n))
        layer.contents.forward_n = keep[-1]
        return layer
    net = host.Net()
    net.set_use_hip_compute(True)
    net.register_custom_layer("Source", creator, lambda layer: L.ncnn_layer_destroy(layer))
    lines = ["Input in0 0 1 data", "Source s 0 1 src", "ReLU r 1 1 src out"]
    assert net.load_param_mem(mw.assemble_param(lines)) == 0 and net.load_model_mem(b"") == 0
    x = np.ones((3, 4), np.float32)
    blob = net.upload(x)
    for _ in range(4):
        assert np.array_equal(net.create_extractor().extract("out"), np.maximum(source, 0))
    for output in ("out", "src"):
        with pytest.raises(RuntimeError):
            net.record("data", blob, output)
    assert np.array_equal(net.create_extractor().extract("out"), np.maximum(source, 0))
    assert np.array_equal(blob.to_numpy(), x)
