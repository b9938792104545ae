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
