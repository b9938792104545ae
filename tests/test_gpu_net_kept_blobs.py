"""Blobs that an extract call leaves behind are what the model defines, also behind a residual block whose readers all quantise: its sum is
written in int8 alone only where the same call runs all of them and keeps nothing (light mode, src/net.cpp:344-600).  Outside light mode every
layer runs on its own and every blob stays."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def net():
    from ncnn_amd import host, zoo
    _, param, blob, _ = zoo.build("resnet50", n_calib=1)
    n = host.Net()
    n.set_use_hip_compute(True)
    assert n.register_int8_layers() == 0 and n.load_param_mem(param) == 0 and n.load_model_mem(blob) == 0
    return n


LEFT, SUM = "res2c_relu_splitncnn_4_1", "res2c_relu"


@pytest.mark.parametrize("light,first,then", [(True, "res3a_branch2a", LEFT), (True, "res3a_branch1", "res2c_relu_splitncnn_4_0"), (False, "res3a_branch2a", LEFT),
                                              (False, "fc1000", LEFT), (False, "fc1000", SUM), (False, "fc1000", "res3a_branch1")])
def test_later_extracts_of_the_same_pass(net, light, first, then):
    x = np.random.default_rng(5).random((2, 3, 64, 80), dtype=np.float32)

    def fresh(name):
        ex = net.create_extractor()
        ex.input("data", x)
        return ex.extract(name)
    ex = net.create_extractor()
    ex.set_lightmode(light)
    ex.input("data", x)
    print("[case] later extract", light, first, then, flush=True)
    assert np.array_equal(ex.extract(first), fresh(first))
    got, want = ex.extract(then), fresh(then)
    assert got.dtype == np.float32 and np.array_equal(got, want)


@pytest.mark.parametrize("batch,h,w", [(1, 64, 80), (2, 224, 224), (4, 224, 224)])
def test_light_mode_changes_no_score(net, batch, h, w):
    """Outside light mode every layer runs on its own and every sum is fp32.  In it the sums are int8, with their shortcuts in the same launch: all of them
    with few tiles; at four images the last stage's pair is left to two launches."""
    x = np.random.default_rng(batch).random((batch, 3, h, w), dtype=np.float32)
    print("[case] light mode", batch, h, w, flush=True)
    scores = []
    for light in (True, False):
        ex = net.create_extractor()
        ex.set_lightmode(light)
        ex.input("data", x)
        scores.append(ex.extract("fc1000"))
    assert np.array_equal(*scores)
