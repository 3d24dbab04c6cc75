"""DeviceMobileNetV2.predict replays a recording: every answer is the one that its launches give, whatever was written
between two calls."""
import numpy as np
import pytest

from tfjs_amd import pyhost, workloads
from tfjs_amd.capi import HipBackendError

pytestmark = pytest.mark.gpu


@pytest.fixture
def model(tmp_path):
    pyhost.init()
    workloads.write_model(str(tmp_path), workloads.mobilenet_v2_weights(seed=3), np.uint8)
    m = workloads.DeviceMobileNetV2(str(tmp_path), 2)
    m.set_input(workloads.mobilenet_v2_input(2))
    yield m
    m.close()


def _launched(model):
    out = model.forward()
    logits = out.download(np.float32, 2000).reshape(2, 1000)
    out.free()
    return logits


def _replayed(model):
    """The logits of a replay: the bits of the launches (slices of k are added in the same order)."""
    got = model.predict()
    assert model._graph is not None
    np.testing.assert_array_equal(got.view(np.uint32), _launched(model).view(np.uint32))
    return got


def test_replays_see_new_pictures_and_new_weights(model):
    model.predict()
    first = _replayed(model)
    rng = np.random.default_rng(0)
    for _ in range(3):
        model.set_input(rng.uniform(-1, 1, (2, 224, 224, 3)))
        assert not np.array_equal(_replayed(model), first)
    # a filter that is searched for Inf / NaN, one that is not, a bias
    pair = next(op for op, _ in model.plan if op["kind"] == "pwdw")
    for name in (pair["w2"], pair["w"], pair["b2"]):
        before = _replayed(model)
        buf, shape = model.weights[name]
        old = buf.download(np.float32, int(np.prod(shape)))
        buf.upload(old * np.float32(0.5) + np.float32(0.01))
        assert not np.array_equal(_replayed(model), before)
        buf.upload(old)
        np.testing.assert_array_equal(_replayed(model), before)


def test_an_infinite_filter_is_not_replayed(model):
    model.predict()
    want = _replayed(model)
    buf, shape = model.weights[next(op["w2"] for op, _ in model.plan if op["kind"] == "pwdw")]
    old = buf.download(np.float32, int(np.prod(shape)))
    for bad in (np.inf, np.nan):
        broken = old.copy()
        broken[7] = bad
        buf.upload(broken)
        for call in (model.predict, model.forward, model.predict):
            with pytest.raises(HipBackendError, match="Inf or NaN"):
                call()
        buf.upload(old)
        assert np.array_equal(model.predict(), want) and model._graph is None
        np.testing.assert_array_equal(_replayed(model), want)


def test_exchanged_buffers_and_knobs_are_not_ignored(model):
    from tfjs_amd.capi import DeviceBuffer, check, load_library
    model.predict()
    want = _replayed(model)

    def changed(change, undo):
        change()
        got = model.predict()
        np.testing.assert_array_equal(got.view(np.uint32), _launched(model).view(np.uint32))
        np.testing.assert_array_equal(_replayed(model).view(np.uint32), got.view(np.uint32))
        undo()
        np.testing.assert_array_equal(model.predict(), want)
        np.testing.assert_array_equal(_replayed(model), want)
        return got

    pair = next(op for op, _ in model.plan if op["kind"] == "pwdw")
    own, shape = model.weights[pair["w"]]
    with DeviceBuffer.from_numpy(np.full(shape, 0.125, np.float32)) as other:
        got = changed(lambda: model.weights.update({pair["w"]: (other, shape)}),
                      lambda: model.weights.update({pair["w"]: (own, shape)}))
        assert not np.array_equal(got, want)
    own = model.input
    with DeviceBuffer.from_numpy(np.full((2, 224, 224, 3), 0.5, np.float32)) as other:
        got = changed(lambda: setattr(model, "input", other), lambda: setattr(model, "input", own))
        assert not np.array_equal(got, want)
    knob = load_library().tfhip_set_tuning
    changed(lambda: check(knob(b"tile", 3)), lambda: check(knob(b"tile", -1)))


def test_another_thread_launches_while_a_recording_is_open(model, monkeypatch):
    from concurrent.futures import ThreadPoolExecutor
    rng = np.random.default_rng(5)
    a, b = rng.uniform(-1, 1, (1, 33, 40)).astype(np.float32), rng.uniform(-1, 1, (1, 40, 50)).astype(np.float32)
    want, products = pyhost.fused_matmul(a, b), []
    want_logits = model.predict()
    with ThreadPoolExecutor(1) as other:
        def multiply(i, op):   # upload, launch and download, while this thread records
            products.append(other.submit(pyhost.fused_matmul, a, b).result())

        launches = model.forward
        monkeypatch.setattr(model, "forward", lambda: launches(before=multiply))
        model.predict()
    monkeypatch.undo()
    assert model._graph is not None and len(products) == len(model.plan)
    for got in products:
        np.testing.assert_array_equal(got, want)
    np.testing.assert_array_equal(_replayed(model), want_logits)
