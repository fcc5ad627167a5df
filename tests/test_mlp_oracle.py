"""The float64 MLP oracle's gradients against central finite differences."""
import numpy as np
import pytest

from oracle import mlp


def test_gradients_finite_differences():
    rng = np.random.default_rng(0)
    sizes = [5, 7, 6, 9]   # 8 bins + 1 log-variance
    params = [(rng.normal(size=(o, i)) * 0.5, rng.normal(size=o) * 0.1) for i, o in zip(sizes[:-1], sizes[1:])]
    x = rng.normal(size=(4, 5))
    t = rng.random((4, 8))
    t /= t.sum(axis=1, keepdims=True)
    tv = rng.normal(size=4)
    loss, grads = mlp.loss_and_grad(params, x, t, tv, 0.3, 0.7)
    eps = 1e-6
    for li, (W, b) in enumerate(params):
        for arr, g in ((W, grads[li][0]), (b, grads[li][1])):
            for idx in [tuple(rng.integers(0, s) for s in arr.shape) for _ in range(5)]:
                old = arr[idx]
                arr[idx] = old + eps
                lp, _ = mlp.loss_and_grad(params, x, t, tv, 0.3, 0.7)
                arr[idx] = old - eps
                lm, _ = mlp.loss_and_grad(params, x, t, tv, 0.3, 0.7)
                arr[idx] = old
                assert abs((lp - lm) / (2 * eps) - g[idx]) < 1e-6 * max(1, abs(g[idx]))


def test_softmax_ce_minimum_at_target():
    """The head loss is minimised (gradient zero) when softmax(logits) = target."""
    t = np.array([[0.1, 0.2, 0.7]])
    W = np.eye(4)[:, :4]
    params = [(np.eye(4), np.zeros(4))]
    x = np.concatenate([np.log(t), [[0.5]]], axis=1)
    _, grads = mlp.loss_and_grad(params, x, t, np.array([0.5]), 1.0)
    assert np.abs(grads[0][1]).max() < 1e-12


def test_prediction_goes_through_an_overridden_output():
    """predict and SurrogateEnsemble.pdt take what a subclass's or an instance's own
    predict_raw or predict gives (no device is touched)."""
    import torch
    from pyatmosphere_amd.surrogate import NB, PDTSurrogate, SurrogateEnsemble
    rng = np.random.default_rng(0)
    out = rng.normal(size=(6, NB + 1))
    x = rng.uniform(-1, 1, (6, 5)).astype(np.float32)

    class Fixed(PDTSurrogate):
        def predict_raw(self, x):
            return out

    lg = out[:, :NB]
    want = np.exp(lg) / np.exp(lg).sum(axis=1, keepdims=True)
    net = Fixed(width=16, depth=2, device=torch.device("cpu"))
    p, lv = net.predict(x)
    assert np.allclose(p, want, rtol=1e-13) and np.array_equal(lv, out[:, NB])
    assert np.allclose(SurrogateEnsemble([net, net], 0.1).pdt(x)[0], want, rtol=1e-13)
    plain = PDTSurrogate(width=16, depth=2, device=torch.device("cpu"))
    plain.predict = lambda x: (want, out[:, NB])
    mean, lv, spread, _ = SurrogateEnsemble([plain, net], 0.1).pdt(x)
    assert np.allclose(mean, want, rtol=1e-13) and np.allclose(lv, out[:, NB]) and spread.max() < 1e-13


def test_inputs_go_through_an_overridden_pad(monkeypatch):
    """A subclass with its own input padding predicts from what it gives."""
    import torch
    from pyatmosphere_amd.surrogate import NB, PDTSurrogate
    from pyatmosphere_amd.surrogate import model

    seen = []

    class Scaled(PDTSurrogate):
        def _pad(self, x):
            return super()._pad(2 * x)

    def call(name, M, fo, fi, h, W, b, y, act, stream):
        assert name == "pa_mlp_layer_bf16"
        if not seen:
            import ctypes
            seen.append(np.ctypeslib.as_array((ctypes.c_float * (M * fi)).from_address(h)).reshape(M, fi).copy())

    monkeypatch.setattr(model, "call", lambda name, *a: call(name, *a) if name != "pa_mlp_to_bf16" else None)
    monkeypatch.setattr(model._lib, "stream_handle", lambda: 0)
    x = np.random.default_rng(1).uniform(-1, 1, (3, 5)).astype(np.float32)
    Scaled(width=32, depth=2, device=torch.device("cpu")).predict_raw(x)
    assert np.array_equal(seen[0][:, :5], 2 * x)


@pytest.mark.parametrize("layers", [16, 17, 256, 257, 1000])
def test_any_number_of_layers(layers):
    """The scratch of a training step and the packed size (0: not for the fused network,
    which takes 16 layers) of networks of any depth (host functions)."""
    from pyatmosphere_amd._lib import call, int_array
    sizes = int_array([16] * layers + [65])
    rows = 5
    assert call("pa_mlp_loss_grads_scratch", layers, sizes, rows) == 4 * (3 * 80 * (layers - 1) + 2 * 328)
    assert (call("pa_mlp_pack_bytes", layers, sizes) > 0) == (layers <= 16)


@pytest.mark.parametrize("layers", [2, 20])
def test_layers_one_by_one_ask_for_the_stream_once(monkeypatch, layers):
    """Networks that go layer by layer do not pay for the current stream at each layer."""
    import torch
    from pyatmosphere_amd.surrogate import PDTSurrogate
    from pyatmosphere_amd.surrogate import model
    asked = []
    monkeypatch.setattr(model, "call", lambda name, *a: None)
    monkeypatch.setattr(model._lib, "stream_handle", lambda: asked.append(1) or 0)
    net = PDTSurrogate(width=32, depth=layers, device=torch.device("cpu"))
    x = np.zeros((3, 5), np.float32)
    net._layer_by_layer(x)          # lays the weights out too
    assert len(asked) <= 2
    asked.clear()
    net._layer_by_layer(x)
    assert len(asked) == 1
