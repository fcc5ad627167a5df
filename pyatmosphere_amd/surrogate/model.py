"""Transmittance-PDT surrogate: a small MLP trained and evaluated with the
project's own HIP kernels (libpa_hip.so pa_mlp_*).

Inputs (5, encoded to [-1, 1]-ish): log10 Cn2, path length L, beam waist w0,
aperture radius a, wavelength.  Outputs: NB = 64 logits of the transmittance
PDT over [0, 1] (softmax -> bin probabilities) and log of the beam-wander
variance sigma_BW,x^2 = <x_c^2> (simulations/beam.py:35-38).

Training: float32 master weights, float32 MFMA GEMMs, softmax
cross-entropy + a ranked-probability (squared CDF distance) term + weighted
log-variance MSE, Adam.  Inference: bf16 MFMA GEMMs
with float32 accumulation and fused bias + SiLU.
"""
from __future__ import annotations

from typing import List, Optional, Sequence, Tuple

import numpy as np
import torch

from .. import _lib
from .._lib import call, ptr, ptr_array

NB = 64
IN_FEATURES = 5
IN_PAD = 16
MAX_FUSED_MEMBERS = 8        # pa_mlp_pdt's limit
DOMAIN = {
    "log10_cn2": (-16.0, -14.0),
    "L": (1e3, 50e3),
    "w0": (0.02, 0.2),
    "a": (0.05, 0.3),
    "wvl": (808e-9, 1550e-9),
}


def encode(log10_cn2, L, w0, a, wvl) -> np.ndarray:
    """(M, 5) float32 network inputs scaled to [-1, 1] over the training domain
    (the path length on a log scale)."""
    cols = []
    for key, v in (("log10_cn2", log10_cn2), ("L", L), ("w0", w0), ("a", a), ("wvl", wvl)):
        lo, hi = DOMAIN[key]
        v = np.asarray(v, np.float64)
        if key == "L":
            v, lo, hi = np.log(v), np.log(lo), np.log(hi)
        cols.append((v - lo) / (hi - lo) * 2 - 1)
    return np.stack(cols, axis=-1).astype(np.float32)


def in_domain(x: np.ndarray, tol: float = 1e-6) -> np.ndarray:
    return np.all(np.abs(x) <= 1 + tol, axis=-1)


def _flat(pairs) -> List[torch.Tensor]:
    return [t for pair in pairs for t in pair]


class PDTSurrogate:
    """MLP with `depth` linear layers of width `width` (SiLU between)."""

    def __init__(self, width: int = 256, depth: int = 4, seed: int = 0, device=None, wv: float = 1.0,
                 wc: float = 4.0):
        self.device = device or torch.device("cuda", torch.cuda.current_device())
        self.sizes = [IN_PAD] + [width] * (depth - 1) + [NB + 1]
        self.wv, self.wc = wv, wc
        rng = np.random.default_rng(seed)
        self.params: List[Tuple[torch.Tensor, torch.Tensor]] = []
        for i, (fi, fo) in enumerate(zip(self.sizes[:-1], self.sizes[1:])):
            fan_in = IN_FEATURES if i == 0 else fi
            W = rng.normal(0, np.sqrt(2.0 / fan_in), size=(fo, fi)).astype(np.float32)
            if i == 0:
                W[:, IN_FEATURES:] = 0.0
            if i == len(self.sizes) - 2:
                W *= 0.1
            b = np.zeros(fo, np.float32)
            self.params.append((torch.from_numpy(W).to(self.device), torch.from_numpy(b).to(self.device)))
        self.m = [(torch.zeros_like(W), torch.zeros_like(b)) for W, b in self.params]
        self.v = [(torch.zeros_like(W), torch.zeros_like(b)) for W, b in self.params]
        self.t = 0
        self._bf16 = None

    # ------------------------------------------------------------ io
    def state(self) -> dict:
        d = {"sizes": np.array(self.sizes), "wv": np.array(self.wv), "wc": np.array(self.wc)}
        for i, (W, b) in enumerate(self.params):
            d[f"W{i}"] = W.cpu().numpy()
            d[f"b{i}"] = b.cpu().numpy()
        return d

    def save(self, path: str) -> None:
        np.savez(path, **self.state())

    @classmethod
    def load(cls, path: str, device=None) -> "PDTSurrogate":
        z = np.load(path, allow_pickle=False)
        sizes = [int(s) for s in z["sizes"]]
        net = cls(width=sizes[1], depth=len(sizes) - 1, device=device, wv=float(z["wv"]),
                  wc=float(z["wc"]) if "wc" in z else 0.0)
        net.params = [(torch.from_numpy(z[f"W{i}"]).to(net.device), torch.from_numpy(z[f"b{i}"]).to(net.device))
                      for i in range(len(sizes) - 1)]
        net.m = [(torch.zeros_like(W), torch.zeros_like(b)) for W, b in net.params]
        net.v = [(torch.zeros_like(W), torch.zeros_like(b)) for W, b in net.params]
        return net

    def numpy_params(self):
        """float64 (W, b) pairs with the input padding removed (oracle layout)."""
        out = []
        for i, (W, b) in enumerate(self.params):
            Wn = W.cpu().numpy().astype(np.float64)
            if i == 0:
                Wn = Wn[:, :IN_FEATURES]
            out.append((Wn, b.cpu().numpy().astype(np.float64)))
        return out

    # ------------------------------------------------------------ training kernels
    def _pad(self, x: np.ndarray) -> torch.Tensor:
        xp = np.zeros((x.shape[0], IN_PAD), np.float32)
        xp[:, :IN_FEATURES] = x
        return torch.from_numpy(xp).to(self.device)

    def loss_and_grads(self, X: torch.Tensor, T: torch.Tensor, TV: torch.Tensor):
        """Mean loss (device scalar) and gradients [(dW, db)] for one batch."""
        M, layers = X.shape[0], len(self.params)
        sizes = self._layer_sizes()
        loss = torch.empty(M + 1, dtype=torch.float32, device=self.device)    # the rows' losses, their mean
        scratch = torch.empty(call("pa_mlp_loss_grads_scratch", layers, sizes, M), dtype=torch.uint8,
                              device=self.device)
        grads = [(torch.empty_like(W), torch.empty_like(b)) for W, b in self.params]
        call("pa_mlp_loss_grads", layers, sizes, M, ptr(X), ptr_array(_flat(self.params)), ptr(T), ptr(TV),
             float(self.wv), float(self.wc), ptr(loss), ptr(loss) + 4 * M, ptr_array(_flat(grads)), ptr(scratch),
             _lib.stream_handle())
        return loss[M], grads

    def adam_step(self, grads, lr: float, b1=0.9, b2=0.999, eps=1e-8) -> None:
        self.t += 1
        layers = list(zip(self.params, grads, self.m, self.v))
        w, g, m, v = (_flat(pairs) for pairs in zip(*layers))
        call("pa_mlp_adam_multi", len(w), _lib.int_array([p.numel() for p in w]), ptr_array(w), ptr_array(g),
             ptr_array(m), ptr_array(v), lr, b1, b2, eps, self.t, _lib.stream_handle())
        self._bf16 = None

    def train(self, x: np.ndarray, target: np.ndarray, tvar: np.ndarray, steps: int, batch: int = 512,
              lr: float = 2e-3, lr_final: float = 5e-5, seed: int = 0, log_every: int = 0) -> List[float]:
        """Adam over shuffled minibatches with a cosine learning-rate decay."""
        rng = np.random.default_rng(seed)
        X = self._pad(x)
        T = torch.from_numpy(np.ascontiguousarray(target, np.float32)).to(self.device)
        TV = torch.from_numpy(np.ascontiguousarray(tvar, np.float32)).to(self.device)
        n = x.shape[0]
        hist = []
        for it in range(steps):
            idx = torch.from_numpy(rng.integers(0, n, size=min(batch, n))).to(self.device)
            loss, grads = self.loss_and_grads(X[idx].contiguous(), T[idx].contiguous(), TV[idx].contiguous())
            frac = it / max(1, steps - 1)
            lr_t = lr_final + 0.5 * (lr - lr_final) * (1 + np.cos(np.pi * frac))
            self.adam_step(grads, lr_t)
            if log_every and (it % log_every == 0 or it == steps - 1):
                hist.append(float(loss.item()))
        return hist

    # ------------------------------------------------------------ inference (bf16 MFMA)
    def _layer_sizes(self):
        return _lib.int_array([self.params[0][0].shape[1]] + [W.shape[0] for W, _ in self.params])

    def _packed(self) -> Optional[torch.Tensor]:
        """The weights in the fused network's order (pa_mlp_pack_bf16), laid out
        once per set of weights; None for networks too wide or deep for it."""
        if self._bf16 is None:
            sizes, layers = self._layer_sizes(), len(self.params)
            size = call("pa_mlp_pack_bytes", layers, sizes)
            if not size:
                return None
            packed = torch.empty(size, dtype=torch.uint8, device=self.device)
            call("pa_mlp_pack_bf16", layers, sizes, ptr_array(_flat(self.params)), ptr(packed), _lib.stream_handle())
            self._bf16 = packed
        return self._bf16 if torch.is_tensor(self._bf16) else None

    def _bf16_layers(self):
        """Per layer (weights, bias, width, padded width, inputs) for the networks
        that the fused launch does not take."""
        if not isinstance(self._bf16, list):
            s = _lib.stream_handle()
            layers = []
            for W, b in self.params:
                fo, fi = W.shape
                fo_p = ((fo + 31) // 32) * 32
                Wp = torch.zeros(fo_p, fi, dtype=torch.float32, device=self.device)
                Wp[:fo] = W
                bp = torch.zeros(fo_p, dtype=torch.float32, device=self.device)
                bp[:fo] = b
                Wb = torch.empty(fo_p, fi, dtype=torch.int16, device=self.device)
                call("pa_mlp_to_bf16", Wp.numel(), ptr(Wp), ptr(Wb), s)
                layers.append((Wb, bp, fo, fo_p, fi))
            self._bf16 = layers
        return self._bf16

    def _layer_by_layer(self, x: np.ndarray) -> torch.Tensor:
        """(M, outputs) device outputs, one launch per layer."""
        h = self._pad(x)
        M, layers, s = h.shape[0], self._bf16_layers(), _lib.stream_handle()
        for i, (Wb, bp, fo, fo_p, fi) in enumerate(layers):
            y = torch.empty(M, fo_p, dtype=torch.float32, device=self.device)
            call("pa_mlp_layer_bf16", M, fo_p, fi, ptr(h), ptr(Wb), ptr(bp), ptr(y), int(i < len(layers) - 1), s)
            h = y if fo_p == fo else y[:, :fo].contiguous()
        return h

    def _plain(self, *names: str) -> bool:
        """Whether neither a subclass nor the instance has its own methods `names`."""
        return all(getattr(getattr(self, f), "__func__", None) is getattr(PDTSurrogate, f) for f in names)

    def predict_raw(self, x: np.ndarray) -> np.ndarray:
        """(M, NB + 1) outputs on bf16 MFMA."""
        out = _outputs([self], x)[0] if self._plain("_pad") else self._layer_by_layer(x)[:, :NB + 1]
        return out.cpu().numpy().astype(np.float64)

    def predict(self, x: np.ndarray) -> Tuple[np.ndarray, np.ndarray]:
        """Bin probabilities (M, NB) of the transmittance PDT and log sigma_BW,x^2."""
        if self._plain("_pad", "predict_raw"):
            return _distributions([self], x)[:2]
        out = self.predict_raw(x)
        lg = out[:, :NB]
        p = np.exp(lg - lg.max(axis=1, keepdims=True))
        return p / p.sum(axis=1, keepdims=True), out[:, NB]


def _outputs(members: Sequence[PDTSurrogate], x: np.ndarray) -> torch.Tensor:
    """(members, M, NB + 1) float32 device outputs; the members share a device.
    Networks of one shape run in one launch."""
    dev, M = members[0].device, x.shape[0]
    packs = [m._packed() for m in members]
    if any(p is None for p in packs) or \
            len(members) > 1 and len({tuple(p.shape for p in _flat(m.params)) for m in members}) > 1:
        if len(members) > 1:
            return torch.cat([_outputs([m], x) for m in members])
        return members[0]._layer_by_layer(x)[None, :, :NB + 1].contiguous()
    xs = np.empty((M, IN_FEATURES), np.float32)
    xs[:] = x
    xd = torch.empty(M, IN_FEATURES, dtype=torch.float32, device=dev)
    xd.copy_(torch.from_numpy(xs).pin_memory(), non_blocking=True)
    out = torch.empty(len(members), M, members[0].params[-1][0].shape[0], dtype=torch.float32, device=dev)
    call("pa_mlp_infer", len(members[0].params), members[0]._layer_sizes(), IN_FEATURES, len(members),
         ptr_array(packs), M, ptr(xd), ptr(out), _lib.stream_handle())
    return out[:, :, :NB + 1].contiguous()


def _distributions(members: Sequence[PDTSurrogate], x: np.ndarray):
    """The members' mean PDT (M, NB), mean log variance (M,) and spread (M,)
    (KS distance between a member and the mean), float64: softmax and ensemble
    statistics on the device, one copy back."""
    logits = _outputs(members, x)
    M = logits.shape[1]
    dist = torch.empty(M * (NB + 2), dtype=torch.float64, device=logits.device)
    call("pa_mlp_pdt", len(members), M, ptr(logits), ptr(dist), _lib.stream_handle())
    host = torch.empty(dist.shape, dtype=dist.dtype, pin_memory=True)
    host.copy_(dist, non_blocking=True)
    torch.cuda.current_stream(dist.device).synchronize()
    # copied out of the staging memory, which an answer that is kept would hold
    parts = host[:M * NB].clone(), host[M * NB:M * (NB + 1)].clone(), host[M * (NB + 1):].clone()
    return parts[0].numpy().reshape(M, NB), parts[1].numpy(), parts[2].numpy()


def ks_binned(p: np.ndarray, q: np.ndarray) -> np.ndarray:
    """Kolmogorov-Smirnov distance between binned distributions over the same
    bins (max |CDF difference| at the bin edges)."""
    return np.abs(np.cumsum(p, axis=-1) - np.cumsum(q, axis=-1)).max(axis=-1)


class SurrogateEnsemble:
    """Members trained from different seeds; the spread of their PDTs is the
    confidence signal.  `pdt(...)` returns the ensemble mean, and a mask of the
    rows whose inputs are outside the training domain or whose members disagree
    by more than `max_spread` (KS between a member and the mean), which the
    caller answers with the full simulation."""

    def __init__(self, members: Sequence[PDTSurrogate], max_spread: float = 0.04):
        self.members = list(members)
        self.max_spread = max_spread

    def pdt(self, x: np.ndarray):
        if 0 < len(self.members) <= MAX_FUSED_MEMBERS and len({m.device for m in self.members}) == 1 \
                and all(type(m) is PDTSurrogate and m._plain("_pad", "predict_raw", "predict") for m in self.members):
            mean, lv, spread = _distributions(self.members, x)
        else:
            preds = [m.predict(x) for m in self.members]
            ps = np.stack([p for p, _ in preds])
            mean = ps.mean(axis=0)
            spread = np.max([ks_binned(p, mean) for p in ps], axis=0)
            lv = np.mean([v for _, v in preds], axis=0)
        fallback = (spread > self.max_spread) | ~in_domain(x)
        return mean, lv, spread, fallback
