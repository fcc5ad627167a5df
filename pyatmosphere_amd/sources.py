"""Field sources (sources.py:8-23 of pyAtmosphere)."""
from dataclasses import dataclass

import numpy as np
import torch

from . import _lib
from ._lib import call, ptr
from .engine import gaussian_factors, to_device, value_key
from .gpu import device
from .theory.sources import GaussianBeam


@dataclass
class Source:
    wvl: float

    @property
    def k(self):
        return 2 * np.pi / self.wvl


class PlaneSource(Source):
    def output(self):
        return 1


class GaussianSource(GaussianBeam, Source):
    """Gaussian beam at z = 0 on the channel grid (sources.py:21-23;
    theory/sources.py:16-18), generated on the device from its two separable
    float64 factors."""

    def factors(self, n, delta):
        return gaussian_factors(n, delta, self.wvl, self.w0, self.F0)

    def output(self):
        grid = self.channel.grid
        n = grid.resolution[0]
        dev = device()
        if torch.cuda.is_current_stream_capturing():    # a graph would keep the factors' addresses
            raise RuntimeError("a source's factors cannot be uploaded or shared under graph capture")
        if getattr(self.factors, "__func__", None) is not GaussianSource.factors:
            # a subclass's or instance's own factors may depend on anything
            kept = (None, to_device(self.factors(n, grid.delta), dev))
        else:
            # the two factors last used stay on the device, by the values they are made from
            key = value_key(n, grid.delta, self.wvl, self.w0, self.F0), dev, _lib.stream_handle()
            kept = self.__dict__.get("_factors")
            if kept is None or kept[0] != key:
                kept = self._factors = (key, to_device(self.factors(n, grid.delta), dev))
        out = torch.empty(n, n, dtype=torch.complex64, device=dev)
        call("pa_outer", n, ptr(out), ptr(kept[1][0]), ptr(kept[1][1]), 1, _lib.stream_handle())
        return out

    def __getstate__(self):
        return {k: v for k, v in self.__dict__.items() if k != "_factors"}
