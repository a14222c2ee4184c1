"""The host side of the x-model (photonic_engines/slos/species.py:123-146), without a GPU."""
import math
from types import SimpleNamespace

import torch

from photonic_engines_amd.imperfections import Distinguishability
from photonic_engines_amd.slos import species


def test_weights_of_an_x_on_another_device(monkeypatch):
    """x need not be where U is: the kernels get the weights as host values."""
    n, x = 4, 0.7
    got = []
    plan = SimpleNamespace(xmodel=lambda U, order, weights, flags: got.append(weights) or torch.zeros(1, 35))
    kernel = SimpleNamespace(_plan=plan, input_modes=[0, 1, 2, 3], rdtype=torch.float32, compensated=False,
                             _out=lambda p, batched: p)
    monkeypatch.setattr(species, "_batched_u", lambda k, U: (U, True))
    monkeypatch.setattr(species, "spec", lambda d: Distinguishability(x=x))
    species.x_mixture(kernel, torch.zeros(1, 4, 4, dtype=torch.complex64), torch.empty((), device="meta"))
    w, = got
    assert isinstance(w, list) and all(isinstance(v, float) for v in w)
    ref = [x ** (n - L) * (1 - x) ** L for L in range(n + 1)]
    ref.append(math.comb(n, n) * ref[n] + math.comb(n, n - 1) * ref[n - 1])
    # x in float32 (half an ulp, 2^-24): x^(n-L) (1-x)^L is off by at most (n - L + L x / (1 - x)) 2^-24 < 3 n 2^-24
    assert all(abs(a - b) <= 3 * n * 2.0 ** -24 * b for a, b in zip(w, ref, strict=True))
