"""The host side of the x-model (photonic_engines/slos/species.py:123-146), without a GPU."""
import ctypes
import math
from types import SimpleNamespace

import numpy as np
import torch

from photonic_engines_amd import _native as nat
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


def test_more_photons_than_modes_are_refused():
    """A subset's photons are the columns of an m x m matrix: with n > m the one-call x-model would write
    past it. The C entries refuse; the layer-by-layer form, which raises for it, gets the call."""
    L = nat.lib()
    for n, m, rc in ((3, 2, nat.SLOS_EINVAL), (13, 10, nat.SLOS_EINVAL), (3, 3, nat.SLOS_OK), (13, 13, nat.SLOS_OK)):
        h = ctypes.c_void_p()
        assert L.slos_plan_create(n, m, nat.MASK_IDS["fock"], (ctypes.c_int32 * n)(*[i % m for i in range(n)]), ctypes.byref(h)) == 0
        b = ctypes.c_size_t()
        assert L.slos_xmodel_workspace(h, 1, 1, 0, ctypes.byref(b)) == rc
        L.slos_plan_destroy(h)
    kernel = SimpleNamespace(_plan=SimpleNamespace(xmodel=lambda *a: torch.zeros(1, 4)), input_modes=[0, 0, 1], compensated=False)
    for m in (2, 3):
        native = species._native_x(kernel, torch.zeros(1, m, m, dtype=torch.complex64), torch.tensor(0.7), 0.7, 1)
        assert (native is None) == (m == 2)


def test_weights_differentiate_twice_at_the_ends():
    """d^2/dx^2 of x^(n-L) (1-x)^L, also where x or 1 - x is zero."""
    n = 4
    for x0 in (0.0, 0.3, 1.0):
        x = torch.tensor(x0, dtype=torch.float64, requires_grad=True)
        w = list(species._weights(x, n, n))[:n + 1]
        for L in range(n + 1):
            g, = torch.autograd.grad(w[L], x, create_graph=True)
            h, = torch.autograd.grad(g, x, retain_graph=True)
            p = np.polynomial.Polynomial([0, 1]) ** (n - L) * np.polynomial.Polynomial([1, -1]) ** L
            assert abs(g.item() - p.deriv()(x0)) < 1e-12 and abs(h.item() - p.deriv(2)(x0)) < 1e-12, (x0, L)
