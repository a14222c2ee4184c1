"""The one-call x-model (slos_xmodel; photonic_engines/slos/species.py:123-146)."""
import itertools
import math

import numpy as np
import pytest
import torch
from helpers import haar_unitary

from photonic_engines_amd.slos import FockSLOSKernel

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _interfering(U, cols, t):
    """|<t| U |cols>|^2 for distinct columns, in FP64."""
    if not cols:
        return 1.0
    a = sum(math.prod([complex(U[t[i], c]) for i, c in enumerate(p)]) for p in itertools.permutations(cols))
    return abs(a) ** 2 / math.prod(math.factorial(t.count(j)) for j in set(t))


def test_more_than_2_to_32_states():
    """4 photons in 566 modes, 4.32e9 states: more than one launch has threads."""
    n, m, x = 4, 566, 0.7
    U = haar_unitary(m, 9).to(torch.complex64)
    k = FockSLOSKernel(n, m, [1] * n + [0] * (m - n), device=DEV)
    S = k.output_size()
    assert S > 1 << 32
    p = k.probs(U.to(DEV), indist=x, order=1)
    mass = float(k.total_mass(p))
    assert abs(mass - (x ** n + n * x ** (n - 1) * (1 - x))) < 1e-5
    rng = np.random.default_rng(3)
    idx = sorted({0, 255, (1 << 28) - 1, 1 << 28, (1 << 32) - 1, 1 << 32, S - 1, *rng.integers(0, S, 12).tolist(),
                  *rng.integers(1 << 32, S, 6).tolist()})
    U64 = U.to(torch.complex128).numpy()
    for i, t in zip(idx, k._plan.unrank(n, idx).tolist()):
        ref = x ** n * _interfering(U64, list(range(n)), t)
        for j in range(n):  # photon j distinguishable, leaving at any of the distinct modes of t
            rest = [c for c in range(n) if c != j]
            for mode in sorted(set(t)):
                less = list(t)
                less.remove(mode)
                ref += x ** (n - 1) * (1 - x) * abs(U64[mode, j]) ** 2 * _interfering(U64, rest, less)
        # (at most 12 factors and a sum of at most 24 permutations' products on 4 layers, each within 2^-24 of
        # the products' own size, which a Haar matrix's entries bound by 24 (4 / m)^4)
        assert abs(float(p[i]) - ref) <= 1e-4 * ref + 1e-6 * 24 * (4 / m) ** 4, (i, t)
