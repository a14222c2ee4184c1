"""Infinite and NaN values reach only the results that depend on them."""
import pytest
import torch

from photonic_engines_amd.slos import FockSLOSKernel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bad", [float("nan"), float("inf")])
@pytest.mark.parametrize("n,m,mask", [(3, 6, "unbunched"), (3, 6, "dual_rail"), (2, 8, "sparse_1in4"), (3, 40, "unbunched")])
def test_adjoint_without_a_child(n, m, mask, bad):
    """One adjoint layer with a non-finite parent amplitude and a non-finite coefficient: dL/dU[j] and the
    parents' gradients are non-finite exactly where an edge joins them."""
    step = {"dual_rail": 2, "sparse_1in4": 4}.get(mask, 1)
    k = FockSLOSKernel(n, m, [1 if j % step == 0 and j // step < n else 0 for j in range(m)], mask=mask, device="cuda")
    p = k._plan
    Sp, Sk = p.sizes[n - 1], p.sizes[n]
    rows = {tuple(s): i for i, s in enumerate(p.unrank(n, range(Sk)).tolist())}
    edges = torch.zeros(Sp, m, dtype=torch.bool)
    for t, parent in enumerate(p.unrank(n - 1, range(Sp)).tolist()):
        for j in range(m):
            edges[t, j] = tuple(sorted([*parent, j])) in rows
    g = torch.ones(1, Sk, dtype=torch.complex64, device="cuda")
    for t in (0, Sp // 2, Sp - 1):                      # a parent's amplitude
        U = torch.ones(1, m, m, dtype=torch.complex64, device="cuda")
        psi = torch.ones(1, Sp, dtype=torch.complex64, device="cuda")
        psi[0, t] = bad
        gU = torch.zeros_like(U)
        p.adjoint_layer(U, n, 0, psi, g, gU)
        assert torch.equal(torch.isfinite(gU[0, :, 0].real).cpu(), ~edges[t])
    for j in (0, m - 1):                                # a coefficient
        U = torch.ones(1, m, m, dtype=torch.complex64, device="cuda")
        U[0, j, 0] = bad
        psi = torch.ones(1, Sp, dtype=torch.complex64, device="cuda")
        gp = p.adjoint_layer(U, n, 0, psi, g, torch.zeros_like(U))
        assert torch.equal(torch.isfinite(gp[0].real).cpu(), ~edges[:, j])
