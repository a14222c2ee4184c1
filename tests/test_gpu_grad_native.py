"""The one-call forward and backward (every layer kept) against the layer-by-layer path that
gradient_checkpointing selects: the same kernels on the same layers."""
import pytest
import torch
from helpers import haar_unitary

from photonic_engines_amd.slos import FockSLOSKernel

pytestmark = pytest.mark.gpu


# one photon up to layers of the group order; rows; several photons in a mode (a column with several
# layers' sums); every mask; more modes than the insert table's adjoint takes
@pytest.mark.parametrize("occ,mask,rows", [
    ([1], "fock", 0), ([0, 1, 0], "fock", 2), ([1, 1, 0, 0], "fock", 0), ([2, 0, 1, 0, 0], "fock", 3),
    ([1] * 6 + [0] * 10, "fock", 0), ([3, 0, 2, 1, 1, 0, 0, 0, 0], "fock", 2), ([1] * 8 + [0] * 16, "fock", 0),
    ([1, 0] * 5, "dual_rail", 2), ([1] * 6 + [0] * 8, "unbunched", 0), ([1, 0, 0, 0] * 3, "sparse_1in4", 0),
    ([1] * 7 + [0] * 6, "tail_empty", 2), ([1] * 3 + [0] * 60, "fock", 2), ([1] * 6 + [0] * 27, "fock", 0),
    ([9, 4], "fock", 0)])
@pytest.mark.parametrize("of", ["probs", "amplitudes"])
def test_one_call_gradients(occ, mask, rows, of):
    n, m = sum(occ), len(occ)
    U0 = haar_unitary(m, 3 * n + m).to(torch.complex64).cuda()
    if rows:
        U0 = torch.stack([haar_unitary(m, 3 * n + m + i).to(torch.complex64).cuda() for i in range(rows)])
    g = torch.Generator("cuda").manual_seed(n + 31 * m)
    res = []
    w = None
    for checkpointing in (False, True):
        k = FockSLOSKernel(n, m, occ, mask=mask, device="cuda", gradient_checkpointing=checkpointing)
        U = U0.clone().requires_grad_()
        out = getattr(k, of)(U)
        if w is None:
            w = torch.randn(out.shape, dtype=out.dtype, device="cuda", generator=g)
            w = torch.where(torch.rand(out.shape, device="cuda", generator=g) < 0.25, torch.zeros_like(w), w)
        (out * w).sum().real.backward()
        res.append((out.detach(), U.grad))
    assert torch.equal(res[0][0], res[1][0])
    # the sums over work groups are in FP64 in either order: one rounding to float32 a layer and one an
    # addition to a column
    scale = res[1][1].abs().amax(dim=(-2, -1), keepdim=True)
    assert ((res[0][1] - res[1][1]).abs() <= 2 * n * 2.0 ** -23 * scale).all()
