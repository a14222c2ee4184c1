"""Batches of many small systems, which take other launches than a few rows do (a launch a layer in place of
the first layers' one, the loss's steps in place of its last layers' one, smaller work groups in the sum of
dL/dU): every row as run alone."""
import pytest
import torch

from photonic_engines_amd.slos import FockSLOSKernel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,m,mask,rows", [(1, 4, "fock", 600), (3, 6, "fock", 600), (4, 6, "fock", 300), (6, 9, "fock", 700), (3, 12, "sparse_1in4", 300),
                                           (5, 10, "dual_rail", 600), (5, 9, "tail_empty", 300), (4, 7, "unbunched", 600),
                                           (2, 130, "fock", 40), (11, 4, "fock", 6000), (8, 6, "fock", 1700)])
def test_rows_are_single_runs(n, m, mask, rows):
    step = {"dual_rail": 2, "sparse_1in4": 4}.get(mask, 1)
    me = m - 2 if mask == "tail_empty" else m
    occ = [0] * m
    for i in range(n):
        occ[step * i % me] += 1
    k = FockSLOSKernel(n, m, occ, mask=mask, device="cuda")
    g = torch.Generator("cuda").manual_seed(rows)
    U = torch.linalg.qr(torch.randn(rows, m, m, dtype=torch.complex64, device="cuda", generator=g))[0].contiguous()
    p = k.probs(U)
    q = k._plan.loss_thin(p, [0.75] * n)
    V = U.clone().requires_grad_()
    w = torch.rand(p.shape[1], device="cuda", generator=g)
    (k.probs(V) * w).sum().backward()
    for b in (0, 1, rows // 2, rows - 1):
        one = k.probs(U[b])
        assert torch.equal(p[b], one), b
        for a, c in zip(q, k._plan.loss_thin(one.unsqueeze(0), [0.75] * n), strict=True):
            assert torch.equal(a[b], c[0]), b
        v = U[b].clone().requires_grad_()
        (k.probs(v) * w).sum().backward()
        # (other kernels and work groups: sums in FP64 or of at most m + n terms in float32 a layer)
        assert ((V.grad[b] - v.grad).abs() <= (m + n) * n * 2.0 ** -23 * v.grad.abs().max()).all(), b
