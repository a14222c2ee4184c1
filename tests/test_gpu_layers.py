"""The layer launches where their work split can go wrong: rows of a batch placed on the XCDs (whole
eights of rows and the rows left over), pairs of adjacent children with remainders of the pair step.
Every form of a layer sums its parents in the same order, so rows and kernels are compared bit for
bit."""
import pytest
import torch
from helpers import haar_unitary, occupation_list

from photonic_engines_amd import _native as nat
from photonic_engines_amd.slos import FockSLOSKernel

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("B", [7, 8, 9, 17])
@pytest.mark.parametrize("n,m,mask", [(8, 9, "fock"), (7, 14, "unbunched"), (5, 8, "fock")])
def test_rows_of_a_batch_are_single_runs(n, m, mask, B):
    U = torch.stack([haar_unitary(m, 900 + b) for b in range(B)]).to(torch.complex64).to(DEV)
    for comp in (False, True):
        k = FockSLOSKernel(n, m, occupation_list(n, m, mask), mask=mask, device=DEV, compensated=comp)
        p = k.probs(U)
        a = k.amplitudes(U)
        for b in range(B):
            assert torch.equal(p[b], k.probs(U[b])), b
            assert torch.equal(a[b], k.amplitudes(U[b])), b


@pytest.mark.parametrize("m", [1, 2, 3, 6, 13])
@pytest.mark.parametrize("n", [7, 8, 11])
def test_pairs_of_children_equal_the_thread_kernel(n, m):
    if n == 11 and m == 13:
        m = 12
    occ = [n // m + (1 if j < n % m else 0) for j in range(m)]
    U = haar_unitary(m, 40 + m).to(torch.complex64).to(DEV).unsqueeze(0).contiguous()
    for flags in (0, nat.FLAG_COMPENSATED):
        k = FockSLOSKernel(n, m, occ, device=DEV)
        for kind in (nat.OUT_PROBS, nat.OUT_AMPS):
            a = k._plan.forward(U, out_kind=kind, flags=flags)
            b = k._plan.forward(U, out_kind=kind, flags=flags | nat.FLAG_SIMPLE)
            assert torch.equal(a, b), (flags, kind)
