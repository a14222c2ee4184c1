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


FRONT = [(1, 5, "fock"), (2, 46, "fock"), (3, 17, "fock"), (3, 18, "fock"), (4, 12, "fock"), (6, 12, "fock"),
         (12, 3, "fock"), (17, 2, "fock"), (20, 1, "fock"), (5, 60, "unbunched"), (4, 22, "unbunched"), (6, 12, "dual_rail"),
         (4, 16, "sparse_1in4"), (5, 9, "tail_empty"), (2, 129, "fock"), (4, 130, "fock"), (2, 1500, "fock")]


@pytest.mark.parametrize("n,m,mask", FRONT)
def test_first_layers_in_one_launch_equal_the_thread_kernel(n, m, mask):
    """Layers up to 16, where the launch of the first layers ends at the latest, each as the forward's
    last one, with bunched and repeated input columns. (Beyond, the block and the thread kernel
    multiply the factorials of a bunched output, no longer whole floats, in another order.)"""
    occ = [n // m + (1 if j < n % m else 0) for j in range(m)] if n > m else occupation_list(n, m, mask)
    k = FockSLOSKernel(n, m, occ, mask=mask, device=DEV)
    cols = [(7 * i) % m for i in range(n)]
    U = torch.stack([haar_unitary(m, 70 + b) for b in range(3)]).to(DEV)
    layers = sorted({1, 2, 3, 4, 5, 6, 16, n - 1, n} & set(range(1, min(n, 16) + 1)))
    for g in layers:
        for kind in (nat.OUT_PROBS, nat.OUT_AMPS):
            for flags in (0, nat.FLAG_COMPENSATED, nat.FLAG_IMMEDIATE):
                Uc = U.to(torch.complex64).contiguous()
                a = k._plan.forward(Uc, modes=cols[:g], layer=g, out_kind=kind, scale=0.7, flags=flags)
                b = k._plan.forward(Uc, modes=cols[:g], layer=g, out_kind=kind, scale=0.7, flags=flags | nat.FLAG_SIMPLE)
                assert torch.equal(a, b), (g, kind, flags)
            a = k._plan.forward(U.contiguous(), modes=cols[:g], layer=g, out_kind=kind, scale=0.7)
            b = k._plan.forward(U.contiguous(), modes=cols[:g], layer=g, out_kind=kind, scale=0.7, flags=nat.FLAG_SIMPLE)
            # (the compiler may fuse the products of |amp|^2 differently in the two kernels)
            assert (a - b).abs().max() <= 4 * 2.0 ** -53 * b.abs().max(), (g, kind)
