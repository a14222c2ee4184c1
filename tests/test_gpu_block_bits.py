"""The block and group-order kernels, forced on every layer they can take (SLOS_FLAG_BLOCK; by themselves
they run on layers of millions of states), against the thread-per-state kernel bit for bit: both sum a
child's parents in ascending photon position."""
import pytest
import torch
from helpers import haar_unitary, occupation_list
from test_gpu_strides import _views

from photonic_engines_amd import _native as nat
from photonic_engines_amd.slos import FockSLOSKernel

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _kernel(n, m, mask, **options):
    occ = [n // m + (1 if j < n % m else 0) for j in range(m)] if n > m else occupation_list(n, m, mask)
    return FockSLOSKernel(n, m, occ, mask=mask, device=DEV, **options)


def _matrices(m, rows, dtype=torch.complex64):
    return torch.stack([haar_unitary(m, 40 + m + b) for b in range(rows)]).to(dtype).to(DEV)


# the shapes of the block kernel's own cases: every mask, 4- and 5-position suffixes, every prefix width (and
# stream-slot count), 64 modes; then pairs of children with remainders of the pair step, from one mode on
SHAPES = [(9, 14, "fock"), (8, 16, "fock"), (7, 18, "tail_empty"), (6, 24, "unbunched"), (10, 9, "fock"), (9, 5, "fock"), (10, 5, "fock"),
          (11, 4, "fock"), (12, 4, "fock"), (13, 3, "fock"), (13, 9, "fock"), (16, 4, "fock"), (20, 3, "fock"), (9, 12, "unbunched"), (10, 20, "dual_rail"), (5, 20, "sparse_1in4"),
          (5, 60, "unbunched"), (5, 64, "fock"), (6, 40, "unbunched"), (6, 30, "fock")]
SHAPES += [(n, 12 if (n, m) == (11, 13) else m, "fock") for n in (7, 8, 11) for m in (1, 2, 3, 6, 13)]


@pytest.mark.parametrize("n,m,mask", SHAPES)
def test_blocks_equal_threads(n, m, mask):
    k = _kernel(n, m, mask)
    U = _matrices(m, 2)
    for flags in (0, nat.FLAG_COMPENSATED, nat.FLAG_IMMEDIATE):
        for kind in (nat.OUT_PROBS, nat.OUT_AMPS):
            # (from 14 photons in a mode on prod t! is no whole float, and the two multiply it in another order)
            if n > 13 and mask == "fock" and (kind == nat.OUT_PROBS or flags == nat.FLAG_IMMEDIATE):
                continue
            a = k._plan.forward(U, out_kind=kind, scale=0.7, flags=flags | nat.FLAG_BLOCK)
            b = k._plan.forward(U, out_kind=kind, scale=0.7, flags=flags | nat.FLAG_SIMPLE)
            assert torch.equal(a, b), (flags, kind)


@pytest.mark.parametrize("n,m,mask", [s for s in SHAPES if s[0] <= 13])
def test_complex128_blocks_equal_threads(n, m, mask):
    k = _kernel(n, m, mask, dtype=torch.complex128)
    U = _matrices(m, 2, torch.complex128)
    for flags in (0, nat.FLAG_IMMEDIATE):
        a = k._plan.forward(U, out_kind=nat.OUT_AMPS, scale=0.7, flags=flags | nat.FLAG_BLOCK)
        b = k._plan.forward(U, out_kind=nat.OUT_AMPS, scale=0.7, flags=flags | nat.FLAG_SIMPLE)
        assert torch.equal(a, b), flags
    a = k._plan.forward(U, scale=0.7, flags=nat.FLAG_BLOCK)
    b = k._plan.forward(U, scale=0.7, flags=nat.FLAG_SIMPLE)
    # (|amp|^2: the compiler may fuse one of its products into the sum in either kernel, one rounding of two
    # that are at most |amp|^2 together; then one rounding by prod t!)
    assert ((a - b).abs() <= 4 * 2.0 ** -53 * b).all()


# rows on the XCDs: whole eights of them, and the rows left over
@pytest.mark.parametrize("B", [7, 8, 9, 17])
@pytest.mark.parametrize("n,m,mask,options", [(8, 9, "fock", {}), (7, 14, "unbunched", {}), (6, 20, "fock", {}), (5, 8, "fock", {}),
                                              (8, 9, "fock", {"dtype": torch.complex128}), (7, 14, "unbunched", {"dtype": torch.complex128})])
def test_rows_of_a_batch_are_single_runs(n, m, mask, options, B):
    k = _kernel(n, m, mask, **options)
    U = _matrices(m, B, k.cdtype)
    for flags in (0,) if options else (0, nat.FLAG_COMPENSATED):
        a = k._plan.forward(U, out_kind=nat.OUT_AMPS, flags=flags | nat.FLAG_BLOCK)
        for b in range(B):
            one = k._plan.forward(U[b:b + 1], out_kind=nat.OUT_AMPS, flags=flags | nat.FLAG_SIMPLE)
            assert torch.equal(a[b], one[0]), (flags, b)


@pytest.mark.parametrize("n,m,mask,options", [(8, 12, "fock", {}), (6, 18, "fock", {}), (7, 16, "unbunched", {}), (6, 12, "dual_rail", {}),
                                              (7, 14, "tail_empty", {}), (8, 12, "fock", {"dtype": torch.complex128}),
                                              (7, 16, "unbunched", {"dtype": torch.complex128})])
def test_strided_matrices(n, m, mask, options):
    k = _kernel(n, m, mask, **options)
    for name, U in _views(m, k.cdtype).items():
        if U.is_conj():
            continue
        p = k._plan.probs(U, 1.0, nat.FLAG_BLOCK)
        packed = U.clone(memory_format=torch.contiguous_format)
        q = k._plan.forward(packed if U.dim() == 3 else packed.unsqueeze(0), flags=nat.FLAG_BLOCK)
        assert torch.equal(p, q if U.dim() == 3 else q[0]), name


def test_one_call_gradient_of_a_set_mask_on_blocks():
    """The readout's adjoint in the block kernel (10.7M states, blocks of 1.5M on average; by size alone)."""
    n, m = 6, 47
    grads = []
    for checkpointing in (False, True):
        k = _kernel(n, m, "unbunched", gradient_checkpointing=checkpointing)
        U = haar_unitary(m, 5).to(torch.complex64).to(DEV).requires_grad_()
        p = k.probs(U)
        (p * (torch.arange(p.numel(), device=DEV) % 7)).sum().backward()
        grads.append(U.grad)
    # (FP64 sums over the work groups in either order: one rounding to float32 a layer, one an addition)
    assert ((grads[0] - grads[1]).abs() <= 2 * n * 2.0 ** -23 * grads[1].abs().max()).all()


def test_long_runs_of_prefixes_without_children():
    """sparse_1in4: of 473,088 prefixes of layer 10 of 11 photons in 44 modes 6,144 have children."""
    k = FockSLOSKernel(11, 44, [1, 0, 0, 0] * 11, mask="sparse_1in4", device=DEV)
    U = _matrices(44, 1)
    for layer in (9, 10, 11):
        for flags in (0, nat.FLAG_COMPENSATED):
            a = k._plan.forward(U, layer=layer, modes=k.input_modes[:layer], flags=flags | nat.FLAG_BLOCK)
            b = k._plan.forward(U, layer=layer, modes=k.input_modes[:layer], flags=flags | nat.FLAG_SIMPLE)
            assert torch.equal(a, b), (layer, flags)


@pytest.mark.parametrize("n,m,mask,dtype", [(8, 26, "fock", torch.complex64), (9, 29, "unbunched", torch.complex64), (8, 24, "fock", torch.complex128)])
def test_rows_of_wide_layers_equal_single_matrices(n, m, mask, dtype):
    """9 rows whose last layers' parents are above the 24 MiB a row up to which whole rows go to one XCD,
    and whose first layers' are below it."""
    k = _kernel(n, m, mask, dtype=dtype)
    U = _matrices(m, 9, dtype)
    p = k._plan.forward(U, out_kind=nat.OUT_PROBS, flags=nat.FLAG_BLOCK)
    for b in (0, 7, 8):
        assert torch.equal(p[b], k._plan.forward(U[b:b + 1], out_kind=nat.OUT_PROBS, flags=nat.FLAG_BLOCK)[0]), b
