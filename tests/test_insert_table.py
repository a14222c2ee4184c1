"""The insert table of the pulls over children: the child of a parent and a mode at or above the
parent's last prefix position, and its copies, from one table word."""
import ctypes

import pytest
import torch
from test_emulator import emu, pull  # noqa: F401  (the compiled emulator, a fixture)

from photonic_engines_amd import _native as nat
from photonic_engines_amd.slos import FockSLOSKernel


@pytest.mark.parametrize("n,m,mask,k,first", [(6, 1, "fock", 6, 0), (6, 5, "fock", 6, 0), (8, 9, "fock", 8, 0),
                                              (9, 7, "tail_empty", 9, 0), (13, 5, "fock", 13, 0), (7, 41, "fock", 7, 0),
                                              (7, 41, "fock", 7, 7_000_000), (11, 32, "fock", 11, 560549704),
                                              (11, 32, "fock", 11, 1121099408 - 200000)])
def test_insert_table_children(emu, n, m, mask, k, first):  # noqa: F811
    emu.emu_check_insert.restype = ctypes.c_int64
    emu.emu_check_insert.argtypes = [ctypes.c_int] * 4 + [ctypes.c_uint64] * 2
    assert emu.emu_check_insert(n, m, pull.MASK_IDS[mask], k, first, 200_000) == 0


@pytest.mark.parametrize("n,m,mask", [(1, 1, "fock"), (2, 3, "fock"), (4, 64, "fock"), (5, 9, "tail_empty"), (4, 64, "unbunched"),
                                      (3, 3, "unbunched"), (6, 24, "dual_rail"), (4, 40, "sparse_1in4"), (8, 12, "fock")])
def test_binary_search_for_positions(emu, n, m, mask):  # noqa: F811
    emu.emu_check_unrank_search.restype = ctypes.c_int64
    emu.emu_check_unrank_search.argtypes = [ctypes.c_int] * 4 + [ctypes.c_uint64] * 2
    for k in range(1, n + 1):
        assert emu.emu_check_unrank_search(n, m, pull.MASK_IDS[mask], k, 100_000, 997) == 0


def _plan(n, m, mask):
    modes = m - 2 if mask == "tail_empty" else m
    step = {"dual_rail": 2, "sparse_1in4": 4}.get(mask, 1)
    occ = [0] * m
    for i in range(n):
        occ[step * i % modes] += 1
    return FockSLOSKernel(n, m, occ, mask=mask, device="cuda")._plan


# (n, m, mask, rows): parent prefixes of 0 to 8 positions, blocks of one parent up to the longest, the
# largest mode count of the table, several rows, and the thread-per-state side of the rule
@pytest.mark.gpu
@pytest.mark.parametrize("n,m,mask,rows", [(5, 41, "fock", 1), (5, 9, "fock", 3), (6, 41, "fock", 1), (7, 12, "fock", 200), (8, 24, "fock", 1),
                                           (9, 18, "tail_empty", 3), (10, 21, "fock", 1), (11, 17, "fock", 1),
                                           (12, 16, "fock", 1), (13, 16, "fock", 1), (9, 9, "fock", 2)])
def test_descents_equal_the_thread_kernel(n, m, mask, rows):
    plan = _plan(n, m, mask)
    q = torch.rand((rows, plan.sizes[n]), device="cuda", generator=torch.Generator("cuda").manual_seed(n * m))
    for k in range(n, 4, -1):
        out = plan.loss_descend(k, q, scale=0.75)
        assert torch.equal(out, plan.loss_descend(k, q, flags=nat.FLAG_SIMPLE, scale=0.75)), k
        q = out


# parent prefixes of 1 to 8 positions on both sides of 16 modes; every parent in the last eight modes;
# a last step of the walk of one parent; the layers of at most five parent photons by a lane a mode, in
# groups of 32 and 64 lanes, and thread per state with many rows; masks with inadmissible children
@pytest.mark.gpu
@pytest.mark.parametrize("n,m,mask,rows", [(5, 33, "fock", 1), (5, 32, "fock", 4), (4, 64, "fock", 2), (6, 8, "fock", 200), (5, 7, "fock", 1200),
                                           (6, 14, "unbunched", 2), (5, 40, "dual_rail", 1), (4, 24, "sparse_1in4", 3),
                                           (1, 1, "fock", 1), (2, 6, "tail_empty", 4), (6, 32, "fock", 1), (7, 16, "fock", 3), (8, 17, "tail_empty", 1),
                                           (8, 24, "fock", 1), (9, 9, "fock", 2), (10, 12, "fock", 1),
                                           (13, 4, "fock", 5), (13, 9, "fock", 1)])
def test_adjoint_against_complex128(n, m, mask, rows):
    """One adjoint layer against the complex128 kernel on random layers. A term of grad_prev is one of
    2 me fused products a component, one of dL/dU a product in float32 sums of at most 2 x 8 parents a
    lane or thread (FP64 beyond): errors within these counts, and two roundings, times the sums of magnitudes."""
    plan = _plan(n, m, mask)
    me = m - 2 if mask == "tail_empty" else m
    g = torch.Generator("cuda").manual_seed(17 * n + m)

    def rand(*shape):
        return torch.randn(shape, dtype=torch.complex64, device="cuda", generator=g)

    U = rand(rows, m, m)
    for k in range(n, 0, -1):
        psi, gk, col = rand(rows, plan.sizes[k - 1]), rand(rows, plan.sizes[k]), k % m
        gU, ref_U, mag_U = torch.zeros_like(U), *(torch.zeros_like(U, dtype=torch.complex128) for _ in range(2))
        out = plan.adjoint_layer(U, k, col, psi, gk, gU)
        wide = [x.to(torch.complex128) for x in (U, psi, gk)]
        ref = plan.adjoint_layer(wide[0], k, col, wide[1], wide[2], ref_U)
        size = [x.abs().to(torch.complex128) for x in wide]
        mag = plan.adjoint_layer(size[0], k, col, size[1], size[2], mag_U)
        eps = 2.0 ** -24 * 2 ** 0.5
        assert ((out - ref).abs() <= (2 * me + 2) * eps * mag.real).all(), k
        assert ((gU - ref_U).abs() <= (2 * 8 + 2) * eps * mag_U.real).all(), k


# every step in one call: steps of the walk and thread per state, then the last layers in one launch: from
# layer n on; from a layer of few states below larger ones; masks; nothing below the table's layers
@pytest.mark.gpu
@pytest.mark.parametrize("n,m,mask,rows", [(1, 1, "fock", 1), (3, 12, "fock", 5), (6, 24, "fock", 2), (9, 5, "fock", 1),
                                           (5, 64, "fock", 1), (12, 3, "fock", 3), (6, 20, "unbunched", 2),
                                           (8, 16, "dual_rail", 1), (7, 14, "tail_empty", 4), (5, 24, "sparse_1in4", 1)])
def test_all_descents_in_one_call(n, m, mask, rows):
    plan = _plan(n, m, mask)
    q = torch.rand((rows, plan.sizes[n]), device="cuda", generator=torch.Generator("cuda").manual_seed(n + m))
    scale = [0.5 + 0.05 * k for k in range(n)]
    out = plan.loss_thin(q, scale)
    assert len(out) == n
    for k in range(n, 0, -1):
        q = plan.loss_descend(k, q, flags=nat.FLAG_SIMPLE, scale=scale[k - 1])
        assert torch.equal(out[k - 1], q), k
