"""Timed cases of the strong-simulation engine: what its users have it compute, from one small
matrix to the frontier size, through the public entry points (`FockSLOSKernel.probs` with its
options, autograd through it, and `UnevenBatch.probs`).

`listed()` names the cases, `draw(rng)` gives others of the same ranges, `prepare` makes a case's
inputs and kernels, `run` is one call, `work` its compulsory bytes and operations, and `exact` the
same outputs in 64 bits by plain torch.
"""
from __future__ import annotations

import math
from itertools import combinations

import torch

from photonic_engines_amd.slos import FockSLOSKernel, UnevenBatch

DEV = "cuda"


# ------------------------------------------------------------------------------------------------
# the cases
# ------------------------------------------------------------------------------------------------

def _case(kind: str, n: int, m: int, **more) -> dict:
    """A case with every option of its kind written out. `input`: the photons in the first modes,
    in every other mode, or two to a mode from mode 0 on. `compensated`: compensated sums.
    `loss`, `indist`, `order`: the arguments of probs."""
    c = {"kind": kind, "n": n, "m": m, "mask": "fock", "input": "first", "dtype": "complex64", "batch": 0,
         "compensated": False}
    c.update(more)
    return c


def listed() -> list[dict]:
    def named(name, c):
        return {"name": name, **c}

    return [
        # a few photons on a small chip, one matrix at a time: the interactive and optimiser-loop call,
        # a matter of launches and host time
        named("probs_n4_m12", _case("probs", 4, 12)),
        # six photons in alternate modes (a table's ordinary row)
        named("probs_n6_m18", _case("probs", 6, 18, input="alternate")),
        # the ordinary full distribution of an experiment of today
        named("probs_n8_m24", _case("probs", 8, 24)),
        # the frontier size, 4.28e9 outputs
        named("probs_n11_m32", _case("probs", 11, 32)),
        # reference-quality output: every layer in complex128
        named("complex128_n10_m20", _case("probs", 10, 20, dtype="complex128")),
        # compensated complex64 sums, the accuracy option between the two
        named("compensated_n9_m22", _case("probs", 9, 22, compensated=True)),
        # collision-free outputs only (threshold detectors, post-selected)
        named("unbunched_n9_m26", _case("probs", 9, 26, mask="unbunched")),
        # 512 unitaries of three shapes in one call (a dataset of circuits)
        named("uneven_512", {"kind": "uneven", "shapes": "4x12x171,6x16x171,8x20x170"}),
        # the lossy output of a real source: every photon number 0..n
        named("lossy_n10_m24", _case("lossy", 10, 24, loss=0.9)),
        # a training step on sampled data: -mean log p over 1,024 outputs, with its gradient
        named("grad_sampled_n6_m16", _case("grad", 6, 16, objective="sampled")),
        # a variational step: the mean of a diagonal observable, dL/dp nonzero everywhere
        named("grad_observable_n8_m24", _case("grad", 8, 24, objective="observable")),
        # partially distinguishable photons, all interfering subsets
        named("xmodel_n8_m24", _case("xmodel", 8, 24, indist=0.9, order=None)),
    ]


def _size(n: int, m: int, mask: str) -> int:
    if mask == "fock":
        return math.comb(m + n - 1, n)
    if mask == "tail_empty":
        return math.comb(m - 2 + n - 1, n)
    if mask == "unbunched":
        return math.comb(m, n)
    b = 2 if mask == "dual_rail" else 4
    return math.comb(m // b, n) * b ** n


def _draw_m(rng, n: int, mask: str, low: float, high: float) -> int | None:
    """A mode count whose distribution has a size spread over the logarithm of [low, high]."""
    step = {"dual_rail": 2, "sparse_1in4": 4}.get(mask, 1)
    target = math.exp(rng.uniform(math.log(low), math.log(high)))
    fits = [m for m in range(max(2, n * step) + (2 if mask == "tail_empty" else 0), 65, step)
            if low <= _size(n, m, mask) <= high]
    return min(fits, key=lambda m: abs(math.log(_size(n, m, mask) / target))) if fits else None


def draw(rng) -> dict:
    while True:
        kind = rng.choice(["probs", "probs", "probs", "complex128", "compensated", "batch", "uneven", "lossy", "grad",
                           "grad", "xmodel"])
        if kind == "uneven":
            shapes = []
            for _ in range(rng.randint(2, 4)):
                n = rng.randint(3, 8)
                m = _draw_m(rng, n, "fock", 200, 3e6)
                if m is not None:
                    b = round(math.exp(rng.uniform(math.log(2), math.log(200))))
                    shapes.append((n, m, max(1, min(b, int(2e8 // _size(n, m, "fock"))))))
            if len(shapes) >= 2:
                return {"kind": "uneven", "shapes": ",".join("%dx%dx%d" % s for s in shapes)}
            continue
        mask = rng.choice(["fock"] * 6 + ["unbunched", "dual_rail", "tail_empty"])
        if kind in ("grad", "xmodel"):
            mask = "fock"
        n = rng.randint(*{"probs": (3, 12), "complex128": (3, 11), "compensated": (4, 10), "batch": (3, 8),
                          "lossy": (3, 10), "grad": (3, 9), "xmodel": (3, 8)}[kind])
        high = {"probs": 4e8, "complex128": 1e8, "compensated": 1e8, "batch": 3e6, "lossy": 1e8, "grad": 2e7,
                "xmodel": 6e6}[kind]
        m = _draw_m(rng, n, mask, 300, high)
        if m is None:
            continue
        more = {"mask": mask}
        if mask == "fock":
            more["input"] = rng.choice(["first", "first", "alternate", "pairs"])
            if more["input"] == "alternate" and 2 * n > m:
                more["input"] = "first"
        if kind == "probs":
            return _case("probs", n, m, **more)
        if kind == "complex128":
            return _case("probs", n, m, dtype="complex128", **more)
        if kind == "compensated":
            return _case("probs", n, m, compensated=True, **more)
        if kind == "batch":
            b = round(math.exp(rng.uniform(math.log(2), math.log(256))))
            return _case("probs", n, m, batch=max(1, min(b, int(2e8 // _size(n, m, mask)))), **more)
        if kind == "lossy":
            return _case("lossy", n, m, loss=round(rng.uniform(0.3, 0.97), 3), **more)
        if kind == "grad":
            return _case("grad", n, m, objective=rng.choice(["sampled", "observable"]), **more)
        return _case("xmodel", n, m, indist=round(rng.uniform(0.6, 0.99), 3), order=rng.choice([None, None, 1, 2, 3]), **more)


# ------------------------------------------------------------------------------------------------
# inputs and calls
# ------------------------------------------------------------------------------------------------

def _haar(m: int, seed: int, count: int) -> torch.Tensor:
    """Haar-random unitaries [count, m, m] in complex128 on the host."""
    g = torch.Generator().manual_seed(seed)
    z = torch.complex(torch.randn(count, m, m, generator=g, dtype=torch.float64),
                      torch.randn(count, m, m, generator=g, dtype=torch.float64))
    q, r = torch.linalg.qr(z)
    d = torch.diagonal(r, dim1=-2, dim2=-1)
    return q * (d / d.abs()).unsqueeze(-2)


def _occupation(c: dict) -> list[int]:
    n, m = c["n"], c["m"]
    occ = [0] * m
    if c["mask"] in ("dual_rail", "sparse_1in4"):
        step = 2 if c["mask"] == "dual_rail" else 4
        at = [step * i for i in range(n)]
    elif c["input"] == "alternate":
        at = [2 * i for i in range(n)]
    elif c["input"] == "pairs":
        at = [i // 2 for i in range(n)]
    else:
        at = list(range(n))
    for j in at:
        occ[j] += 1
    return occ


def _shapes(c: dict) -> list[tuple[int, int, int]]:
    return [tuple(int(v) for v in s.split("x")) for s in c["shapes"].split(",")]


def _unitaries(c: dict, seed: int):
    """The case's unitaries on the GPU in its dtype (a list of batches for the uneven batch)."""
    if c["kind"] == "uneven":
        return [_haar(m, seed * 1009 + i, b).to(torch.complex64).to(DEV) for i, (_, m, b) in enumerate(_shapes(c))]
    U = _haar(c["m"], seed, max(1, c["batch"])).to(getattr(torch, c["dtype"])).to(DEV)
    return U if c["batch"] else U[0]


def _observable(c: dict, seed: int) -> torch.Tensor:
    """A diagonal observable's value on every output, in [-1, 1]."""
    g = torch.Generator(device=DEV).manual_seed(seed + 77)
    return torch.rand(_size(c["n"], c["m"], c["mask"]), generator=g, device=DEV) * 2 - 1


def _samples(c: dict, seed: int) -> torch.Tensor:
    """A training set: 1,024 outputs of another matrix, the one to be learnt (the quantiles
    (i + u) / 1024 of its distribution's cumulative sum)."""
    target = _haar(c["m"], seed + 40, 1).to(DEV)
    columns = [j for j, k in enumerate(_occupation(c)) for _ in range(k)]
    p = _exact_probs(_Space(c["n"], c["m"], c["mask"]), target, columns)[0]
    g = torch.Generator().manual_seed(seed + 78)
    at = (torch.arange(1024, dtype=torch.float64) + torch.rand(1024, generator=g, dtype=torch.float64)) / 1024
    cdf = torch.cumsum(p, 0)
    return torch.searchsorted(cdf, at.to(p.device) * cdf[-1]).clamp_(max=p.numel() - 1)


def prepare(case: dict, seed: int) -> dict:
    U = _unitaries(case, seed)
    if case["kind"] == "uneven":
        kernels = [FockSLOSKernel(n, m, [1] * n + [0] * (m - n), device=DEV) for n, m, _ in _shapes(case)]
        return {"kind": "uneven", "U": U, "kernel": UnevenBatch(kernels), "kernels": kernels}
    k = FockSLOSKernel(case["n"], case["m"], _occupation(case), mask=case["mask"], device=DEV,
                       dtype=getattr(torch, case["dtype"]), compensated=case["compensated"])
    s = {"kind": case["kind"], "U": U, "kernel": k}
    if case["kind"] == "lossy":
        s["loss"] = case["loss"]
    elif case["kind"] == "xmodel":
        s["indist"], s["order"] = case["indist"], case["order"]
    elif case["kind"] == "grad":
        if case["objective"] == "sampled":
            s["index"] = _samples(case, seed)
        else:
            s["weight"] = _observable(case, seed)
    return s


def run(state: dict):
    k, U = state["kernel"], state["U"]
    kind = state["kind"]
    if kind == "probs" or kind == "uneven":
        return k.probs(U)
    if kind == "lossy":
        return k.probs(U, loss=state["loss"]).probs
    if kind == "xmodel":
        return k.probs(U, indist=state["indist"], order=state["order"])
    U = U.detach().requires_grad_(True)
    p = k.probs(U)
    if "index" in state:
        loss = -torch.log(p[state["index"]]).mean()
    else:
        loss = (p * state["weight"]).sum()
    loss.backward()
    return {"probs": p.detach(), "loss": loss.detach(), "grad": U.grad}


# ------------------------------------------------------------------------------------------------
# compulsory work
# ------------------------------------------------------------------------------------------------

def _forward_work(n: int, m: int, mask: str, amp: int) -> tuple[float, float]:
    """Every layer written once and read once (`amp` bytes an amplitude, half that a probability), and
    a complex multiply-add for every (state, photon that can be taken away)."""
    S = [_size(k, m, mask) for k in range(n + 1)]
    bytes_ = sum(amp * S[k - 1] for k in range(1, n + 1)) + sum(amp * S[k] for k in range(1, n)) + amp // 2 * S[n]
    if mask in ("fock", "tail_empty"):
        edges = sum(S[k - 1] * (m - 2 if mask == "tail_empty" else m) for k in range(1, n + 1))
    else:
        edges = sum(S[k] * k for k in range(1, n + 1))
    return float(bytes_), 8.0 * edges


def work(case: dict) -> dict:
    if case["kind"] == "uneven":
        each = [(b, _forward_work(n, m, "fock", 8)) for n, m, b in _shapes(case)]
        return {"bytes": sum(b * w[0] for b, w in each), "flops": sum(b * w[1] for b, w in each)}
    n, m, mask = case["n"], case["m"], case["mask"]
    nbytes, flops = _forward_work(n, m, mask, 16 if case["dtype"] == "complex128" else 8)
    S = [_size(k, m, mask) for k in range(n + 1)]
    if case["kind"] == "lossy":
        # each photon number's block from the one above: read, written
        nbytes += sum(4.0 * (S[k] + S[k - 1]) for k in range(1, n + 1))
        flops += 2.0 / 8.0 * flops
    elif case["kind"] == "grad":
        # the layers backwards: the gradient of layer k and layer k-1 itself read, its gradient written
        nbytes += 4.0 * S[n] + sum(8.0 * (S[k] + 2 * S[k - 1]) for k in range(1, n + 1))
        flops *= 3.0
    elif case["kind"] == "xmodel":
        # every set of distinguishable photons once: its distribution (and, if it interferes, its
        # amplitudes) written and read; one real multiply-add an edge to raise it
        b = n if case["order"] is None else case["order"]
        nbytes = 4.0 * S[n]
        flops = 0.0
        for L in range(0, n + 1):
            if L <= b or L < n:
                sets = math.comb(n, L)
                nbytes += sets * 2 * 4.0 * S[n - L] * (1 if L else 0)
                flops += sets * 2.0 * m * S[n - L] * (1 if L else 0)
            if L <= b and n - L >= 2:
                w = _forward_work(n - L, m, mask, 8)
                nbytes += math.comb(n, L) * w[0]
                flops += math.comb(n, L) * w[1]
    rows = max(1, case["batch"])
    return {"bytes": rows * nbytes, "flops": rows * flops}


# ------------------------------------------------------------------------------------------------
# the same outputs in 64 bits, by plain torch
# ------------------------------------------------------------------------------------------------

class _Space:
    """The sorted position tuples of a mask in lexicographic order. count[r][x]: how many sorted
    r-tuples begin at a position >= x; after[x]: the smallest position that may follow x."""

    def __init__(self, n: int, m: int, mask: str):
        self.size = m - 2 if mask == "tail_empty" else m
        width = {"unbunched": 1, "dual_rail": 2, "sparse_1in4": 4}.get(mask, 0)
        after = [min(self.size, (x // width + 1) * width) if width else x for x in range(self.size)]
        count = [[1] * (self.size + 1)]
        for _ in range(n):
            row = [0] * (self.size + 1)
            for x in range(self.size - 1, -1, -1):
                row[x] = row[x + 1] + count[-1][after[x]]
            count.append(row)
        self.sizes = [r[0] for r in count]
        self.repeats = width == 0
        self.after = torch.tensor(after + [self.size], device=DEV)
        self.count = [torch.tensor(r, device=DEV) for r in count]
        self.ascending = [r.flip(0).contiguous() for r in self.count]

    def tuples(self, k: int, begin: int, end: int) -> list[torch.Tensor]:
        """The k positions of the k-tuples begin..end-1."""
        left = torch.arange(begin, end, device=DEV)
        low = torch.zeros_like(left)
        at = []
        for i in range(k):
            c = self.count[k - i]
            behind = c[low] - left                    # tuples from this one on, among those >= low here
            x = self.size - torch.searchsorted(self.ascending[k - i], behind)
            left = c[x] - behind
            at.append(x)
            low = self.after[x]
        return at

    def parents(self, at: list[torch.Tensor]):
        """(index of the tuple without photon l, its mode, whether it counts) for every photon l."""
        k = len(at)
        low = [torch.zeros_like(at[0])] + [self.after[x] for x in at[:-1]]
        tail = [None] * (k + 2)
        tail[k] = tail[k + 1] = torch.zeros_like(at[0])
        for i in range(k - 1, 0, -1):
            c = self.count[k - i]
            tail[i] = tail[i + 1] + c[low[i]] - c[at[i]]
        head = torch.zeros_like(at[0])
        for i in range(k):
            c = self.count[k - 1 - i]
            index = head if i == k - 1 else head + c[low[i]] - c[at[i + 1]] + tail[i + 2]
            keep = None if i == 0 or not self.repeats else at[i] != at[i - 1]
            yield index, at[i], keep
            if i < k - 1:
                head = head + c[low[i]] - c[at[i]]

    def factorials(self, at: list[torch.Tensor]) -> torch.Tensor:
        """The product of the occupations' factorials."""
        run = torch.ones_like(at[0], dtype=torch.float64)
        f = run.clone()
        for i in range(1, len(at)):
            run = torch.where(at[i] == at[i - 1], run + 1, torch.ones_like(run))
            f = f * run
        return f


def _raised(space: _Space, k: int, column: torch.Tensor, lower: torch.Tensor, finish=None) -> torch.Tensor:
    """Layer k [R, S_k] from layer k-1 [R, S_(k-1)] and the coefficient columns [R, m]; `finish` of a
    range's values and positions is kept in their place."""
    R, S = lower.shape[0], space.sizes[k]
    chunk = max(1 << 16, (1 << 24) // R)
    parts = []
    out = None
    for a in range(0, S, chunk):
        b = min(S, a + chunk)
        at = space.tuples(k, a, b)
        acc = 0
        for index, mode, keep in space.parents(at):
            term = column[:, mode] * lower[:, index]
            acc = acc + (term if keep is None else term * keep)
        acc = finish(acc, at) if finish else acc
        if acc.requires_grad:
            parts.append(acc)
        else:
            if out is None:
                out = torch.empty(R, S, dtype=acc.dtype, device=DEV)
            out[:, a:b] = acc
    return torch.cat(parts, 1) if parts else out


def _exact_probs(space: _Space, U: torch.Tensor, columns: list[int]) -> torch.Tensor:
    """Probabilities [B, S] of the photons in `columns`, U [B, m, m] in complex128."""
    norm = 1.0
    for c in set(columns):
        norm /= math.factorial(columns.count(c))
    psi = torch.ones(U.shape[0], 1, dtype=torch.complex128, device=DEV)

    def readout(amp, at):
        return (amp.real ** 2 + amp.imag ** 2) * (norm * space.factorials(at) if space.repeats else norm)

    for k, c in enumerate(columns, 1):
        psi = _raised(space, k, U[:, :, c], psi, readout if k == len(columns) else None)
    return psi


def _exact_xmodel(space: _Space, U: torch.Tensor, columns: list[int], x: float, order) -> torch.Tensor:
    """The mixture over the interfering subsets: a distinguishable photon enters by the classical
    transport |U[j, c]|^2. waiting[T]: what is still to be raised by the photons T."""
    n = len(columns)
    most = n if order is None else order
    waiting: dict = {}

    def add(T, q):
        waiting[T] = waiting[T] + q if T in waiting else q

    for L in range(n, -1, -1):
        if L <= most:
            for T in combinations(range(n), L):
                good = [columns[i] for i in range(n) if i not in T]
                q = _exact_probs(space, U, good) if good else torch.ones(1, 1, dtype=torch.float64, device=DEV)
                add(T, q * (x ** (n - L) * (1 - x) ** L))
        sets = [T for T in waiting if len(T) == L and L]
        for i in range(0, len(sets), 16):
            some = sets[i:i + 16]
            w = torch.cat([U[:, :, columns[T[0]]].abs() ** 2 for T in some])
            up = _raised(space, n - L + 1, w, torch.cat([waiting.pop(T) for T in some]))
            for r, T in enumerate(some):
                add(T[1:], up[r:r + 1])
    return waiting[()]


def exact(case: dict, seed: int):
    U = _unitaries(case, seed)
    if case["kind"] == "uneven":
        out = []
        for (n, m, _), u in zip(_shapes(case), U):
            space = _Space(n, m, "fock")
            out.append(torch.cat([_exact_probs(space, u[i:i + 16].to(torch.complex128), list(range(n)))
                                  for i in range(0, u.shape[0], 16)]))
        return out
    n, m = case["n"], case["m"]
    space = _Space(n, m, case["mask"])
    columns = [j for j, c in enumerate(_occupation(case)) for _ in range(c)]
    U = U.to(torch.complex128).reshape(-1, m, m)
    if case["kind"] == "xmodel":
        return _exact_xmodel(space, U, columns, case["indist"], case["order"])[0]
    if case["kind"] == "grad":
        U.requires_grad_(True)
        p = _exact_probs(space, U, columns)[0]
        if case["objective"] == "sampled":
            loss = -torch.log(p[_samples(case, seed)]).mean()
        else:
            loss = (p * _observable(case, seed)).sum()
        loss.backward()
        return {"probs": p.detach(), "loss": loss.detach(), "grad": U.grad[0]}
    p = torch.cat([_exact_probs(space, U[i:i + 8], columns) for i in range(0, U.shape[0], 8)])
    if case["kind"] == "probs":
        return p if case["batch"] else p[0]
    # uniform loss: one photon fewer, each of the k photons equally likely
    eta = case["loss"]
    blocks = [p]
    for k in range(n, 0, -1):
        below = torch.zeros(1, space.sizes[k - 1], dtype=torch.float64, device=DEV)
        for a in range(0, space.sizes[k], 1 << 24):
            b = min(space.sizes[k], a + (1 << 24))
            at = space.tuples(k, a, b)
            copies = [sum((other == x).to(torch.float64) for other in at) for x in at] if space.repeats else None
            for l, (index, _, keep) in enumerate(space.parents(at)):
                q = blocks[0][0, a:b] / k
                if copies is not None:
                    q = q * copies[l]
                below[0].index_add_(0, index, q if keep is None else q * keep)
        blocks.insert(0, below)
    return [q[0] * (math.comb(n, k) * eta ** k * (1 - eta) ** (n - k)) for k, q in enumerate(blocks)]
