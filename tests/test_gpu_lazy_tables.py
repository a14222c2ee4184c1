"""Tables that a plan makes at the first call that needs them."""
import threading

import pytest
import torch
from helpers import haar_unitary

from photonic_engines_amd.slos import FockSLOSKernel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("call", ["loss", "gradient", "x-model"])
def test_first_use_beside_another_threads_capture(call):
    """Another thread records a graph, in the mode in which allocations of any thread would end it, while
    this one makes the first loss, gradient or x-model call of a plan whose forward has run."""
    n, m = 8, 12
    U = haar_unitary(m, 3).to(torch.complex64).cuda()

    def run(k):
        if call == "loss":
            return k._plan.loss_thin(p, [0.5] * n)[3]
        if call == "x-model":
            return k.probs(U, indist=0.7, order=2)
        V = U.clone().requires_grad_()
        return torch.autograd.grad(k.probs(V).square().sum(), V)[0]

    def kernel():
        return FockSLOSKernel(n, m, [1] * n + [0] * (m - n), device="cuda")

    p = kernel().probs(U).unsqueeze(0)
    ref = run(kernel())  # (and torch's allocator holds the buffers afterwards)
    k = kernel()
    k.probs(U)
    a = torch.zeros(16, device="cuda")
    g = torch.cuda.CUDAGraph()
    begun, go_on, failed = threading.Event(), threading.Event(), []

    def record():
        try:
            with torch.cuda.stream(torch.cuda.Stream()):
                g.capture_begin(capture_error_mode="global")
                begun.set()
                a.add_(1)
                go_on.wait(60)
                g.capture_end()
        except Exception as e:  # noqa: BLE001
            failed.append(e)
            begun.set()

    torch.cuda.synchronize()
    t = threading.Thread(target=record)
    t.start()
    begun.wait(60)
    try:
        out = run(k)
    finally:
        go_on.set()
        t.join()
    assert not failed, failed
    assert torch.equal(out, ref)
    for i in range(1, 4):
        g.replay()
        assert float(a.sum()) == 16 * i
