"""GPU: circuits recorded into a HIP graph.

A replay computes with the values that the graph was recorded with (and with
the current contents of the parameter tensors it reads), whatever the program
has run on the device since: each replay is compared with an eager run of the
same circuit, and eager work of other circuits lies between them.
"""
import gc

import numpy as np
import pytest
import torch

import torchquantum_amd as tq
import torchquantum_amd.functional as tqf
from torchquantum_amd import engine as E

gpu = pytest.mark.gpu
DEV = "cuda"


def _capture(f):
    """The graph of f() and its output, after warm-up passes on a side stream."""
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        for _ in range(3):
            f()
    torch.cuda.current_stream().wait_stream(side)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        out = f()
    return g, out


def _other_work(k):
    """More eager flushes than the upload ring has slots, of circuits of another size."""
    for j in range(12):
        q = tq.QuantumDevice(n_wires=7, bsz=2, device=DEV)
        for w in range(7):
            tqf.rx(q, w, params=torch.full((2, 1), 0.1 * (k + j + w), device=DEV))
            tqf.u2(q, w, params=torch.full((1, 2), 0.3 * (k + w)))
        q.get_states_1d()


@gpu
@pytest.mark.parametrize("mode", ["fused", "pergate"])
@pytest.mark.parametrize("n,rows", [(6, 3), (10, 400)])
def test_captured_circuit(mode, n, rows):
    """Gates with host values (one block or one per row: 400 rows of 2x2 blocks are several launches of host words),
    with values in a GPU tensor, and fixed ones.  The same kernels on the same numbers as the eager run, so equal."""
    theta = torch.rand(1, 1, device=DEV)
    phi = torch.rand(rows, 1)
    opts = tq.EngineOptions(mode=mode, jit="off")

    def run():
        q = tq.QuantumDevice(n_wires=n, bsz=rows, device=DEV)
        q.engine_options = opts
        with torch.no_grad():
            for w in range(n):
                tqf.rx(q, w, params=theta)
                tqf.crz(q, [w, (w + 1) % n], params=phi)
                tqf.u2(q, w, params=torch.tensor([[0.4, 0.7]]))
                tqf.hadamard(q, w)
            return q.get_states_1d()

    g, out = _capture(run)
    for k in range(4):
        E._plan_cache.clear()            # as after many other circuits: the graph's plan has to outlive the cache
        gc.collect()
        theta.fill_(0.3 + k)
        _other_work(k)
        g.replay()
        torch.cuda.synchronize()
        got = out.clone()
        assert torch.equal(got, run()), k
        assert np.isfinite(got.cpu().numpy()).all()


@gpu
def test_captured_circuit_without_matrices():
    st = torch.randn(3, 32, dtype=torch.complex64, device=DEV)

    def run():
        q = tq.QuantumDevice(n_wires=5, bsz=3, device=DEV)
        q.set_states(st)
        tqf.swap(q, [0, 3])
        tqf.swap(q, [1, 4])
        return q.get_states_1d()

    g, out = _capture(run)
    for k in range(3):
        E._plan_cache.clear()
        gc.collect()
        st.copy_(torch.randn(3, 32, dtype=torch.complex64, device=DEV))
        _other_work(k)
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, run())


@gpu
def test_pauli_sums_of_a_given_state_are_refused():
    """Coefficients and index tables come from host memory: their copies are refused while a graph is recorded, as
    torch refuses a copy from pageable memory, and work after the recording as before."""
    n = 9
    strings, coef = ["XZ" + "I" * (n - 2), "I" * (n - 1) + "Z"], [0.5, -1.5]
    q = tq.QuantumDevice(n_wires=n, bsz=2, device=DEV)
    d = tq.NoiseDevice(n_wires=4, bsz=2, device=DEV)
    for w in range(n):
        tqf.ry(q, w, params=torch.tensor([[0.3 + w]], device=DEV))
        if w < 4:
            tqf.ry(d, w, params=torch.tensor([[0.3 + w]], device=DEV))
    st = q.get_states_1d().detach()
    calls = [lambda: tq.expval_pauli_sum(q, strings, coef),
             lambda: tq.expval_joint_analytical(d, "XZIY"),
             lambda: torch.autograd.grad(tq.autograd.expval_pauli_strings(st.requires_grad_(), n, strings).sum(), st)[0]]
    want = [f().clone() for f in calls]
    for f in calls:
        with pytest.raises(RuntimeError, match="captured"):
            with torch.cuda.graph(torch.cuda.CUDAGraph()):
                f()
    for _ in range(10):              # every buffer of the ring is still in use
        for f, w in zip(calls, want):
            assert torch.equal(f(), w)
