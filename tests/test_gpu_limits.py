"""GPU: batches whose per-row results are more than one launch has threads for (2^32, one wavefront a result)."""
import numpy as np
import pytest
import torch

from circuits import apply_ops_tq

gpu = pytest.mark.gpu
DEV = "cuda"


def _unit_rows(rows, n, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    st = torch.randn(rows, 1 << n, dtype=torch.complex64, device=DEV, generator=g)
    return st / torch.linalg.vector_norm(st, dim=1, keepdim=True)


@gpu
def test_gradients_of_many_rows():
    """200 trainable gates in one stage and 2^26 / 200 rows and one: each row's gradients are those of a batch of
    the row alone, on the per-gate kernels.  Unit states and unit lam, 200 gates whose rounding (6e-8 each) adds as
    a random walk: 5e-5 as for the shorter circuits of the parity tests."""
    import torchquantum_amd as tq
    from torchquantum_amd import engine as E
    n, rows = 5, (1 << 26) // 200 + 1
    rng = np.random.default_rng(5)
    ops = []
    for _ in range(200):
        w = [int(x) for x in rng.choice(n, 2, replace=False)]
        ops.append(dict(name="crx", wires=w, params=rng.uniform(0, 6, (1, 1)), inverse=False))
    psi, lam = _unit_rows(rows, n, 1), _unit_rows(rows, n, 2)
    some = torch.tensor([0, 1, rows // 2, rows - 1], device=DEV)

    def grads(a, b, **kw):
        q = tq.QuantumDevice(n_wires=n, bsz=len(a), device=DEV)
        apply_ops_tq(q, ops, DEV, requires_grad=True)
        c = E.compile_tape(q._tape, n, len(a), tq.EngineOptions(**kw), torch.device(DEV))
        return E.adjoint(c, a, b, c.pool(q._tape, True, True))[0]

    got = grads(psi, lam, mode="fused", stage_bits=n, jit="off")
    assert got.shape == (rows, 200)
    want = grads(psi[some].contiguous(), lam[some].contiguous(), mode="pergate")
    assert (got[some] - want).abs().max() < 5e-5
    assert bool((got != 0).any(1).all())            # no row left out


@gpu
def test_pauli_values_of_many_rows():
    """90 strings of 8 wires in one pass and 2^26 / 90 rows and one: values and gradients of rows in every part of
    the batch against the oracle.  Unit states, sums over 256 amplitudes: 1e-5 as in the parity tests."""
    import torchquantum_amd as tq
    from oracle import statevector as O
    n, rows = 8, (1 << 26) // 90 + 1
    rng = np.random.default_rng(6)
    strings = sorted({"".join(rng.choice(list("IXYZ"), n)) for _ in range(120)})[:90]
    st = _unit_rows(rows, n, 3).requires_grad_()
    some = [0, 1, rows // 2, rows - 2, rows - 1]
    v = st[some].detach().cpu().numpy().astype(np.complex128)
    want = np.stack([O.expval_pauli(v, s) for s in strings], axis=1)
    got = tq.autograd.expval_pauli_strings(st, n, strings)
    assert np.abs(got[some].detach().cpu().numpy() - want).max() < 1e-5
    total = tq.autograd.expval_pauli_sum_state(st, n, strings, [1.0 / 90] * 90)
    assert np.abs(total[some].detach().cpu().numpy() - want.mean(1)).max() < 1e-5
    (g,) = torch.autograd.grad(total.sum(), st)
    # <P> is quadratic: Re <psi | gradient> = 2 <P>
    dot = (st.detach().conj() * g).sum(1).real / 2
    assert (dot - total.detach()).abs().max() < 1e-5


@gpu
def test_z_values_of_many_rows():
    """<Z> of every wire for 2^24 rows and one of 4 wires, against |psi|^2 in float64."""
    import torchquantum_amd as tq
    n, rows = 4, (1 << 24) + 1
    st = _unit_rows(rows, n, 4)
    got = tq.autograd.ExpvalZAll.apply(st, n)
    sign = torch.tensor([[1.0 - 2.0 * (j >> (n - 1 - w) & 1) for w in range(n)] for j in range(1 << n)],
                        dtype=torch.float64, device=DEV)
    for r0 in range(0, rows, 1 << 22):
        p = st[r0:r0 + (1 << 22)].abs().double() ** 2
        assert (got[r0:r0 + (1 << 22)] - p @ sign).abs().max() < 1e-5
