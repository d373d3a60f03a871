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
