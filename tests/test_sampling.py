"""Shot sampling (measure / expval_joint_sampling / expval_joint_sampling_grouping,
torchquantum/measurement/measurements.py:37-229) on the tqsv_sample kernels.

The reference draws with Python's random.choices, so its exact shot stream
cannot be reproduced (parity of individual shots is unpinned by design);
what is pinned is the distribution: chi-square against the oracle's |psi|^2,
zero-probability outcomes never drawn, the reference docstring's Bell-state
examples (measurements.py:188-200), and sampled means against the analytic
expectations within 5 standard errors."""
import numpy as np
import pytest
import torch

import torchquantum_amd as tq
import torchquantum_amd.functional as tqf
from torchquantum_amd.measurement import _parity_expval
from oracle import statevector as O

gpu = pytest.mark.gpu


def test_gen_bitstrings():
    assert tq.gen_bitstrings(2) == ["00", "01", "10", "11"]
    assert len(tq.gen_bitstrings(5)) == 32


def test_find_observable_groups():
    # the reference's own example (measurements.py:78-79): XXII and IIZZ share a basis
    g = tq.find_observable_groups(["XXII", "IIZZ", "ZZII"])
    assert g == {"XXZZ": ["XXII", "IIZZ"], "ZZII": ["ZZII"]}
    rng = np.random.default_rng(0)
    obs = list({"".join(rng.choice(list("IXYZ"), 5)) for _ in range(40)})
    g = tq.find_observable_groups(obs)
    assert sorted(m for ms in g.values() for m in ms) == sorted(obs)
    for basis, members in g.items():
        for m in members:
            assert all(c == "I" or basis[k] == c for k, c in enumerate(m)), (basis, m)


def test_parity_from_indices():
    """(-1)^popcount(idx & mask) with wire 0 as the most significant bit."""
    idx = torch.tensor([[0b000, 0b100, 0b110, 0b111]])
    # ZII looks at wire 0 (bit 2): +1, -1, -1, -1
    assert torch.allclose(_parity_expval(idx, "ZII", 3), torch.tensor([-0.5]))
    # IZZ: wires 1, 2 (bits 1, 0): +1, +1, -1, +1
    assert torch.allclose(_parity_expval(idx, "IZZ", 3), torch.tensor([0.5]))
    assert torch.allclose(_parity_expval(idx, "III", 3), torch.tensor([1.0]))


def _random_state_dev(n, bsz, seed):
    rng = np.random.default_rng(seed)
    v = rng.normal(size=(bsz, 2 ** n)) + 1j * rng.normal(size=(bsz, 2 ** n))
    v /= np.linalg.norm(v, axis=1, keepdims=True)
    q = tq.QuantumDevice(n_wires=n, bsz=bsz, device="cuda")
    q.set_states(torch.tensor(v, dtype=torch.complex64, device="cuda"))
    return q, v


@gpu
def test_reference_docstring_bell():
    """measurements.py:188-200: H(0), X(1), CNOT(0,1) -> II = 1, XX = 1, ZZ = -1."""
    x = tq.QuantumDevice(n_wires=2, device="cuda")
    tqf.hadamard(x, wires=0)
    tqf.x(x, wires=1)
    tqf.cnot(x, wires=[0, 1])
    for obs, want in (("II", 1.0), ("XX", 1.0), ("ZZ", -1.0)):
        got = tq.expval_joint_sampling(x, obs, n_shots=8192, seed=1)
        assert got.shape == (1,) and abs(float(got[0]) - want) < 1e-2, (obs, got)


@gpu
def test_chi_square_against_oracle():
    from scipy.stats import chi2
    n, bsz, shots = 5, 3, 40000
    q, v = _random_state_dev(n, bsz, 3)
    idx = tq.sample_indices(q, shots, seed=123).cpu().numpy()
    assert idx.shape == (bsz, shots) and idx.min() >= 0 and idx.max() < 2 ** n
    for r in range(bsz):
        p = np.abs(v[r]) ** 2
        obs = np.bincount(idx[r], minlength=2 ** n)
        stat = float(((obs - shots * p) ** 2 / (shots * p)).sum())
        assert chi2.sf(stat, 2 ** n - 1) > 1e-6, (r, stat)
    # the same seed gives the same shots; another seed does not
    assert np.array_equal(idx, tq.sample_indices(q, shots, seed=123).cpu().numpy())
    assert not np.array_equal(idx, tq.sample_indices(q, shots, seed=124).cpu().numpy())


@gpu
def test_zero_probability_never_drawn():
    """GHZ over 14 wires spans 4 probability blocks; only |0..0> and |1..1> appear."""
    n = 14
    q = tq.QuantumDevice(n_wires=n, bsz=2, device="cuda")
    tqf.hadamard(q, wires=0)
    for w in range(n - 1):
        tqf.cnot(q, wires=[w, w + 1])
    idx = tq.sample_indices(q, 20000, seed=5).cpu().numpy()
    assert set(np.unique(idx)) <= {0, 2 ** n - 1}
    frac = (idx == 0).mean()
    assert abs(frac - 0.5) < 5 * 0.5 / np.sqrt(idx.size)
    counts = tq.measure(q, n_shots=100, seed=9)
    assert len(counts) == 2 and len(counts[0]) == 2 ** n
    assert sum(counts[0].values()) == 100
    assert set(k for k, c in counts[0].items() if c) <= {"0" * n, "1" * n}


@gpu
def test_sampled_expvals_match_analytic():
    """20 wires (256 probability blocks per row): sampled <P> within 5 standard
    errors of the analytic value, for single strings and grouped strings."""
    n, bsz, shots = 20, 2, 16384
    q = tq.QuantumDevice(n_wires=n, bsz=bsz, device="cuda")
    rng = np.random.default_rng(2)
    for layer in range(3):
        for w in range(n):
            tqf.ry(q, wires=w, params=torch.tensor(rng.uniform(0, 2 * np.pi, (bsz, 1)), dtype=torch.float32,
                                                   device="cuda"))
        for w in range(0, n - 1, 2):
            tqf.cnot(q, wires=[w, w + 1])
    obs_list = ["Z" + "I" * (n - 1), "IXZ" + "I" * (n - 3), "Y" * 2 + "I" * (n - 2), "I" * (n - 1) + "X"]
    exact = tq.expval_joint_analytical_batch(q, obs_list).detach().cpu().numpy()
    tol = 5.0 / np.sqrt(shots)
    for k, o in enumerate(obs_list):
        got = tq.expval_joint_sampling(q, o, n_shots=shots, seed=10 + k).numpy()
        assert np.all(np.abs(got - exact[:, k]) < tol), (o, got, exact[:, k])
    grouped = tq.expval_joint_sampling_grouping(q, obs_list, n_shots_per_group=shots, seed=50)
    assert set(grouped) == set(obs_list)
    for k, o in enumerate(obs_list):
        assert np.all(np.abs(grouped[o].numpy() - exact[:, k]) < tol), o


@gpu
def test_sampling_against_oracle_state():
    """The distribution of a circuit's output, with the oracle computing |psi|^2."""
    from scipy.stats import chi2
    n = 6
    ops = [("hadamard", [0]), ("ry", [1], 0.7), ("cnot", [0, 2]), ("rx", [3], 1.9), ("cz", [2, 3]),
           ("u3", [4], (0.3, 1.1, -0.4)), ("swap", [4, 5]), ("crx", [5, 1], 2.2)]
    q = tq.QuantumDevice(n_wires=n, bsz=1, device="cuda")
    oo = []
    for op in ops:
        name, wires = op[0], op[1]
        p = None if len(op) == 2 else np.atleast_1d(np.asarray(op[2], dtype=np.float64))
        tqf.func_name_dict[name](q, wires=wires,
                                 params=None if p is None else torch.tensor(p[None], dtype=torch.float32,
                                                                            device="cuda"))
        oo.append(dict(name=name, wires=wires, params=p, inverse=False))
    st = O.run_ops(oo, n, 1)
    p = np.abs(st[0]) ** 2
    shots = 60000
    idx = tq.sample_indices(q, shots, seed=77).cpu().numpy()[0]
    obs = np.bincount(idx, minlength=2 ** n)
    nz = p > 1e-12
    assert obs[~nz].sum() == 0
    stat = float(((obs[nz] - shots * p[nz]) ** 2 / (shots * p[nz])).sum())
    assert chi2.sf(stat, int(nz.sum()) - 1) > 1e-6, stat


def _uniforms(seed, bsz, shots):
    """The documented uniforms: splitmix64(seed ^ splitmix64(row * shots + shot)), top 53 bits."""
    m = (1 << 64) - 1

    def mix(x):
        x = (x + 0x9E3779B97F4A7C15) & m
        x = ((x ^ (x >> 30)) * 0xBF58476D1CE4E5B9) & m
        x = ((x ^ (x >> 27)) * 0x94D049BB133111EB) & m
        return x ^ (x >> 31)

    return np.array([(mix(seed ^ mix(w)) >> 11) / 2.0 ** 53 for w in range(bsz * shots)]).reshape(bsz, shots)


@gpu
@pytest.mark.parametrize("n", [1, 5, 6, 7, 11, 12, 13, 15])
@pytest.mark.parametrize("holes", [False, True])
def test_shots_invert_the_cumulative_distribution(n, holes):
    """Every shot is the amplitude whose slice of the cumulative |psi|^2 holds its uniform, to the rounding of the
    probabilities (each within 2^-23 of itself in float32, so their sums within 2^-23 of the total; four times
    that is allowed); blocks and segments cut short, whole and empty."""
    bsz, shots, seed = 3, 500, 12345
    q, v = _random_state_dev(n, bsz, 40 + n)
    if holes:                       # mass in a few places only: empty segments and blocks between them
        keep = np.zeros(2 ** n, dtype=bool)
        keep[np.random.default_rng(n).choice(2 ** n, max(1, 2 ** n // 50), replace=False)] = True
        v = v * keep
        q.set_states(torch.tensor(v, dtype=torch.complex64, device="cuda"))
    v = q.get_states_1d().cpu().numpy().astype(np.complex128)
    idx = tq.sample_indices(q, shots, seed=seed).cpu().numpy()
    u = _uniforms(seed, bsz, shots)
    for b in range(bsz):
        p = np.abs(v[b]) ** 2
        cum = np.cumsum(p)
        t, tol = u[b] * cum[-1], 4 * 2.0 ** -23 * cum[-1]
        assert (p[idx[b]] > 0).all()
        assert (t <= cum[idx[b]] + tol).all() and (t >= cum[idx[b]] - p[idx[b]] - tol).all()
