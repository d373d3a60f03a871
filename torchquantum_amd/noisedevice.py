"""Density-matrix device: torchquantum's ``NoiseDevice``
(torchquantum/device/noisedevices.py:36-105, gate application
torchquantum/functional/gate_wrapper.py:265-321 and :433-440).

The density matrix rho of n wires is kept as a 2n-wire register on the same
engine as the statevectors: flat index r * 2^n + c holds rho[r, c] (the
reference's layout, ``densities`` of shape [bsz] + [2] * 2n, |r><c|).  Then

    vec(U rho U^dagger) = (U (x) conj(U)) vec(rho),

so a gate U on wires W is the gate U on register wires W (the row index)
followed by conj(U) on register wires W + n (the column index).  Every gate
kernel, the fused stages and the adjoint gradient apply unchanged; gradients
w.r.t. gate parameters flow through both copies.

A channel with Kraus operators K_k on wires W acts on vec(rho) as the
superoperator sum_k K_k (x) conj(K_k): one dense op on register wires
(W, W + n).  Channels are not unitary, so the adjoint sweep cannot pass
through them: a differentiable pass with a channel raises.

Deliberate differences from the reference (both are errors there):
* the reference computes rho U^dagger as ``rho @ conj(U)``
  (gate_wrapper.py:287-305, no transpose), which is wrong for every
  non-symmetric U (RY, U3, ...); here it is rho U^dagger;
* ``measure`` draws from |rho_ii|^2 there (measurements.py:48-58 squares the
  probabilities again); here from rho_ii.
"""
from __future__ import annotations

import functools
from typing import List, Optional, Sequence, Union

import numpy as np
import torch
import torch.nn as nn

from . import engine as E
from .autograd import _PHASE, pauli_masks
from .device import QuantumDevice, _default_device

C_DTYPE = torch.complex64

__all__ = ["NoiseDevice", "superoperator", "amplitude_damping_kraus", "phase_damping_kraus",
           "depolarizing_kraus", "bit_flip_kraus", "phase_flip_kraus"]


def superoperator(kraus: Sequence[np.ndarray]) -> np.ndarray:
    """sum_k K_k (x) conj(K_k): the channel rho -> sum_k K_k rho K_k^dagger
    acting on vec(rho) (row-major: index r * d + c)."""
    ks = [np.asarray(k, dtype=np.complex128) for k in kraus]
    d = ks[0].shape[0]
    if any(k.shape != (d, d) for k in ks):
        raise ValueError("Kraus operators must be square and of one size")
    return sum((k[:, None, :, None] * np.conj(k)[None, :, None, :]).reshape(d * d, d * d) for k in ks)


def amplitude_damping_kraus(gamma: float) -> List[np.ndarray]:
    g = float(gamma)
    return [np.array([[1, 0], [0, np.sqrt(1 - g)]]), np.array([[0, np.sqrt(g)], [0, 0]])]


def phase_damping_kraus(lam: float) -> List[np.ndarray]:
    l_ = float(lam)
    return [np.array([[1, 0], [0, np.sqrt(1 - l_)]]), np.array([[0, 0], [0, np.sqrt(l_)]])]


def depolarizing_kraus(p: float) -> List[np.ndarray]:
    """rho -> (1 - p) rho + p/3 (X rho X + Y rho Y + Z rho Z)."""
    p = float(p)
    x = np.array([[0, 1], [1, 0]])
    y = np.array([[0, -1j], [1j, 0]])
    z = np.array([[1, 0], [0, -1]])
    return [np.sqrt(1 - p) * np.eye(2), np.sqrt(p / 3) * x, np.sqrt(p / 3) * y, np.sqrt(p / 3) * z]


def bit_flip_kraus(p: float) -> List[np.ndarray]:
    p = float(p)
    return [np.sqrt(1 - p) * np.eye(2), np.sqrt(p) * np.array([[0, 1], [1, 0]])]


def phase_flip_kraus(p: float) -> List[np.ndarray]:
    p = float(p)
    return [np.sqrt(1 - p) * np.eye(2), np.sqrt(p) * np.array([[1, 0], [0, -1]])]


class NoiseDevice(nn.Module):
    """Density matrices of ``bsz`` rows on ``n_wires`` wires, starting in
    |0..0><0..0| (noisedevices.py:36-74).  The functional gates and the gate
    methods apply U rho U^dagger; the channel methods apply Kraus maps."""

    def __init__(self, n_wires: int, device_name: str = "noisedevice", bsz: int = 1,
                 device: Union[torch.device, str, None] = None, record_op: bool = False):
        super().__init__()
        if n_wires < 1:
            raise ValueError("n_wires must be >= 1")
        self.n_wires = n_wires
        self.device_name = device_name
        self.record_op = record_op
        self.op_history: List[dict] = []
        self.reg = QuantumDevice(2 * n_wires, bsz=bsz,
                                 device=device if device is not None else _default_device())

    # ------------------------------------------------------------ plumbing
    @property
    def bsz(self) -> int:
        return self.reg.bsz

    @property
    def device(self) -> torch.device:
        return self.reg.device

    @property
    def engine_options(self):
        return self.reg.engine_options

    @engine_options.setter
    def engine_options(self, v):
        self.reg.engine_options = v

    def _push(self, op: E.TapeOp):
        """A gate U on wires W: U on the row wires, conj(U) on the column wires."""
        n = self.n_wires
        self.reg._push(op)
        self.reg._push(E.TapeOp(op.name, tuple([w + n for w in op.wires]), op.params, op.inverse, op.version,
                                not op.conj, op.nonunitary))

    def flush(self, options: Optional[E.EngineOptions] = None):
        self.reg.flush(options)

    # ------------------------------------------------------------ channels
    def kraus(self, wires: Union[int, Sequence[int]], kraus_ops: Sequence[np.ndarray]):
        """rho -> sum_k K_k rho K_k^dagger on ``wires`` (K_k: 2^k x 2^k, wires[0]
        the most significant bit, as for the gates)."""
        self._channel(wires, superoperator(kraus_ops))

    def _channel(self, wires: Union[int, Sequence[int]], S: np.ndarray):
        """Record a channel given as its superoperator.  The matrix stays on
        the host, where the flush builds its matrix pool."""
        ws = [int(wires)] if isinstance(wires, (int, np.integer)) else [int(w) for w in wires]
        n = self.n_wires
        if len(set(ws)) != len(ws) or any(not 0 <= w < n for w in ws):
            raise ValueError(f"bad wires {ws} for {n} wires")
        if S.shape[0] != 1 << (2 * len(ws)):
            raise ValueError(f"Kraus operators of size {int(np.sqrt(S.shape[0]))} do not match {len(ws)} wire(s)")
        if len(ws) > 5:
            raise ValueError("channels act on at most 5 wires (a 2^(2k) superoperator, 2k <= 10)")
        mat = torch.from_numpy(S.astype(np.complex64))
        reg_wires = tuple(ws) + tuple(w + n for w in ws)
        self.reg._push(E.TapeOp("qubitunitaryfast", reg_wires, mat, False, mat._version, nonunitary=True))

    def _each(self, wires, kraus_ops: Sequence[np.ndarray]):
        S = superoperator(kraus_ops)
        for w in ([wires] if isinstance(wires, (int, np.integer)) else wires):
            self._channel(int(w), S)

    def amplitude_damping(self, wires, gamma: float):
        self._each(wires, amplitude_damping_kraus(gamma))

    def phase_damping(self, wires, lam: float):
        self._each(wires, phase_damping_kraus(lam))

    def depolarizing(self, wires, p: float):
        self._each(wires, depolarizing_kraus(p))

    def bit_flip(self, wires, p: float):
        self._each(wires, bit_flip_kraus(p))

    def phase_flip(self, wires, p: float):
        self._each(wires, phase_flip_kraus(p))

    # ------------------------------------------------------------ state
    @property
    def densities(self) -> torch.Tensor:
        """[bsz] + [2] * 2n: densities[b, r..., c...] = rho_b[r, c]."""
        return self.reg.states

    @densities.setter
    def densities(self, value: torch.Tensor):
        value = torch.as_tensor(value)
        bsz = value.shape[0]
        v = value.reshape(bsz, -1)
        if v.shape[1] != 1 << (2 * self.n_wires):
            raise ValueError(f"density has {v.shape[1]} entries per row, expected {1 << (2 * self.n_wires)}")
        self.reg.states = v

    @property
    def density(self) -> torch.Tensor:
        """The initial |0..0><0..0| as [2] * 2n (the reference's buffer)."""
        d = torch.zeros(1 << (2 * self.n_wires), dtype=C_DTYPE, device=self.reg._sv_device())
        d[0] = 1.0
        return d.reshape([2] * (2 * self.n_wires))

    def matrices(self) -> torch.Tensor:
        """[bsz, 2^n, 2^n] view of the density matrices."""
        d = 1 << self.n_wires
        return self.reg.get_states_1d().reshape(self.bsz, d, d)

    def get_probs_1d(self) -> torch.Tensor:
        """Diagonals rho_ii, [bsz, 2^n] (noisedevices.py:88-92)."""
        return torch.diagonal(self.matrices(), offset=0, dim1=1, dim2=2)

    def get_prob_1d(self) -> torch.Tensor:
        """Diagonal of the initial density (noisedevices.py:94-97)."""
        d = 1 << self.n_wires
        return torch.diagonal(self.density.reshape(d, d), offset=0, dim1=0, dim2=1)

    def reset_states(self, bsz: int):
        self.reg.reset_states(bsz)

    def trace(self) -> torch.Tensor:
        return self.get_probs_1d().sum(-1)

    def purity(self) -> torch.Tensor:
        """tr(rho^2) = sum |rho_ij|^2 (rho Hermitian), [bsz]."""
        m = self.matrices()
        return (m.real ** 2 + m.imag ** 2).sum((-1, -2))

    @property
    def name(self):
        return self.__class__.__name__

    def __repr__(self):
        return (f" class: {self.name} \n device name: {self.device_name} \n number of qubits: {self.n_wires} \n"
                f" batch size: {self.bsz} \n current computing device: {self.reg._sv_device()} \n"
                f" recording op history: {self.record_op} \n"
                f" current states: {repr(self.get_probs_1d().cpu().detach().numpy())}")

    def _apply(self, fn, recurse=True):
        return super()._apply(fn, recurse)


# ----------------------------------------------------------------------------
# expectations on densities: Tr(rho P) for Pauli strings
# ----------------------------------------------------------------------------
def _string_tables(n: int, observables: Sequence[str]):
    """For T strings: the gathered index r * 2^n + (r ^ x) and its sign
    (-1)^popcount(r & z), [T, 2^n] each, and i^nY as its real and imaginary
    parts, [T] each."""
    d = 1 << n
    masks = [pauli_masks(obs, n) for obs in observables]
    x, z, ny = (np.array(v, dtype=np.int64) for v in zip(*masks))
    r = np.arange(d, dtype=np.int64)
    par = r & z[:, None]
    for sh in (16, 8, 4, 2, 1):
        par ^= par >> sh
    ph = _PHASE[ny % 4]
    return (r * d + (r ^ x[:, None]), (1 - 2 * (par & 1)).astype(np.float32),
            ph.real.astype(np.float32), ph.imag.astype(np.float32))


_small_tables = functools.lru_cache(maxsize=32)(_string_tables)
SMALL_TABLE = 1 << 16          # entries of a table that is kept for the next call with the same strings
RING_TABLE = 1 << 18           # entries of a table that goes through the pinned upload buffers, which stay allocated
CHUNK = 1 << 24                # entries gathered at a time over all rows (128 MiB, and their products as much)


def density_expval_strings(dev: NoiseDevice, observables: Sequence[str]) -> torch.Tensor:
    """Re Tr(rho P_t) for Pauli strings (char k <-> wire k) -> [bsz, T].

    P|r> = i^{nY} (-1)^{popcount(r & z)} |r ^ x>, so
    Tr(rho P) = i^{nY} sum_r (-1)^{popcount(r & z)} rho[r, r ^ x]:
    a gather of 2^n entries of the 4^n per row and string (differentiable; the
    gradient reaches the gates through the engine's adjoint sweep)."""
    n = dev.n_wires
    flat = dev.reg.get_states_1d()                         # [bsz, 4^n]
    d = 1 << n
    observables = list(observables)
    if not observables:
        raise RuntimeError("no observables")
    cols = []
    per = max(1, CHUNK // (flat.shape[0] << n))
    for t0 in range(0, len(observables), per):
        obs = tuple(observables[t0:t0 + per])
        idx, sgn, re, im = (_small_tables if len(obs) * d <= SMALL_TABLE else _string_tables)(n, obs)
        put = E.upload if len(obs) * d <= RING_TABLE else _copied
        g = flat[:, put(idx.reshape(-1), flat.device)].reshape(-1, len(obs), d)
        s = (g * put(sgn, flat.device)).sum(-1)                # sum_r sign rho[r, r^x]
        cols.append(s.real * E.upload(re, flat.device) - s.imag * E.upload(im, flat.device))    # Re(i^ny s)
    return torch.cat(cols, dim=-1)


def _copied(host: np.ndarray, device: torch.device) -> torch.Tensor:
    return torch.from_numpy(host).to(device)
