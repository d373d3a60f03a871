"""The work that is timed: circuits, gradients, expectation values and shots, at the sizes they are used at.

``listed()`` gives the cases, ``draw(rng)`` one more of the same ranges, ``prepare(case, seed)`` what a program
holds before the call, ``run(state)`` one pass through the public entry points, ``work(case)`` the bytes and
operations that pass cannot do without, and ``exact(case, seed)`` its outputs in 64 bits from plain torch.

A case's circuit (gates, wires, Pauli strings) follows from the case alone; the angles, inputs and states follow
from the seed.
"""
import math
import random

import torch

import torchquantum_amd as tq
import torchquantum_amd.functional as tqf
from torchquantum_amd.batch import CircuitBatch

GPU = "cuda"
EXACT_AMPS = 1 << 25          # circuits on states above this are too slow to repeat in 64 bits


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------
def listed():
    return [
        # Variational training at the size the framework is quoted on: RX, RY, RZ on every wire and a CNOT ring,
        # ten times, per-row input angles, a Pauli-sum loss and the gradient of every angle.
        {"name": "gradient_24q_64rows", "kind": "gradient", "n": 24, "rows": 64, "layers": 10},
        # The same at the size of a quick experiment, whose state the last-level cache can nearly hold.
        {"name": "gradient_20q_16rows", "kind": "gradient", "n": 20, "rows": 16, "layers": 10},
        # A small model with an odd number of rows: short launches, stages below the size that is compiled.
        {"name": "gradient_13q_37rows", "kind": "gradient", "n": 13, "rows": 37, "layers": 4},
        # Inference, forward only: RY on every wire, CZ on even and odd pairs, <Z> of every wire.
        {"name": "layers_20q_16rows", "kind": "layers", "n": 20, "rows": 16, "layers": 20},
        # The largest state of the benchmark (32 GiB), with a three-wire gate after every fifth layer.
        {"name": "layers_30q_4rows", "kind": "layers", "n": 30, "rows": 4, "layers": 20},
        # Serving a small fixed circuit recorded once: U3 on every wire, a CNOT ring, eight times; latency counts.
        {"name": "replay_10q_32rows", "kind": "replay", "n": 10, "rows": 32, "layers": 8},
        # Many independent circuits of different sizes and depths in one launch, <Z_0> of each.
        {"name": "batch_64circuits", "kind": "batch", "circuits": 64, "n_max": 22, "depth_max": 40, "structure": 1},
        # One step of a hybrid classifier: encoder, ansatz, <Z> read-out, a linear head, cross entropy, backward.
        {"name": "training_10q_256rows", "kind": "training", "n": 10, "rows": 256, "layers": 4},
        # The energy of a spin Hamiltonian with longer strings in a given state, and its gradient there.
        {"name": "energy_22q_8rows", "kind": "energy", "n": 22, "rows": 8, "strings": 80, "grad": True, "structure": 2},
        # Gate by gate without fusion, one to six wires wide, controlled, diagonal, exchanging and dense.
        {"name": "gates_24q_5rows", "kind": "gates", "n": 24, "rows": 5, "gates": 40, "structure": 3},
        # Noisy circuits on density matrices: rotations, a CNOT ring and a depolarizing channel on every wire.
        {"name": "density_10q_3rows", "kind": "density", "n": 10, "rows": 3, "layers": 3},
        # Shots from a batch of states.
        {"name": "shots_20q_16rows", "kind": "shots", "n": 20, "rows": 16, "shots": 8192},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _rows(rng, n, cap, most):
    """Rows spread over their logarithm, with rows * 2^n at most 2^cap."""
    return _log(rng, 1, max(1, min(most, 1 << max(0, cap - n))))


def draw(rng):
    kind = rng.choice(["gradient", "gradient", "layers", "layers", "replay", "batch", "training", "energy", "energy",
                       "gates", "density", "shots"])
    structure = rng.randrange(1, 10 ** 6)
    if kind == "gradient":
        n = rng.randint(5, 23)
        return {"kind": kind, "n": n, "rows": _rows(rng, n, 26, 300), "layers": rng.randint(1, 4)}
    if kind == "layers":
        n = rng.randint(5, 27)
        return {"kind": kind, "n": n, "rows": _rows(rng, n, 28, 300), "layers": rng.randint(2, 7)}
    if kind == "replay":
        n = rng.randint(4, 13)
        return {"kind": kind, "n": n, "rows": _rows(rng, n, 18, 200), "layers": rng.randint(2, 8)}
    if kind == "batch":
        return {"kind": kind, "circuits": _log(rng, 5, 64), "n_max": rng.randint(10, 22),
                "depth_max": rng.randint(8, 40), "structure": structure}
    if kind == "training":
        n = rng.randint(4, 16)
        return {"kind": kind, "n": n, "rows": max(4, _rows(rng, n, 20, 600)), "layers": rng.randint(1, 4)}
    if kind == "energy":
        n = rng.randint(6, 25)
        return {"kind": kind, "n": n, "rows": _rows(rng, n, 27, 100), "strings": _log(rng, 4, 100),
                "grad": rng.random() < 0.6, "structure": structure}
    if kind == "gates":
        n = rng.randint(7, 26)
        return {"kind": kind, "n": n, "rows": _rows(rng, n, 27, 100), "gates": rng.randint(15, 45),
                "structure": structure}
    if kind == "density":
        n = rng.randint(3, 10)
        return {"kind": kind, "n": n, "rows": _rows(rng, 2 * n, 22, 50), "layers": rng.randint(1, 4)}
    n = rng.randint(4, 25)
    return {"kind": kind, "n": n, "rows": _rows(rng, n, 27, 100), "shots": _log(rng, 16, 20000)}


# ---------------------------------------------------------------------------
# circuits: lists of (gate name, wires, columns of the angle vector)
# ---------------------------------------------------------------------------
def _ansatz(n, layers, first=0):
    """RX, RY, RZ on every wire, then a CNOT ring, per layer."""
    out, k = [], first
    for _ in range(layers):
        for name in ("rx", "ry", "rz"):
            for w in range(n):
                out.append((name, (w,), (k,)))
                k += 1
        out += [("cnot", (w, (w + 1) % n), ()) for w in range(n)]
    return out


def _brick(n, layers):
    """RY on every wire, CZ on even then odd pairs, a three-wire gate after every fifth layer from 24 wires on."""
    r, out, k = random.Random(n), [], 0
    for layer in range(layers):
        for w in range(n):
            out.append(("ry", (w,), (k,)))
            k += 1
        for start in (0, 1):
            out += [("cz", (w, w + 1), ()) for w in range(start, n - 1, 2)]
        if n >= 24 and layer % 5 == 4:
            out.append((r.choice(["toffoli", "cswap"]), tuple(r.sample(range(n), 3)), ()))
    return out


def _u3_ring(n, layers):
    out, k = [], 0
    for _ in range(layers):
        for w in range(n):
            out.append(("u3", (w,), (k, k + 1, k + 2)))
            k += 3
        out += [("cnot", (w, (w + 1) % n), ()) for w in range(n)]
    return out


def _uneven(case):
    """[(wires, circuit)]: 8 (or fewer) to n_max wires, 4 to depth_max layers of random one- and two-wire gates."""
    r, out = random.Random(case["structure"]), []
    for _ in range(case["circuits"]):
        n, depth = r.randint(min(8, case["n_max"]), case["n_max"]), r.randint(4, case["depth_max"])
        prog, k = [], 0
        for _ in range(depth * n):
            name = r.choice(["hadamard", "rx", "ry", "rz", "u3", "cnot", "cz", "swap"])
            m = {"rx": 1, "ry": 1, "rz": 1, "u3": 3}.get(name, 0)
            prog.append((name, tuple(r.sample(range(n), 2 if name in ("cnot", "cz", "swap") else 1)),
                         tuple(range(k, k + m))))
            k += m
        out.append((n, prog))
    return out


def _mixed(case):
    """Gates of every shape the unfused path has: one wire, controlled, diagonal, exchanging, dense to six wires."""
    r, n, out, k = random.Random(case["structure"]), case["n"], [], 0
    names = ["hadamard", "rx", "ry", "rz", "u3", "cnot", "cz", "swap", "crx", "rzz", "rxx", "toffoli", "cswap",
             "dense2", "dense3", "dense4", "dense5", "dense6"]
    for i in range(case["gates"]):
        name = names[i % len(names)]
        wide = {"cnot": 2, "cz": 2, "swap": 2, "crx": 2, "rzz": 2, "rxx": 2, "toffoli": 3, "cswap": 3}.get(name, 1)
        if name.startswith("dense"):
            wide = int(name[5:])
        m = {"rx": 1, "ry": 1, "rz": 1, "u3": 3, "crx": 1, "rzz": 1, "rxx": 1}.get(name, 0)
        out.append((name, tuple(r.sample(range(n), wide)), tuple(range(k, k + m))))
        k += m
    return out


def _strings(case):
    """Pauli strings and weights: the terms of a spin chain in a field, then random strings of two to six letters."""
    r, n, out = random.Random(case["structure"]), case["n"], []
    chain = [{w: p, (w + 1) % n: p} for p in "XYZ" for w in range(n)] + [{w: "X"} for w in range(n)]
    r.shuffle(chain)
    for i in range(case["strings"]):
        if i % 4 != 3 and chain:
            d = chain.pop()
        else:
            d = {w: r.choice("XYZ") for w in r.sample(range(n), r.randint(2, min(6, n)))}
        out.append(("".join(d.get(w, "I") for w in range(n)), r.uniform(-1, 1)))
    return out


def _loss_terms(n):
    """sum_i <Z_i Z_i+1> around the ring + 0.5 sum_i <X_i>."""
    zz = ["".join("Z" if w in (i, (i + 1) % n) else "I" for w in range(n)) for i in range(n)]
    x = ["".join("X" if w == i else "I" for w in range(n)) for i in range(n)]
    return zz + x, [1.0] * n + [0.5] * n


def _columns(prog):
    return sum(len(cols) for _, _, cols in prog)


def _generator(seed):
    return torch.Generator(device=GPU).manual_seed(int(seed))


def _angles(g, count, spread=None):
    """`count` angles: uniform over a turn, or normal with the given spread (a trained or freshly set up ansatz)."""
    if spread is None:
        return torch.rand(count, device=GPU, generator=g) * (2 * math.pi)
    return torch.randn(count, device=GPU, generator=g) * spread


def _random_states(g, rows, n):
    v = torch.randn(rows, 1 << n, 2, device=GPU, generator=g)
    s = torch.view_as_complex(v)
    for r in range(rows):
        s[r] /= torch.linalg.vector_norm(v[r])
    return s


def _dense(g, prog):
    """A random unitary for every dense gate, complex64."""
    out = {}
    for i, (name, wires, _) in enumerate(prog):
        if name.startswith("dense"):
            d = 1 << len(wires)
            z = torch.randn(d, d, 2, generator=torch.Generator().manual_seed(i + int(g.initial_seed())),
                            dtype=torch.float64)
            out[i] = torch.linalg.qr(torch.view_as_complex(z))[0].to(torch.complex64).to(GPU)
    return out


def _record(qdev, prog, params, dense=None):
    for i, (name, wires, cols) in enumerate(prog):
        if name.startswith("dense"):
            tqf.qubitunitaryfast(qdev, wires=list(wires), params=dense[i])
        elif cols:
            tqf.func_name_dict[name](qdev, wires=list(wires), params=params[i])
        else:
            tqf.func_name_dict[name](qdev, wires=list(wires))


def _gate_params(prog, theta):
    """{gate index: its [1, P] parameter tensor}, as separate tensors of a program's own."""
    return {i: theta[cols[0]:cols[-1] + 1].clone().reshape(1, -1) for i, (_, _, cols) in enumerate(prog) if cols}


def _set_ansatz(module, theta):
    """The module's [1, 1] parameters, in the order of _ansatz's columns."""
    with torch.no_grad():
        for k, p in enumerate(module.parameters()):
            p.copy_(theta[k])


# ---------------------------------------------------------------------------
# prepare and run
# ---------------------------------------------------------------------------
def prepare(case, seed):
    kind, g = case["kind"], _generator(seed)
    s = {"case": case}
    n, rows = case.get("n"), case.get("rows")
    if kind == "gradient":
        s["ansatz"] = tq.RXYZCXLayer0({"n_wires": n, "n_blocks": case["layers"]}).to(GPU)
        _set_ansatz(s["ansatz"], _angles(g, 3 * n * case["layers"], 0.1))
        s["params"] = list(s["ansatz"].parameters())
        s["phi"] = torch.rand(rows, 1, device=GPU, generator=g) * math.pi
        s["strings"], s["weights"] = _loss_terms(n)
    elif kind == "layers":
        s["prog"] = _brick(n, case["layers"])
        s["params"] = _gate_params(s["prog"], _angles(g, _columns(s["prog"])))
        s["measure"] = tq.MeasureAll(tq.PauliZ)
    elif kind == "replay":
        prog = _u3_ring(n, case["layers"])
        params = _gate_params(prog, _angles(g, _columns(prog)))
        s["replay"] = tq.CircuitReplay(lambda q: _record(q, prog, params), n_wires=n, bsz=rows)
        s["measure"] = tq.MeasureAll(tq.PauliZ)
    elif kind == "batch":
        theta = _angles(g, max(_columns(p) for _, p in _uneven(case))).cpu().double().numpy()
        circuits = [(m, [{"name": name, "wires": list(w), "params": theta[list(cols)] if cols else None,
                          "inverse": False} for name, w, cols in prog]) for m, prog in _uneven(case)]
        s["batch"] = CircuitBatch(circuits, device=GPU)
    elif kind == "training":
        s["encoder"] = tq.GeneralEncoder([{"input_idx": [i], "func": "ry", "wires": [i]} for i in range(n)])
        s["ansatz"] = tq.RXYZCXLayer0({"n_wires": n, "n_blocks": case["layers"]}).to(GPU)
        _set_ansatz(s["ansatz"], _angles(g, 3 * n * case["layers"]))
        s["head"] = torch.nn.Linear(n, 4).to(GPU)
        with torch.no_grad():
            s["head"].weight.copy_(torch.randn(4, n, device=GPU, generator=g) * 0.5)
            s["head"].bias.copy_(torch.randn(4, device=GPU, generator=g) * 0.1)
        s["params"] = list(s["ansatz"].parameters()) + list(s["head"].parameters())
        s["measure"] = tq.MeasureAll(tq.PauliZ)
        s["x"] = torch.rand(rows, n, device=GPU, generator=g) * math.pi
        s["y"] = torch.randint(0, 4, (rows,), device=GPU, generator=g)
    elif kind == "energy":
        s["states"] = _random_states(g, rows, n).requires_grad_(case["grad"])
        terms = _strings(case)
        s["strings"], s["weights"] = [t for t, _ in terms], [w for _, w in terms]
    elif kind == "gates":
        s["prog"] = _mixed(case)
        s["params"] = _gate_params(s["prog"], _angles(g, _columns(s["prog"])))
        s["dense"] = _dense(g, s["prog"])
        s["states"] = _random_states(g, rows, n)
    elif kind == "density":
        s["prog"] = _ansatz(n, case["layers"])
        s["params"] = _gate_params(s["prog"], _angles(g, _columns(s["prog"])))
        s["measure"] = tq.MeasureAll(tq.PauliZ)
    elif kind == "shots":
        s["qdev"] = tq.QuantumDevice(n_wires=n, bsz=rows, device=GPU)
        s["qdev"].set_states(_random_states(g, rows, n))
        s["seed"] = int(seed)
    else:
        raise ValueError(f"unknown kind {kind!r}")
    if kind in ("gradient", "layers", "training", "density"):
        run(s)                               # plans the circuit; large states queue their stage kernels' compiles
        tq.wait_for_compiled_stages()
    return s


def run(s):
    case = s["case"]
    kind, n, rows = case["kind"], case.get("n"), case.get("rows")
    if kind == "gradient":
        q = tq.QuantumDevice(n_wires=n, bsz=rows, device=GPU)
        for w in range(n):
            tqf.ry(q, w, params=s["phi"])
        s["ansatz"](q)
        loss = tq.expval_pauli_sum(q, s["strings"], s["weights"]).mean()
        grads = torch.autograd.grad(loss, s["params"])
        return {"loss": loss.detach(), "gradient": torch.cat([x.reshape(-1) for x in grads])}
    if kind == "layers":
        q = tq.QuantumDevice(n_wires=n, bsz=rows, device=GPU)
        _record(q, s["prog"], s["params"])
        return s["measure"](q)
    if kind == "replay":
        return s["measure"](s["replay"]())
    if kind == "batch":
        return s["batch"].run()
    if kind == "training":
        q = tq.QuantumDevice(n_wires=n, bsz=rows, device=GPU)
        s["encoder"](q, s["x"])
        s["ansatz"](q)
        logits = s["head"](s["measure"](q))
        loss = torch.nn.functional.cross_entropy(logits, s["y"])
        grads = torch.autograd.grad(loss, s["params"])
        return {"logits": logits.detach(), "loss": loss.detach(), "head": [grads[-2], grads[-1]],
                "ansatz": torch.cat([x.reshape(-1) for x in grads[:-2]])}
    if kind == "energy":
        q = tq.QuantumDevice(n_wires=n, bsz=rows, device=GPU)
        q.set_states(s["states"])
        if not case["grad"]:
            return tq.expval_joint_analytical_batch(q, s["strings"])
        energy = tq.expval_pauli_sum(q, s["strings"], s["weights"])
        (grad,) = torch.autograd.grad(energy.sum(), s["states"])
        return {"energy": energy.detach(), "gradient": grad}
    if kind == "gates":
        q = tq.QuantumDevice(n_wires=n, bsz=rows, device=GPU)
        q.engine_options = tq.EngineOptions(mode="pergate")
        q.set_states(s["states"])
        _record(q, s["prog"], s["params"], s["dense"])
        return q.get_states_1d()
    if kind == "density":
        q = tq.NoiseDevice(n, bsz=rows, device=GPU)
        for i, (name, wires, cols) in enumerate(s["prog"]):
            if cols:
                tqf.func_name_dict[name](q, wires=list(wires), params=s["params"][i])
            else:
                tqf.func_name_dict[name](q, wires=list(wires))
            if name == "cnot" and wires[1] == 0:              # the ring is closed: noise on every wire
                q.depolarizing(list(range(n)), 0.02)
        return {"densities": q.densities, "z": s["measure"](q)}
    return tq.sample_indices(s["qdev"], case["shots"], seed=s["seed"])


# ---------------------------------------------------------------------------
# the least work of a pass
# ---------------------------------------------------------------------------
def _flops_per_amp(prog):
    """Real operations per amplitude: 14 for a one-wire complex matrix (runs on one wire count once), 6 for a real
    one, 8 * 2^k for a dense block of k wires, half of that where one control halves the amplitudes."""
    total, open_runs = 0.0, set()
    for name, wires, _ in prog:
        if name in ("rx", "ry", "rz", "u3", "hadamard") and len(wires) == 1:
            if wires[0] not in open_runs:
                total += 14.0
                open_runs.add(wires[0])
            continue
        open_runs.difference_update(wires)
        if name.startswith("dense"):
            total += 8.0 * (1 << len(wires))
        elif name == "rxx":
            total += 14.0
        elif name in ("crx", "rzz"):
            total += 7.0
    return total


def work(case):
    kind = case["kind"]
    if kind == "batch":
        circuits = _uneven(case)
        return {"bytes": sum(16.0 * (1 << n) for n, _ in circuits),
                "flops": sum(_flops_per_amp(p) * (1 << n) for n, p in circuits)}
    n, rows = case["n"], case["rows"]
    amps = float(rows) * (1 << n)
    if kind in ("gradient", "training"):
        # the state and its gradient each written and read once; forward, both sides of the adjoint, the sums
        return {"bytes": 32.0 * amps, "flops": amps * case["layers"] * n * (14.0 + 28.0 + 12.0)}
    if kind == "layers":
        return {"bytes": 16.0 * amps, "flops": amps * 6.0 * n * case["layers"]}
    if kind == "replay":
        return {"bytes": 16.0 * amps, "flops": amps * 14.0 * n * case["layers"]}
    if kind == "energy":
        return {"bytes": (16.0 if case["grad"] else 8.0) * amps, "flops": amps * 4.0 * case["strings"]}
    if kind == "gates":
        return {"bytes": 16.0 * amps, "flops": amps * _flops_per_amp(_mixed(case))}
    if kind == "density":
        amps = float(rows) * (1 << (2 * n))
        return {"bytes": 16.0 * amps, "flops": amps * case["layers"] * n * (28.0 + 32.0)}
    return {"bytes": 8.0 * amps + 8.0 * rows * case["shots"], "flops": 3.0 * amps}


# ---------------------------------------------------------------------------
# the same in 64 bits, plain torch
# ---------------------------------------------------------------------------
_PAULI = {"x": torch.tensor([[0, 1], [1, 0]], dtype=torch.complex128),
          "y": torch.tensor([[0, -1j], [1j, 0]], dtype=torch.complex128),
          "z": torch.tensor([[1, 0], [0, -1]], dtype=torch.complex128)}


def _matrix(name, a):
    """[..., 2, 2] complex128 of a one-wire gate; a: [..., P] angles in float64."""
    if name == "hadamard":
        return torch.tensor([[1, 1], [1, -1]], dtype=torch.complex128, device=GPU) / math.sqrt(2)
    if name == "u3":
        t, p, m = a[..., 0], a[..., 1], a[..., 2]
        c, s = torch.cos(t / 2), torch.sin(t / 2)
        e = [c, -torch.exp(1j * m) * s, torch.exp(1j * p) * s, torch.exp(1j * (p + m)) * c]
        return torch.stack([x.to(torch.complex128) for x in e], -1).reshape(a.shape[:-1] + (2, 2))
    half = a[..., 0, None, None] / 2
    return torch.cos(half) * torch.eye(2, dtype=torch.complex128, device=GPU) - \
        1j * torch.sin(half) * _PAULI[name[1]].to(GPU)


def _wire_pair(psi, n, w):
    """The two halves of every amplitude pair of wire w, as views."""
    v = psi.view(psi.shape[0], 1 << w, 2, -1)
    return v[:, :, 0], v[:, :, 1]


def _one_wire(psi, n, w, u):
    a, b = _wire_pair(psi, n, w)
    u = u.reshape((-1, 1, 1, 2, 2)) if u.dim() == 3 else u
    a0 = a.clone()
    a.mul_(u[..., 0, 0]).add_(u[..., 0, 1] * b)
    b.mul_(u[..., 1, 1]).add_(u[..., 1, 0] * a0)


def _where(psi, n, bits):
    """View of the amplitudes with the given {wire: value}."""
    return psi.view([psi.shape[0]] + [2] * n)[tuple([slice(None)] + [bits.get(w, slice(None)) for w in range(n)])]


def _swap_parts(psi, n, p, q):
    a, b = _where(psi, n, p), _where(psi, n, q)
    t = a.clone()
    a.copy_(b)
    b.copy_(t)


def _k_wires(psi, n, wires, u):
    k = len(wires)
    v = psi.view([psi.shape[0]] + [2] * n)
    axes = [1 + w for w in wires]
    t = v.movedim(axes, list(range(1 + n - k, 1 + n)))
    shape = t.shape
    t = (t.reshape(-1, 1 << k) @ u.mT.contiguous()).reshape(shape)
    v.copy_(t.movedim(list(range(1 + n - k, 1 + n)), axes))


def _gate(psi, n, name, wires, a, dense=None):
    """One gate in place; a: its angles, [P] or [rows, P], float64."""
    if name == "cnot":
        _swap_parts(psi, n, {wires[0]: 1, wires[1]: 0}, {wires[0]: 1, wires[1]: 1})
    elif name == "cz":
        _where(psi, n, {wires[0]: 1, wires[1]: 1}).neg_()
    elif name == "swap":
        _swap_parts(psi, n, {wires[0]: 0, wires[1]: 1}, {wires[0]: 1, wires[1]: 0})
    elif name == "toffoli":
        c = {wires[0]: 1, wires[1]: 1}
        _swap_parts(psi, n, {**c, wires[2]: 0}, {**c, wires[2]: 1})
    elif name == "cswap":
        c = {wires[0]: 1}
        _swap_parts(psi, n, {**c, wires[1]: 0, wires[2]: 1}, {**c, wires[1]: 1, wires[2]: 0})
    elif name == "crx":
        u = torch.eye(4, dtype=torch.complex128, device=GPU)
        u[2:, 2:] = _matrix("rx", a)
        _k_wires(psi, n, wires, u)
    elif name in ("rzz", "rxx"):
        p = _PAULI[name[1]].to(GPU)
        u = torch.cos(a[0] / 2) * torch.eye(4, dtype=torch.complex128, device=GPU) - \
            1j * torch.sin(a[0] / 2) * torch.kron(p, p)
        _k_wires(psi, n, wires, u)
    elif name.startswith("dense"):
        _k_wires(psi, n, wires, dense)
    else:
        _one_wire(psi, n, wires[0], _matrix(name, a))


def _basis(rows, n):
    psi = torch.zeros(rows, 1 << n, dtype=torch.complex128, device=GPU)
    psi[:, 0] = 1
    return psi


def _forward(psi, n, prog, theta, dense=None):
    for i, (name, wires, cols) in enumerate(prog):
        a = theta[cols[0]:cols[-1] + 1] if cols else None
        _gate(psi, n, name, wires, a, dense.get(i) if dense else None)
    return psi


def _z_all(psi, n):
    p = psi.real ** 2 + psi.imag ** 2
    out = []
    for w in range(n):
        v = p.view(p.shape[0], 1 << w, 2, -1).sum((1, 3))
        out.append(v[:, 0] - v[:, 1])
    return torch.stack(out, 1)


def _apply_string(psi, n, string):
    """P psi for one Pauli string."""
    x = z = ny = 0
    for w, c in enumerate(string):
        bit = 1 << (n - 1 - w)
        x |= bit if c in "XY" else 0
        z |= bit if c in "ZY" else 0
        ny += c == "Y"
    src = torch.arange(1 << n, device=GPU) ^ x
    par = src & z
    for sh in (16, 8, 4, 2, 1):
        par = par ^ (par >> sh)
    return psi[:, src] * ((1 - 2 * (par & 1)).double() * (1j ** (ny % 4)))


def _reverse(psi, lam, n, prog, theta):
    """Gradients of RX, RY, RZ angles: Im <lam|P|psi> / 2 after each gate, both states un-applied as the sweep goes."""
    out = torch.zeros_like(theta)
    for name, wires, cols in reversed(prog):
        if cols:
            p, (l0, l1) = _PAULI[name[1]].to(GPU), _wire_pair(lam, n, wires[0])
            x0, x1 = _wire_pair(psi, n, wires[0])
            d = [(l.conj() * x).sum() for l, x in ((l0, x0), (l0, x1), (l1, x0), (l1, x1))]
            out[cols[0]] = (d[0] * p[0, 0] + d[1] * p[0, 1] + d[2] * p[1, 0] + d[3] * p[1, 1]).imag / 2
        for v in (psi, lam):
            _gate(v, n, name, wires, -theta[cols[0]:cols[-1] + 1] if cols else None)
    return out


def exact(case, seed):
    kind, g = case["kind"], _generator(seed)
    n, rows = case.get("n"), case.get("rows")
    most = EXACT_AMPS << 2 if kind in ("energy", "gates") else EXACT_AMPS           # few passes over the state
    if kind == "shots" or (n and rows and rows << (2 * n if kind == "density" else n) > most):
        return None
    if kind == "batch":
        circuits = _uneven(case)
        theta = _angles(g, max(_columns(p) for _, p in circuits)).double()
        return torch.stack([_z_all(_forward(_basis(1, m), m, p, theta), m)[0, 0] for m, p in circuits])
    if kind in ("layers", "replay"):
        prog = _brick(n, case["layers"]) if kind == "layers" else _u3_ring(n, case["layers"])
        return _z_all(_forward(_basis(rows, n), n, prog, _angles(g, _columns(prog)).double()), n)
    if kind == "gradient":
        prog = _ansatz(n, case["layers"])
        theta = _angles(g, _columns(prog), 0.1).double()
        phi = (torch.rand(rows, 1, device=GPU, generator=g) * math.pi).double()
        psi = _basis(rows, n)
        for w in range(n):
            _one_wire(psi, n, w, _matrix("ry", phi))
        _forward(psi, n, prog, theta)
        lam = torch.zeros_like(psi)
        for string, weight in zip(*_loss_terms(n)):
            lam += weight * _apply_string(psi, n, string)
        loss = (psi.conj() * lam).sum().real / rows
        return {"loss": loss, "gradient": _reverse(psi, lam.mul_(2.0 / rows), n, prog, theta)}
    if kind == "training":
        prog = _ansatz(n, case["layers"])
        theta = _angles(g, _columns(prog)).double()
        weight = (torch.randn(4, n, device=GPU, generator=g) * 0.5).double().requires_grad_()
        bias = (torch.randn(4, device=GPU, generator=g) * 0.1).double().requires_grad_()
        x = (torch.rand(rows, n, device=GPU, generator=g) * math.pi).double()
        y = torch.randint(0, 4, (rows,), device=GPU, generator=g)
        psi = _basis(rows, n)
        for w in range(n):
            _one_wire(psi, n, w, _matrix("ry", x[:, w:w + 1]))
        _forward(psi, n, prog, theta)
        z = _z_all(psi, n).requires_grad_()
        logits = z @ weight.T + bias
        loss = torch.nn.functional.cross_entropy(logits, y)
        gz, gw, gb = torch.autograd.grad(loss, (z, weight, bias))
        lam = torch.zeros_like(psi)
        for w in range(n):
            (a, b), (p, q) = _wire_pair(lam, n, w), _wire_pair(psi, n, w)
            a.add_(p * (2 * gz[:, w, None, None]))
            b.sub_(q * (2 * gz[:, w, None, None]))
        return {"logits": logits.detach(), "loss": loss.detach(), "head": [gw, gb],
                "ansatz": _reverse(psi, lam, n, prog, theta)}
    if kind == "energy":
        psi = _random_states(g, rows, n).to(torch.complex128)
        grad, each = torch.zeros_like(psi), []
        for string, weight in _strings(case):
            p = _apply_string(psi, n, string)
            each.append((psi.conj() * p).sum(1).real)
            grad += (2 * weight) * p
        if not case["grad"]:
            return torch.stack(each, 1)
        return {"energy": sum(w * e for (_, w), e in zip(_strings(case), each)), "gradient": grad}
    if kind == "gates":
        prog = _mixed(case)
        theta = _angles(g, _columns(prog)).double()
        dense = {i: u.to(torch.complex128) for i, u in _dense(g, prog).items()}
        return _forward(_random_states(g, rows, n).to(torch.complex128), n, prog, theta, dense)
    # density: vec(rho) on 2n wires, U on the row wires and conj(U) on the column wires
    prog = _ansatz(n, case["layers"])
    theta = _angles(g, _columns(prog)).double()
    rho = _basis(rows, 2 * n)
    for name, wires, cols in prog:
        if cols:
            u = _matrix(name, theta[cols[0]:cols[0] + 1])
            _one_wire(rho, 2 * n, wires[0], u)
            _one_wire(rho, 2 * n, wires[0] + n, u.conj())
            continue
        _gate(rho, 2 * n, "cnot", wires, None)
        _gate(rho, 2 * n, "cnot", tuple(w + n for w in wires), None)
        if wires[1] == 0:
            eye = torch.eye(2, dtype=torch.complex128)
            channel = sum(f * torch.kron(k, k.conj()) for f, k in
                          [(1 - 0.02, eye)] + [(0.02 / 3, _PAULI[p]) for p in "xyz"]).to(GPU)
            for w in range(n):
                _k_wires(rho, 2 * n, (w, w + n), channel)
    probs = torch.diagonal(rho.view(rows, 1 << n, 1 << n), dim1=1, dim2=2).real
    z = [probs.reshape(rows, 1 << w, 2, -1).sum((1, 3)) for w in range(n)]
    return {"densities": rho.reshape([rows] + [2] * (2 * n)), "z": torch.stack([v[:, 0] - v[:, 1] for v in z], 1)}
