"""The native recording and plan keys (csrc/tqsv_host.cpp) against the general Python path they stand in for."""
import itertools

import numpy as np
import pytest
import torch

import torchquantum_amd as tq
import torchquantum_amd.functional as tqf
from torchquantum_amd import _native as N
from torchquantum_amd import engine as E
from torchquantum_amd import operator as op

NQ, BSZ = 5, 3
WIRES = [0, 4, 5, -1, True, np.int64(2), [1], (2,), [0, 3], (3, 0), [2, 2], [0, 9], [1, 2, 3], np.array([1, 4]), []]
PARAMS = [None, 0.3, [0.1, 0.2, 0.3], torch.tensor(0.4), torch.rand(1), torch.rand(BSZ), torch.rand(1, 1),
          torch.rand(BSZ, 1), torch.rand(1, 3), torch.rand(BSZ, 3), torch.rand(3, BSZ).T, torch.rand(1, 1).double(),
          torch.rand(1, 1).to(torch.complex64), torch.rand(1, 1, requires_grad=True), torch.rand(1, 2)]


def _outcome(f):
    """What a recording leaves behind: the tape entries, or the exception's type and text."""
    q = tq.QuantumDevice(n_wires=NQ, bsz=BSZ, device="cpu")
    try:
        f(q)
    except Exception as e:      # noqa: BLE001 -- compared with the other path's
        return type(e), str(e)
    return [(o.name, o.wires, [type(w) for w in o.wires], o.inverse, o.version, o.conj, o.nonunitary,
             None if o.params is None else (o.params.dtype, tuple(o.params.shape), o.params.tolist())) for o in q._tape]


@pytest.mark.parametrize("name", ["rx", "u3", "hadamard", "cnot", "crx", "toffoli", "multicnot", "swap", "i"])
def test_gates_as_the_general_path_records_them(name):
    params = PARAMS if name in ("rx", "u3", "crx") else [None, torch.rand(1, 1)]
    for w, p, inv in itertools.product(WIRES, params, (False, True, 1)):
        got = _outcome(lambda q: tqf.func_name_dict[name](q, w, params=p, inverse=inv))
        want = _outcome(lambda q: tqf.gate_wrapper(name, q, w, p, inverse=inv))
        assert got == want, (name, w, p, inv)


def _ops():
    """Operators in every state a call can meet them in, and whether the call itself has to run."""
    a, b, c, d, e, f = (op.RX(has_params=True, trainable=True) for _ in range(6))
    b = op.RX()
    b.params = torch.rand(BSZ, 1)                    # a plain tensor instead of a parameter
    c.register_forward_pre_hook(lambda m, i: None)
    d.forward = lambda q_device, wires=None: tqf.rz(q_device, wires, params=torch.ones(1, 1))
    e.func = tqf.ry
    f.inverse = True
    g = op.RX()
    g.params = torch.rand(1)                         # one dimension: the call reshapes it
    return [a, b, c, d, e, f, g, op.Hadamard(), op.RX(), op.I()]


class _Doubled(op.RX):
    def forward(self, q_device, wires=None):
        super().forward(q_device, wires=wires)
        super().forward(q_device, wires=wires)


@pytest.mark.parametrize("record_op", [False, True])
def test_layers_as_the_operator_calls_record_them(record_op):
    for o in _ops() + [_Doubled(has_params=True), op.CNOT()]:
        for w in (2, [2], [0, 3], 7, [1, 1]):
            seen = []
            for each in (True, False):
                torch.manual_seed(0)

                def rec(q):
                    q.record_op = record_op
                    op.apply_each(q, [o], [w]) if each else o(q, wires=w)
                    seen.append((list(q.op_history), o.wires))
                seen.append(_outcome(rec))
            assert seen[:len(seen) // 2] == seen[len(seen) // 2:], (o, w)


def test_hooks_run():
    layer = tq.Op1QAllLayer(op.RY, 4, has_params=True, trainable=True)
    ran = []
    layer.ops_all[2].register_forward_hook(lambda m, i, o: ran.append(m))
    layer(tq.QuantumDevice(n_wires=4, device="cpu"))
    assert ran == [layer.ops_all[2]]
    h = torch.nn.modules.module.register_module_forward_hook(lambda m, i, o: ran.append(m))
    try:
        layer(tq.QuantumDevice(n_wires=4, device="cpu"))
    finally:
        h.remove()
    assert len([m for m in ran if isinstance(m, op.RY)]) == 1 + 4 + 1


def _python_key(tape):
    return tuple((o.name, o.wires, o.inverse, o.conj, None if o.params is None else
                  ("m", o.params.shape) if o.params.is_complex() else
                  (o.params.shape, o.params.requires_grad, o.params.is_cuda, o.params.dtype)) for o in tape)


def test_structure_is_equal_exactly_where_the_plan_is():
    one = [E.TapeOp(nm, w, p, inv, 0, cj) for nm in ("rx", "r", "xr") for w in ((0,), (1,), (0, 1))
           for p in (None, torch.rand(1, 1), torch.rand(1, 1, requires_grad=True), torch.rand(2, 1),
                     torch.rand(1, 1).double(), torch.rand(1, 2, 2).to(torch.complex64),
                     torch.rand(1, 2, 2, requires_grad=True).to(torch.complex64), torch.rand(2, 2).to(torch.complex64))
           for inv in (False, True) for cj in (False, True)]
    tapes = [[]] + [[o] for o in one] + [[one[0], o] for o in one[::7]] + [[o, one[0]] for o in one[::7]]
    keys = [(N.host().structure(t), _python_key(t)) for t in tapes]
    for a, b in itertools.combinations(keys, 2):
        assert (a[0] == b[0]) == (a[1] == b[1])


def test_stale_parameters_and_pointers():
    p = [torch.rand(3, 2), torch.rand(1, 2), torch.rand(4, 6)[:, 1:5:2], torch.rand(2, 3).T]
    tape = [E.TapeOp("u2", (0,), t, False, t._version) for t in p] + [E.TapeOp("hadamard", (0,), None)]
    assert N.host().stale(tape) == -1
    out = np.zeros((4, 3), dtype=np.int64)
    N.host().pointers(tape, np.array([3, 0, 2, 1], dtype=np.int32), out)
    want = [[t.data_ptr(), t.stride(0) if t.shape[0] > 1 else 0, t.stride(1)] for t in (p[3], p[0], p[2], p[1])]
    assert out.tolist() == want
    p[2].add_(1)
    assert N.host().stale(tape) == 2
    for bad in (np.array([4], dtype=np.int32), np.array([-1], dtype=np.int32), np.array([0], dtype=np.int64)):
        with pytest.raises(ValueError):
            N.host().pointers(tape, bad, out)
    for f in (N.host().stale, N.host().structure):
        with pytest.raises(TypeError):
            f([None])


def test_recording_and_planning_without_the_extension(monkeypatch, tmp_path):
    """Where nothing is built, gates and layers are recorded and plans made for the CPU as with the extension;
    only what runs on a GPU asks for it."""
    layers = [tq.Op1QAllLayer(op.U3, 4, has_params=True, trainable=True), tq.Op2QAllLayer(op.CNOT, 4, circular=True),
              tq.EntanglePairwise(op.CRX, 4, has_params=True)]

    def rec(q):
        tqf.rx(q, 1, params=torch.full((1, 1), 0.3))
        q.h(wires=2)
        for layer in layers:
            layer(q)

    want = _outcome(rec)
    monkeypatch.setattr(N, "HOST_PATH", tmp_path / "_tqhost.so")
    monkeypatch.setattr(N, "_host", None)
    assert N.host(False) is N._Unbuilt
    assert len(want) == 13 and _outcome(rec) == want
    q = tq.QuantumDevice(n_wires=4, device="cpu")
    rec(q)
    c = E.compile_tape(q._tape, 4, 1, E.EngineOptions(), "cpu")
    assert c is E.compile_tape(list(q._tape), 4, 1, E.EngineOptions(), "cpu")
    q._tape[0].params.add_(1)
    with pytest.raises(RuntimeError, match="modified in place"):
        q.flush()


@pytest.mark.parametrize("layer", [lambda: tq.Op1QAllLayer(op.RX, 6, has_params=True),
                                   lambda: tq.EntanglePairwise(op.CNOT, 7)])
def test_layers_with_too_few_ops(layer):
    """A list shorter than the wires raises as its index does, after the gates that it has."""
    layer, q = layer(), tq.QuantumDevice(n_wires=7, device="cpu")
    assert len(layer.ops_all) == 6
    del layer.ops_all[4:]
    with pytest.raises(IndexError):
        layer(q)
    assert len(q._tape) == 4


def test_layers_that_go_over_their_ops():
    """The templates that run the ops they have do so with more and with fewer of them."""
    ring = tq.Op2QAllLayer(op.CNOT, 5, circular=True)
    rand = tq.RandomLayer([0, 1, 2], n_ops=6, seed=1)
    del ring.ops_all[3:], rand.op_list[4:]
    q = tq.QuantumDevice(n_wires=5, device="cpu")
    ring(q)
    assert [o.wires for o in q._tape] == [(0, 1), (1, 2), (2, 3)]
    rand(q)
    assert len(q._tape) == 3 + 4
    one = tq.Op1QAllLayer(op.RX, 3, has_params=True)
    one.ops_all.append(op.RX(has_params=True))
    one(q)
    assert len(q._tape) == 3 + 4 + 3


def test_replaced_module_calls_run(monkeypatch):
    """Tracers replace nn.Module's own call and attribute look-up while they run: a layer's ops go through them."""
    layer = tq.Op1QAllLayer(op.RY, 3, has_params=True)
    seen = []
    call, get = torch.nn.Module.__call__, torch.nn.Module.__getattr__
    with monkeypatch.context() as m:
        m.setattr(torch.nn.Module, "__call__", lambda self, *a, **k: (seen.append(self), call(self, *a, **k))[1])
        layer(tq.QuantumDevice(n_wires=3, device="cpu"))
    assert seen == [layer, *layer.ops_all]
    seen.clear()
    with monkeypatch.context() as m:
        m.setattr(torch.nn.Module, "__getattr__", lambda self, k: (seen.append((self, k)), get(self, k))[1])
        layer(tq.QuantumDevice(n_wires=3, device="cpu"))
    assert [s for s in seen if s[1] == "params"] == [(o, "params") for o in layer.ops_all]


class _Computed(op.RX):
    params = property(lambda self: 2 * self._parameters["params"])


class _Watched(op.RX):
    def __getattribute__(self, k):
        return torch.ones(1, 1) if k == "params" else super().__getattribute__(k)


@pytest.mark.parametrize("cls", [_Computed, _Watched])
def test_computed_parameters_are_asked_for(cls):
    o = op.RX(has_params=True, init_params=[0.25])
    o.__class__ = cls
    q = tq.QuantumDevice(n_wires=2, device="cpu")
    op.apply_each(q, [o], [1])
    assert float(q._tape[0].params) == (0.5 if cls is _Computed else 1.0)


@pytest.mark.parametrize("what", ["history", "global hook"])
def test_hooks_that_turn_on_observation(what):
    """What a hook of one op turns on applies to the ops after it in the layer."""
    layer, q, ran, handles = tq.Op1QAllLayer(op.RY, 4, has_params=True), tq.QuantumDevice(n_wires=4, device="cpu"), [], []

    def hook(m, i):
        if what == "history":
            q.record_op = True
        else:
            handles.append(torch.nn.modules.module.register_module_forward_hook(lambda m, i, o: ran.append(m)))

    layer.ops_all[1].register_forward_pre_hook(hook)
    try:
        layer(q)
    finally:
        for h in handles:
            h.remove()
    if what == "history":
        assert [h["wires"] for h in q.op_history] == [1, 2, 3]
    else:
        assert [m for m in ran if isinstance(m, op.RY)][-2:] == list(layer.ops_all)[2:]
