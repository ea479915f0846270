"""Timed cases: what a user of unitair_amd runs, over the sizes it is used at.

A case is a dict of plain values.  `listed` names the fixed ones, `draw` gives
one more of the same ranges, `prepare` makes on the GPU what a program holds
before the call, `run` is one pass through the public entry points, `work` is
what a pass cannot do without and `exact` its result in 64 bits from plain
torch.

Families ("path" of a case):
  layer_calls  a small circuit written as drop-in calls, one after another
  gate         one apply_operator call (1 to 10 target qubits, one operator, or
               one operator per state)
  all_qubits   apply_all_qubits
  to_qubits    apply_to_qubits with one gate on each listed qubit
  phase        apply_phase with one angle vector for a batch of states
  index_maps   permute_qubits, swap and multi_cz
  gate_grad    apply_operator forward and backward through autograd
  circuit      a mixed circuit as a compiled FusedProgram
  blocks       a 4/5-qubit dense-block circuit (CircuitRunner, dense_blocks)
  adjoint      loss and all gradients of a batched rotation circuit
"""
import math
import os
import random
import sys

import numpy as np
import torch

_PKG = os.path.join(os.getcwd(), "qcware-unitair_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

from unitair_amd import adjoint, simulation, workloads  # noqa: E402
from unitair_amd.circuits import Circuit, CircuitRunner, Gate  # noqa: E402
from unitair_amd.fusion import FusedProgram  # noqa: E402

_DTYPES = {"c64": torch.complex64, "c128": torch.complex128}
_REAL = {"c64": torch.float32, "c128": torch.float64}
_BYTES = {"c64": 8, "c128": 16}

_CNOT = np.array([[1, 0, 0, 0], [0, 1, 0, 0], [0, 0, 0, 1], [0, 0, 1, 0]], dtype=np.complex128)


# -------------------------------------------------------------------- cases --

def listed():
    return [
        # the smallest calls: one layer of the 12-qubit, batch-8 parity circuit
        # as a program writes it, 12 one-qubit gates, 6 CNOTs and a phase; the
        # states are a few hundred kilobytes, so what counts is the call itself
        {"name": "layer_calls_12q_b8_c128", "path": "layer_calls", "n": 12, "batch": 8,
         "dtype": "c128"},
        # one gate of the 24-qubit benchmark circuit through the drop-in call
        {"name": "gate_2q_24q_c64", "path": "gate", "n": 24, "batch": 1, "k": 2,
         "per_state": False, "dtype": "c64", "layout": 3},
        # many small circuits side by side, each with its own operator (the
        # use that unitair's tutorial leads with): small states, an odd batch
        {"name": "gate_2q_10q_b3001_per_state_c64", "path": "gate", "n": 10, "batch": 3001,
         "k": 2, "per_state": True, "dtype": "c64", "layout": 5},
        # a wide block (an oracle or a fused sub-circuit) on the benchmark state
        {"name": "gate_8q_24q_c64", "path": "gate", "n": 24, "batch": 1, "k": 8,
         "per_state": False, "dtype": "c64", "layout": 7},
        # the same in double precision, which reference runs use
        {"name": "gate_7q_22q_c128", "path": "gate", "n": 22, "batch": 1, "k": 7,
         "per_state": False, "dtype": "c128", "layout": 11},
        # a Hadamard-like layer on every qubit of the benchmark state
        {"name": "all_qubits_24q_c64", "path": "all_qubits", "n": 24, "batch": 1,
         "dtype": "c64"},
        # a cost layer: one diagonal, a batch of states (an odd number of them)
        {"name": "phase_16q_b301_c64", "path": "phase", "n": 16, "batch": 301, "dtype": "c64"},
        # relabelling and entangling without arithmetic on the benchmark state
        {"name": "index_maps_24q_c64", "path": "index_maps", "n": 24, "batch": 1,
         "dtype": "c64", "layout": 13},
        # training step of one gate: output, gradient of the state and of the
        # operator
        {"name": "gate_grad_2q_22q_b3_c64", "path": "gate_grad", "n": 22, "batch": 3, "k": 2,
         "dtype": "c64", "layout": 17},
        # the 24-qubit, 200-gate benchmark circuit
        {"name": "circuit_24q_200_c64", "path": "circuit", "n": 24, "batch": 1, "gates": 200,
         "dtype": "c64", "layout": 2},
        # the dense-block benchmark circuit, two qubits under its full size
        {"name": "blocks_26q_80_c64", "path": "blocks", "n": 26, "gates": 80, "dtype": "c64",
         "layout": 4},
        # the batched gradient workload at its benchmark size
        {"name": "adjoint_16q_b1024_l10_c64", "path": "adjoint", "n": 16, "batch": 1024,
         "layers": 10, "dtype": "c64"},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _batch_for(rng, n, amps_lo, amps_hi):
    """A batch for which batch * 2^n lies between the two sizes (at least 1)."""
    lo = max(1, amps_lo >> n)
    hi = max(lo, amps_hi >> n)
    return _log_int(rng, lo, hi)


def draw(rng: random.Random):
    path = rng.choice(["layer_calls", "gate", "gate", "gate", "gate", "all_qubits", "to_qubits",
                       "phase", "index_maps", "gate_grad", "circuit", "blocks", "adjoint"])
    dt = rng.choice(["c64", "c64", "c128"])
    layout = rng.randrange(1 << 30)
    if path == "layer_calls":
        return {"path": path, "n": rng.randint(8, 16), "batch": _log_int(rng, 1, 33),
                "dtype": dt}
    if path == "gate":
        if rng.random() < 0.3:       # one operator per state
            n = rng.randint(7, 14)
            return {"path": path, "n": n, "batch": _batch_for(rng, n, 1 << 16, 1 << 24),
                    "k": rng.randint(1, 3), "per_state": True, "dtype": dt, "layout": layout}
        if rng.random() < 0.5:       # ordinary gates, small states to large ones
            n = rng.randint(10, 26)
            return {"path": path, "n": n, "batch": _batch_for(rng, n, 1 << 14, 1 << 24),
                    "k": rng.randint(1, 5), "per_state": False, "dtype": dt, "layout": layout}
        k = rng.randint(6, 10)       # wide blocks
        n = rng.randint(14, 24)
        top = (1 << 33) >> k         # at most 2^33 multiply-adds
        return {"path": path, "n": n,
                "batch": _batch_for(rng, n, 1 << 18, min(1 << 24, max(1 << 18, top))), "k": k,
                "per_state": False, "dtype": dt, "layout": layout}
    if path in ("all_qubits", "to_qubits"):
        n = rng.randint(12, 25)
        case = {"path": path, "n": n, "batch": _batch_for(rng, n, 1 << 16, 1 << 24),
                "dtype": dt}
        if path == "to_qubits":
            case.update(gates=rng.randint(2, n), layout=layout)
        return case
    if path == "phase":
        n = rng.randint(8, 22)
        return {"path": path, "n": n, "batch": _batch_for(rng, n, 1 << 16, 1 << 25),
                "dtype": dt}
    if path == "index_maps":
        n = rng.randint(10, 25)
        return {"path": path, "n": n, "batch": _batch_for(rng, n, 1 << 16, 1 << 24),
                "dtype": dt, "layout": layout}
    if path == "gate_grad":
        n = rng.randint(10, 23)
        return {"path": path, "n": n, "batch": _batch_for(rng, n, 1 << 16, 1 << 23),
                "k": rng.randint(1, 4), "dtype": dt, "layout": layout}
    if path == "circuit":
        n = rng.randint(14, 25)
        return {"path": path, "n": n, "batch": _batch_for(rng, n, 1 << 14, 1 << 22),
                "gates": rng.randint(40, 200), "dtype": dt, "layout": layout}
    if path == "blocks":
        return {"path": path, "n": rng.randint(16, 25), "gates": rng.randint(10, 80),
                "dtype": dt, "layout": layout}
    n = rng.randint(8, 18)
    return {"path": "adjoint", "n": n, "batch": _batch_for(rng, n, 1 << 16, 1 << 24),
            "layers": rng.randint(2, 10), "dtype": dt}


# ----------------------------------------------------------------- inputs ----

def _gen(seed, salt):
    g = torch.Generator(device="cuda")
    g.manual_seed((int(seed) * 1000003 + salt * 7919 + 12345) & 0x7fffffffffff)
    return g


def _states(case, seed, salt=0):
    """Normalised random states, (batch, 2^n), or (2^n,) for a batch of one."""
    n, batch = case["n"], case.get("batch", 1)
    real = _REAL[case["dtype"]]
    shape = (2 ** n, 2) if batch == 1 else (batch, 2 ** n, 2)
    x = torch.randn(shape, generator=_gen(seed, salt), device="cuda", dtype=real)
    x = torch.view_as_complex(x)
    return x / torch.linalg.vector_norm(x, dim=-1, keepdim=True)


def _unitaries(shape, dim, seed, salt, dtype):
    """Haar-random unitaries: Gaussian columns, orthonormalised one after the
    other (few wide matrices by QR, with R's diagonal made positive)."""
    rng = np.random.default_rng([int(seed), salt])
    m = rng.standard_normal(shape + (dim, dim)) + 1j * rng.standard_normal(shape + (dim, dim))
    if dim > 8:
        q, r = np.linalg.qr(m)
        d = np.diagonal(r, axis1=-2, axis2=-1)
        q = q * (d / np.abs(d))[..., None, :]
    else:
        q = np.zeros_like(m)
        for c in range(dim):
            v = m[..., c]
            for _ in range(2):       # twice: orthogonal to rounding
                v = v - (q * (q.conj() * v[..., :, None]).sum(-2)[..., None, :]).sum(-1)
            q[..., c] = v / np.linalg.norm(v, axis=-1, keepdims=True)
    return torch.from_numpy(np.ascontiguousarray(q)).to("cuda", _DTYPES[dtype])


def _angles(shape, seed, salt, dtype):
    return torch.rand(shape, generator=_gen(seed, salt), device="cuda",
                      dtype=_REAL[dtype]) * (2 * math.pi)


def _qubits(case, k):
    """The gate's qubits, in the order the program lists them."""
    return random.Random(case["layout"]).sample(range(case["n"]), k)


def _layer_gates(case, seed):
    """One layer as (operator, qubits) pairs and the angles of its phase."""
    n = case["n"]
    ops = _unitaries((n,), 2, seed, 1, case["dtype"])
    gates = [(ops[q], [q]) for q in range(n)]
    cnot = torch.from_numpy(_CNOT).to("cuda", _DTYPES[case["dtype"]])
    gates += [(cnot, [i, i + 1]) for i in range(0, n - 1, 2)]
    phi = np.random.default_rng([int(seed), 2]).uniform(0, 2 * np.pi, 2)
    angles = workloads.single_qubit_phase_angles(n, n // 2, *phi)
    return gates, torch.from_numpy(angles).to("cuda", _REAL[case["dtype"]])


def _circuit(case, seed):
    """The benchmark's gate mix: 60 % 1-qubit, 10 % each CNOT, CZ, 2-qubit and
    full-length phases, placed by the case and filled from the seed."""
    n, total = case["n"], case["gates"]
    place = random.Random(case["layout"])
    each = total // 10
    kinds = ["cnot", "cz", "dense2", "phase"] * each
    kinds += ["dense1"] * (total - len(kinds))
    place.shuffle(kinds)
    m1 = _unitaries((total,), 2, seed, 3, "c128").cpu().numpy()
    m2 = _unitaries((total,), 4, seed, 4, "c128").cpu().numpy()
    gates = []
    for i, kind in enumerate(kinds):
        if kind == "dense1":
            gates.append(Gate("dense", (place.randrange(n),), matrix=m1[i]))
        elif kind == "dense2":
            gates.append(Gate("dense", tuple(place.sample(range(n), 2)), matrix=m2[i]))
        elif kind == "phase":
            gates.append(Gate("phase", (), angles=_angles((2 ** n,), seed, 100 + i,
                                                          case["dtype"])))
        else:
            gates.append(Gate(kind, tuple(place.sample(range(n), 2))))
    return Circuit(n, gates)


def _blocks(case, seed):
    """Four 5-qubit gates to each 4-qubit one, as in the benchmark."""
    place = random.Random(case["layout"])
    n, total = case["n"], case["gates"]
    sizes = [4 if i % 5 == 4 else 5 for i in range(total)]
    place.shuffle(sizes)
    m5 = _unitaries((total,), 32, seed, 5, "c128").cpu().numpy()
    m4 = _unitaries((total,), 16, seed, 6, "c128").cpu().numpy()
    return Circuit(n, [Gate("dense", tuple(place.sample(range(n), k)),
                            matrix=(m5 if k == 5 else m4)[i]) for i, k in enumerate(sizes)])


def _maps(case):
    """A qubit order, a pair to swap and a ring of CZ pairs."""
    n = case["n"]
    place = random.Random(case["layout"])
    perm = place.sample(range(n), n)
    pair = tuple(place.sample(range(n), 2))
    ring = [(q, (q + 1) % n) for q in range(n)]
    return perm, pair, ring


def prepare(case, seed):
    path, dtype = case["path"], case["dtype"]
    st = {"path": path, "n": case["n"]}
    if path == "layer_calls":
        st["psi"] = _states(case, seed)
        st["gates"], st["angles"] = _layer_gates(case, seed)
    elif path in ("gate", "gate_grad"):
        k = case["k"]
        st["psi"] = _states(case, seed)
        shape = (case["batch"],) if case.get("per_state") and case["batch"] > 1 else ()
        st["op"] = _unitaries(shape, 2 ** k, seed, 1, dtype)
        st["qubits"] = _qubits(case, k)
        if path == "gate_grad":
            st["psi"].requires_grad_(True)
            st["op"].requires_grad_(True)
            st["grad"] = _states(case, seed, 1)
    elif path == "all_qubits":
        st["psi"] = _states(case, seed)
        st["op"] = _unitaries((), 2, seed, 1, dtype)
    elif path == "to_qubits":
        st["psi"] = _states(case, seed)
        st["qubits"] = _qubits(case, case["gates"])
        st["ops"] = list(_unitaries((case["gates"],), 2, seed, 1, dtype))
    elif path == "phase":
        st["psi"] = _states(case, seed)
        st["angles"] = _angles((2 ** case["n"],), seed, 1, dtype)
    elif path == "index_maps":
        st["psi"] = _states(case, seed)
        st["perm"], st["pair"], ring = _maps(case)
        st["ring"] = torch.tensor(ring, device="cuda")
    elif path == "circuit":
        st["psi"] = _states(case, seed)
        st["program"] = FusedProgram(_circuit(case, seed), dtype=_DTYPES[dtype], compiled=True)
    elif path == "blocks":
        st["psi"] = _states(case, seed)
        st["runner"] = CircuitRunner(_blocks(case, seed), dtype=_DTYPES[dtype],
                                     dense_blocks=True)
    else:
        shape = (case["batch"], case["layers"], case["n"])
        for i, name in enumerate(("theta", "phi")):
            st[name] = _angles(shape, seed, 1 + i, dtype).requires_grad_(True)
        st["dtype"] = _DTYPES[dtype]
    return st


# ------------------------------------------------------------------- a pass --

def run(st):
    path = st["path"]
    if path == "layer_calls":
        x = st["psi"]
        for op, qubits in st["gates"]:
            x = simulation.apply_operator(op, qubits, x)
        return simulation.apply_phase(st["angles"], x)
    if path == "gate":
        return simulation.apply_operator(st["op"], st["qubits"], st["psi"])
    if path == "gate_grad":
        out = simulation.apply_operator(st["op"], st["qubits"], st["psi"])
        g_op, g_psi = torch.autograd.grad(out, (st["op"], st["psi"]), st["grad"])
        return out.detach(), g_op, g_psi
    if path == "all_qubits":
        return simulation.apply_all_qubits(st["op"], st["psi"])
    if path == "to_qubits":
        return simulation.apply_to_qubits(st["ops"], st["qubits"], st["psi"])
    if path == "phase":
        return simulation.apply_phase(st["angles"], st["psi"])
    if path == "index_maps":
        return (simulation.permute_qubits(st["perm"], st["psi"]),
                simulation.swap(st["psi"], st["pair"]),
                simulation.multi_cz(st["ring"], st["psi"]))
    if path == "circuit":
        return st["program"].run(st["psi"].clone())      # runs in place: a fresh input each
    if path == "blocks":
        return st["runner"].run(st["psi"].clone())
    loss = adjoint.sum_z_loss(st["theta"], st["phi"], st["n"], st["dtype"], compiled=True)
    g_theta, g_phi = torch.autograd.grad(loss.sum(), (st["theta"], st["phi"]))
    return loss.detach(), g_theta, g_phi


# --------------------------------------------------------------------- work --

def work(case):
    """Bytes and operations of a pass: the inputs read once, the outputs
    written once (8 flops to a complex multiply-add, 6 to a multiply)."""
    path, n, b = case["path"], case["n"], _BYTES[case["dtype"]]
    amps = case.get("batch", 1) << n
    state = amps * b
    if path == "layer_calls":     # a chain of calls, each with a tensor as its result
        calls = n + len(range(0, n - 1, 2))
        return {"bytes": 2 * state * (calls + 1) + (b // 2 << n),
                "flops": amps * (16 * n + 32 * (calls - n) + 6)}
    if path == "gate":
        ops = (case["batch"] if case["per_state"] else 1) * 4 ** case["k"]
        return {"bytes": 2 * state + ops * b, "flops": amps * 8 * 2 ** case["k"]}
    if path == "gate_grad":       # out; grad_psi and grad_op from psi and grad
        return {"bytes": 5 * state, "flops": 3 * amps * 8 * 2 ** case["k"]}
    if path == "all_qubits":
        return {"bytes": 2 * state, "flops": amps * 16 * n}
    if path == "to_qubits":
        return {"bytes": 2 * state, "flops": amps * 16 * case["gates"]}
    if path == "phase":
        return {"bytes": 2 * state + (b // 2 << n), "flops": amps * 6}
    if path == "index_maps":
        return {"bytes": 6 * state, "flops": amps}
    if path == "circuit":
        each = case["gates"] // 10
        ones = case["gates"] - 4 * each
        return {"bytes": 2 * state + each * (b // 2 << n),
                "flops": amps * (16 * ones + 32 * each + 6 * each)}
    if path == "blocks":
        fours = case["gates"] // 5
        return {"bytes": 2 * state,
                "flops": amps * 8 * (16 * fours + 32 * (case["gates"] - fours))}
    # forward, then state and co-state back: three gates' work for each gate;
    # a state that is made from the angles and left behind
    layers = case["layers"]
    params = case["batch"] * layers * n
    return {"bytes": state + 2 * 2 * params * (b // 2),
            "flops": 3 * amps * layers * n * (16 + 6) + 2 * amps * layers * n * 8}


# -------------------------------------------------------------------- exact --

def _order_index(order, n):
    """idx with x[..., idx] = x with its qubits reordered: new qubit q is old
    qubit order[q]."""
    i = torch.arange(2 ** n, device="cuda")
    idx = torch.zeros_like(i)
    for q, p in enumerate(order):
        idx |= ((i >> (n - 1 - q)) & 1) << (n - 1 - p)
    return idx


def _act(op, qubits, x, n):
    """(2^k, 2^k) or (batch, 2^k, 2^k) operator on the listed qubits of (batch, 2^n)."""
    k, batch = len(qubits), x.shape[0]
    idx = _order_index(list(qubits) + [q for q in range(n) if q not in qubits], n)
    y = torch.matmul(op.contiguous(), x[:, idx].reshape(batch, 2 ** k, -1))
    out = torch.empty_like(x)
    out[:, idx] = y.reshape(batch, -1)
    return out


def _rows(x, case):
    return x.to(torch.complex128).reshape(case.get("batch", 1), 2 ** case["n"])


def _like(x, case):
    return x.reshape(-1) if case.get("batch", 1) == 1 else x


def _signs(pairs, n):
    x = torch.arange(2 ** n, device="cuda")
    par = torch.zeros_like(x)
    for a, b in pairs:
        par ^= (x >> (n - 1 - a)) & (x >> (n - 1 - b)) & 1
    return 1.0 - 2.0 * par.to(torch.float64)


def _turn(kind, t, x, n, q):
    """RY(t) or RZ(t) on qubit q of (batch, 2^n), one angle a state."""
    batch = x.shape[0]
    v = x.reshape(batch, 2 ** q, 2, -1)
    c = torch.cos(t / 2).reshape(batch, 1, 1)
    s = torch.sin(t / 2).reshape(batch, 1, 1)
    if kind == "z":
        ph = torch.complex(c, s)
        return torch.stack([v[:, :, 0] * ph.conj(), v[:, :, 1] * ph], 2).reshape(batch, -1)
    return torch.stack([c * v[:, :, 0] - s * v[:, :, 1], s * v[:, :, 0] + c * v[:, :, 1]],
                       2).reshape(batch, -1)


def _adjoint_exact(theta, phi, n):
    """Loss and gradients, a slice of the batch at a time: psi and lam = H psi
    are carried back gate by gate; the derivative of <psi|H|psi> with respect
    to the angle of exp(-i t/2 P) is Im <lam|P|psi> right after the gate."""
    batch, layers, _ = theta.shape
    ring = [(q, (q + 1) % n) for q in range(n)] if n > 2 else [(0, 1)]
    sign = _signs(ring, n)
    x = torch.arange(2 ** n, device="cuda")
    pop = sum(((x >> i) & 1) for i in range(n))
    obs = (n - 2 * pop).to(torch.float64)
    loss = torch.empty(batch, dtype=torch.float64, device="cuda")
    grads = {k: torch.empty_like(theta) for k in "yz"}
    step = max(1, (1 << 25) >> n)
    for lo in range(0, batch, step):
        sl = slice(lo, min(batch, lo + step))
        th, ph = theta[sl], phi[sl]
        psi = torch.zeros(th.shape[0], 2 ** n, dtype=torch.complex128, device="cuda")
        psi[:, 0] = 1
        for l in range(layers):
            for q in range(n):
                psi = _turn("z", ph[:, l, q], psi, n, q)
                psi = _turn("y", th[:, l, q], psi, n, q)
            psi = psi * sign
        loss[sl] = (psi.abs() ** 2 * obs).sum(1)
        both = torch.cat([psi, psi * obs])
        m = th.shape[0]
        for l in reversed(range(layers)):
            both = both * sign
            for kind, ang in (("y", th), ("z", ph)):
                for q in range(n):
                    v = both[:m].reshape(m, 2 ** q, 2, -1)
                    w = both[m:].reshape(m, 2 ** q, 2, -1)
                    if kind == "y":      # P psi = (-i psi1, i psi0)
                        d = -1j * w[:, :, 0].conj() * v[:, :, 1] + \
                            1j * w[:, :, 1].conj() * v[:, :, 0]
                    else:
                        d = w[:, :, 0].conj() * v[:, :, 0] - w[:, :, 1].conj() * v[:, :, 1]
                    grads[kind][sl, l, q] = d.imag.sum((1, 2))
                    t = ang[:, l, q]
                    both = _turn(kind, -torch.cat([t, t]), both, n, q)
    return loss, grads["y"], grads["z"]


def exact(case, seed):
    path, n, dtype = case["path"], case["n"], case["dtype"]
    if path == "adjoint":
        shape = (case["batch"], case["layers"], n)
        th, ph = (_angles(shape, seed, 1 + i, dtype).to(torch.float64) for i in range(2))
        return _adjoint_exact(th, ph, n)
    x = _rows(_states(case, seed), case)
    c128 = torch.complex128
    if path == "layer_calls":
        gates, angles = _layer_gates(case, seed)
        for op, qubits in gates:
            x = _act(op.to(c128), qubits, x, n)
        return _like(x * torch.exp(-1j * angles.to(torch.float64)), case)
    if path in ("gate", "gate_grad"):
        k = case["k"]
        shape = (case["batch"],) if case.get("per_state") and case["batch"] > 1 else ()
        op = _unitaries(shape, 2 ** k, seed, 1, dtype).to(c128)
        qubits = _qubits(case, k)
        out = _act(op, qubits, x, n)
        if path == "gate":
            return _like(out, case)
        g = _rows(_states(case, seed, 1), case)
        g_psi = _act(op.conj().transpose(-1, -2), qubits, g, n)
        idx = _order_index(qubits + [q for q in range(n) if q not in qubits], n)
        gm, xm = (t[:, idx].reshape(t.shape[0], 2 ** k, -1) for t in (g, x))
        g_op = torch.zeros(2 ** k, 2 ** k, dtype=c128, device="cuda")
        for i in range(2 ** k):
            for j in range(2 ** k):
                g_op[i, j] = (gm[:, i] * xm[:, j].conj()).sum()
        return _like(out, case), g_op, _like(g_psi, case)
    if path == "all_qubits":
        op = _unitaries((), 2, seed, 1, dtype).to(c128)
        for q in range(n):
            x = _act(op, [q], x, n)
        return _like(x, case)
    if path == "to_qubits":
        ops = _unitaries((case["gates"],), 2, seed, 1, dtype).to(c128)
        for op, q in zip(ops, _qubits(case, case["gates"])):
            x = _act(op, [q], x, n)
        return _like(x, case)
    if path == "phase":
        return _like(x * torch.exp(-1j * _angles((2 ** n,), seed, 1, dtype).to(torch.float64)),
                     case)
    if path == "index_maps":
        perm, pair, ring = _maps(case)
        swapped = list(range(n))
        swapped[pair[0]], swapped[pair[1]] = pair[1], pair[0]
        outs = [x[:, _order_index(order, n)] for order in (perm, swapped)]
        outs.append(x * _signs(ring, n))
        return tuple(_like(o, case) for o in outs)
    circuit = _circuit(case, seed) if path == "circuit" else _blocks(case, seed)
    for g in circuit.gates:
        if g.kind == "phase":
            x = x * torch.exp(-1j * g.angles.to(torch.float64))
        else:
            x = _act(torch.from_numpy(g.dense_matrix()).to("cuda"), list(g.qubits), x, n)
    return _like(x, case)
