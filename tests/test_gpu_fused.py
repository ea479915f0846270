"""Fused passes (ua_run_fused_pass via unitair_amd.fusion) against the oracle."""
import numpy as np
import pytest
import torch

from unitair_amd.fusion import FusedProgram
from unitair_amd.gates import haar_unitary
from unitair_amd.initializations import seeded_state_np
from oracle import circuits as oc
from oracle import unitair_np as U
from test_fusion_plan import random_mixed_circuit

pytestmark = pytest.mark.gpu
TOL = {torch.complex64: 1e-5, torch.complex128: 1e-12}


def rel_err(out, ref):
    return float(np.max(np.abs(out - ref)) / max(1e-300, np.max(np.abs(ref))))


@pytest.mark.parametrize("dt", [torch.complex64, torch.complex128])
@pytest.mark.parametrize("n,batch", [(4, 3), (5, 1), (8, 2), (11, 1), (12, 3), (13, 1), (16, 2), (20, 1)])
def test_fused_random_circuits(device, dt, n, batch):
    circ = random_mixed_circuit(n, 80, seed=n * 7 + batch)
    prog = FusedProgram(circ, dtype=dt, device=device)
    psi = seeded_state_np(n, (batch,), seed=n)
    ref = np.stack([oc.run_closed_form(circ.gates, p) for p in psi])
    x = torch.from_numpy(psi).to(device, dt)
    out = prog.run(x).cpu().numpy()
    assert rel_err(out, ref) < TOL[dt] * 10, (prog.num_passes, n)
    assert np.max(U.fidelity_error(ref, out)) < TOL[dt]


def test_fused_layered_12q_batch8_c128(device):
    from unitair_amd.workloads import layered_circuit_12q
    circ = layered_circuit_12q(seed=1)
    psi = seeded_state_np(12, (8,), seed=11)
    ref = np.stack([oc.run_closed_form(circ.gates, p) for p in psi])
    prog = FusedProgram(circ, dtype=torch.complex128, device=device)
    out = prog.run(torch.from_numpy(psi).to(device)).cpu().numpy()
    assert rel_err(out, ref) < 1e-12


@pytest.mark.parametrize("dt", [torch.complex64, torch.complex128])
def test_fused_random_circuit_24q(device, dt):
    from test_gpu_parity import _circuit_24q_and_oracle
    circ, psi, ref = _circuit_24q_and_oracle()
    prog = FusedProgram(circ, dtype=dt, device=device)
    out = prog.run(torch.from_numpy(psi).to(device, dt)).cpu().numpy()
    fid = float(U.fidelity_error(ref, out))
    mae = U.max_abs_error(ref, out)
    print(f"fused 24q {dt}: {prog.num_passes} passes, fidelity error {fid:.3e}, max-abs {mae:.3e}")
    # achieved: complex64 ~3e-13 / ~6e-10, complex128 ~1e-16 / ~1e-17
    bar = {torch.complex64: (1e-10, 1e-7), torch.complex128: (1e-14, 1e-14)}[dt]
    assert fid < bar[0] and mae < bar[1], (fid, mae)


def test_fused_graph_replay_matches_eager(device):
    n = 14
    circ = random_mixed_circuit(n, 60, seed=5)
    prog = FusedProgram(circ, dtype=torch.complex64, device=device)
    psi = torch.from_numpy(seeded_state_np(n, (2,), seed=3)).to(device, torch.complex64)
    eager = prog.run(psi.clone())
    state = psi.clone()
    prog.capture(state)
    for _ in range(3):
        state.copy_(psi)                 # eager work between replays
        torch.cuda.synchronize()
        prog.replay()
        torch.cuda.synchronize()
        assert torch.equal(state, eager)


# ---- compiled passes (ua_compile_fused_pass / ua_run_compiled_pass): the same
# circuits, every pass with 12 tile bits run by its own compiled kernel

@pytest.mark.parametrize("dt", [torch.complex64, torch.complex128])
@pytest.mark.parametrize("n,batch", [(8, 2), (12, 3), (13, 1), (16, 2), (20, 1)])
def test_compiled_random_circuits(device, dt, n, batch):
    """Under 12 qubits the tiles are smaller and the passes stay interpreted."""
    circ = random_mixed_circuit(n, 80, seed=n * 7 + batch)
    prog = FusedProgram(circ, dtype=dt, device=device, compiled=True)
    assert (prog.num_compiled > 0) == (n >= 12)
    psi = seeded_state_np(n, (batch,), seed=n)
    ref = np.stack([oc.run_closed_form(circ.gates, p) for p in psi])
    out = prog.run(torch.from_numpy(psi).to(device, dt)).cpu().numpy()
    assert rel_err(out, ref) < TOL[dt] * 10, (prog.num_passes, n)
    assert np.max(U.fidelity_error(ref, out)) < TOL[dt]


@pytest.mark.parametrize("dt,phase_angles", [(torch.complex64, False),
                                             (torch.complex128, False),
                                             (torch.complex64, True)])
def test_compiled_random_circuit_24q(device, dt, phase_angles):
    from test_gpu_parity import _circuit_24q_and_oracle
    circ, psi, ref = _circuit_24q_and_oracle()
    prog = FusedProgram(circ, dtype=dt, device=device, compiled=True,
                        phase_angles=phase_angles)
    assert prog.num_compiled == prog.num_passes
    out = prog.run(torch.from_numpy(psi).to(device, dt)).cpu().numpy()
    fid = float(U.fidelity_error(ref, out))
    mae = U.max_abs_error(ref, out)
    print(f"compiled 24q {dt} (phase angles: {phase_angles}): {prog.num_passes} passes, "
          f"fidelity error {fid:.3e}, max-abs {mae:.3e}")
    bar = {torch.complex64: (1e-10, 1e-7), torch.complex128: (1e-14, 1e-14)}[dt]
    assert fid < bar[0] and mae < bar[1], (fid, mae)


def _per_state_items(n, batch, seed, device, dt):
    """Gate items of a random mixed circuit plus per-state 1-qubit matrices,
    diagonals and CZ-layer masks (the forms the adjoint and serving loops
    build), on state bits inside and outside the tile."""
    from unitair_amd.fusion import _Item, _items_from_circuit, _merge_1q
    rng = np.random.default_rng(seed)
    items = _merge_1q(_items_from_circuit(random_mixed_circuit(n, 50, seed=seed)))
    items = [it for it in items if it.kind != "wide"]
    for _ in range(40):
        r = rng.random()
        b = int(rng.integers(n))
        if r < 0.4:
            m = np.stack([haar_unitary(2, rng) for _ in range(batch)])
            items.append(_Item("dense1", (b,), torch.from_numpy(m).to(device, dt), True))
        elif r < 0.7:
            d = np.exp(1j * rng.uniform(0, 2 * np.pi, size=(batch, 2)))
            items.append(_Item("diag1", (b,), torch.from_numpy(d).to(device, dt), True))
        elif r < 0.85:
            masks = rng.integers(0, 2 ** (n - 1), size=batch, dtype=np.int64)
            items.append(_Item("cz_layer", (), torch.from_numpy(masks).to(device), True))
        else:
            a, c = rng.choice(n, 2, replace=False)
            items.append(_Item("cnot" if r < 0.93 else "cz", (int(a), int(c))))
    return items


@pytest.mark.parametrize("dt", [torch.complex64, torch.complex128])
@pytest.mark.parametrize("n,batch,reorder", [(12, 4, True), (14, 3, True), (14, 2, False),
                                             (17, 2, True)])
def test_compiled_matches_interpreter_per_state_data(device, dt, n, batch, reorder):
    """Compiled passes against the interpreter (pinned against the oracle by
    the tests above and by the serving and adjoint tests) on the op kinds and
    per-state data those loops use."""
    items = _per_state_items(n, batch, seed=n * 3 + batch, device=device, dt=dt)
    interp = FusedProgram.from_items(items, n, dt, device, reorder=reorder)
    comp = FusedProgram.from_items(items, n, dt, device, reorder=reorder, compiled=True)
    assert comp.num_compiled == comp.num_passes
    psi = torch.from_numpy(seeded_state_np(n, (batch,), seed=5)).to(device, dt)
    a = interp.run(psi.clone()).cpu().numpy()
    c = comp.run(psi.clone()).cpu().numpy()
    assert rel_err(c, a) < {torch.complex64: 1e-5, torch.complex128: 1e-13}[dt]


def test_compiled_graph_replay_matches_eager(device):
    """Captured before any eager run: the program loaded its kernels when it
    was built, so the capture records launches only."""
    n = 14
    circ = random_mixed_circuit(n, 61, seed=5)    # a structure no other test compiles
    prog = FusedProgram(circ, dtype=torch.complex64, device=device, compiled=True)
    assert prog.num_compiled > 0
    psi = torch.from_numpy(seeded_state_np(n, (2,), seed=3)).to(device, torch.complex64)
    state = psi.clone()
    prog.capture(state)
    eager = prog.run(psi.clone())
    for _ in range(3):
        state.copy_(psi)
        torch.cuda.synchronize()
        prog.replay()
        torch.cuda.synchronize()
        assert torch.equal(state, eager)


def test_compiled_phase_angles_accuracy(device):
    """A compiled complex64 pass that reads phase angles forms exp(-1j angle)
    itself (reduction by pi/2 and polynomials up to |angle| 256, sincosf
    beyond): against float64 exp on angles in [-300, 300] and special values."""
    from unitair_amd.circuits import Circuit, Gate
    n = 12
    rng = np.random.default_rng(0)
    ang = rng.uniform(-300, 300, 2 ** n).astype(np.float32)
    ang[:10] = [0.0, np.pi / 2, -np.pi / 2, np.pi, 2 * np.pi, 256.0, -256.0, 256.5, 1e-30,
                -3 * np.pi / 4]
    ang[10:2000] = rng.uniform(0, 2 * np.pi, 1990).astype(np.float32)
    circ = Circuit(n, [Gate("phase", (), angles=ang)])
    prog = FusedProgram(circ, torch.complex64, device, compiled=True, phase_angles=True)
    assert prog.num_compiled == prog.num_passes == 1
    out = prog.run(torch.ones(1, 2 ** n, dtype=torch.complex64, device=device))
    err = np.abs(out.cpu().numpy()[0] - np.exp(-1j * ang.astype(np.float64)))
    assert np.max(err) < 3e-7, (int(np.argmax(err)), float(np.max(err)))


@pytest.mark.parametrize("n,tile_bits", [(16, 12), (16, 14), (17, 13)])
def test_compiled_tile_sizes(device, n, tile_bits):
    """Compiled passes on 12-, 13- and 14-bit complex64 tiles against the oracle."""
    circ = random_mixed_circuit(n, 90, seed=n + tile_bits)
    prog = FusedProgram(circ, dtype=torch.complex64, device=device, compiled=True,
                        tile_bits=tile_bits)
    fused = [st for st in prog.steps if st[0] == "fused"]
    assert fused and all(st[1].tile_bits == tile_bits for st in fused)
    assert prog.num_compiled == len(fused)
    psi = seeded_state_np(n, (2,), seed=9)
    ref = np.stack([oc.run_closed_form(circ.gates, p) for p in psi])
    out = prog.run(torch.from_numpy(psi).to(device, torch.complex64)).cpu().numpy()
    assert rel_err(out, ref) < 1e-4
    assert np.max(U.fidelity_error(ref, out)) < 1e-5


@pytest.mark.parametrize("n,batch", [(13, 2), (14, 1)])
def test_compiled_every_gate_of_a_cube(device, n, batch):
    """1-qubit gates on each cube bit and 2-qubit gates on every ordered pair
    of them, in one stage of a 13-bit tile (complex64: lane-private matrix-core
    products).  16 gates of at most 8 rounded terms each: 16 * 8 * 2^-24 =
    7.7e-6 of the largest amplitude's group."""
    from unitair_amd.circuits import Circuit, Gate
    rng = np.random.default_rng(41)
    low = [n - 1 - b for b in range(4)]              # the qubits of index bits 0..3
    gates = [Gate("dense", (q,), matrix=haar_unitary(2, rng)) for q in low]
    gates += [Gate("dense", (a, b), matrix=haar_unitary(4, rng))
              for a in low for b in low if a != b]
    prog = FusedProgram(Circuit(n, gates), device=device, reorder=False, merge_1q=False,
                        compiled=True)
    assert prog.num_passes == 1 and prog.num_compiled == 1
    psi = seeded_state_np(n, (batch,), seed=5)
    ref = np.stack([oc.run_closed_form(gates, p) for p in psi])
    out = prog.run(torch.from_numpy(psi).to(device, torch.complex64)).cpu().numpy()
    assert rel_err(out, ref) < 1e-5


def test_plan_recipes_together_match_one_by_one(device):
    """PlanTemplate.evaluate_all against evaluate: per-state rotations (real or
    imaginary entries: the same bits), general per-state gates (rounding) and
    single diagonals, shared and per-state."""
    from unitair_amd.fusion import PlanTemplate, _Item
    g = torch.Generator(device=device).manual_seed(8)
    B = 5

    def rnd(*shape):
        return torch.randn(*shape, generator=g, device=device, dtype=torch.complex64)
    t = torch.randn(B, generator=g, device=device)
    c, s = torch.cos(t), torch.sin(t)
    rot = torch.stack([torch.stack([c, -s], -1), torch.stack([s, c], -1)], -2).to(torch.complex64)
    items = [_Item("diag1", (0,), torch.polar(torch.ones(B, 2, device=device),
                                              rnd(B, 2).real).contiguous(), True),
             _Item("dense1", (0,), rot.contiguous(), True),
             _Item("dense1", (1,), rnd(B, 2, 2), True), _Item("diag1", (1,), rnd(B, 2), True),
             _Item("diag1", (2,), np.array([1, 1j]), False), _Item("dense1", (2,), np.eye(2), False)]
    d = lambda i: ("as_dense1", ("item", i))
    recipes = [("product", ("item", 1), d(0)), ("product", d(0), ("item", 1)), d(0), d(3),
               ("product", ("item", 2), d(3)), ("product", d(3), ("item", 2)), ("item", 2), d(4),
               ("product", ("item", 5), d(4)), ("product", d(3), ("product", d(3), ("item", 2)))]
    got = PlanTemplate.evaluate_all(recipes, items)
    for i, (r, a) in enumerate(zip(recipes, got)):
        b = PlanTemplate.evaluate(r, items)
        assert (a.kind, a.bits, a.per_state) == (b.kind, b.bits, b.per_state)
        x, y = torch.as_tensor(a.data), torch.as_tensor(b.data)
        assert x.shape == y.shape and x.dtype == y.dtype
        assert not isinstance(a.data, torch.Tensor) or a.data.is_contiguous()
        if i < 4:
            assert torch.equal(x, y)
        else:
            assert torch.allclose(x, y, rtol=1e-6, atol=1e-6)


@pytest.mark.parametrize("compiled", [False, True])
@pytest.mark.parametrize("dt", [torch.complex64, torch.complex128])
@pytest.mark.parametrize("n,batch,m", [(8, 2, 1), (12, 3, 1), (13, 4, 4), (16, 3, 2), (16, 2, 0)])
def test_run_from_a_source(device, dt, n, batch, m, compiled):
    """The first m states read from another tensor, which stays as it is: the
    same bits as a copy and a run in place (several pass structures each)."""
    g = torch.Generator(device=device).manual_seed(n)
    x = torch.randn(batch, 2 ** n, generator=g, device=device, dtype=dt)
    src = torch.randn(m, 2 ** n, generator=g, device=device, dtype=dt)
    for seed in (3, 4):
        circ = random_mixed_circuit(n, 50, seed=seed)
        prog = FusedProgram(circ, dtype=dt, device=device, compiled=compiled)
        a, b, kept = x.clone(), x.clone(), src.clone()
        a[:m] = src
        prog.run(a)
        prog.run(b, kept)
        assert torch.equal(a, b) and torch.equal(kept, src)
    with pytest.raises(ValueError):
        prog.run(x, torch.zeros(batch + 1, 2 ** n, dtype=dt, device=device))
    if compiled and n >= 12 and m:
        with pytest.raises(ValueError, match="overlap"):
            prog.run(x, x[batch - m:])
