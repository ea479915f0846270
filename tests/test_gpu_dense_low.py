"""2- and 3-qubit gates whose targets lie within one wavefront's block of
amplitudes (dense_low_kernel) against the oracle, and bit for bit against the
general kernel, which takes the same products in the same order: it runs the
same call on a state one element off the alignment."""
import numpy as np
import pytest
import torch

from unitair_amd import _lib
from unitair_amd import simulation as sim
from oracle import unitair_np as U

pytestmark = pytest.mark.gpu

# an output sums 2 * 2^k <= 16 products, each rounded once: 16 half-ulps of the
# sum of their magnitudes, itself a few times the largest output
TOL = {torch.float32: 4e-6, torch.complex64: 4e-6, torch.float64: 8e-15, torch.complex128: 8e-15}
NP = {torch.complex64: np.complex64, torch.complex128: np.complex128,
      torch.float32: np.float32, torch.float64: np.float64}
# target index bits; per k: lowest, lines split, the block's last bit, beyond it
BITS = {2: [(0, 1), (1, 2), (3, 0), (7, 2), (0, 7), (8, 1), (6, 4), (11, 2), (9, 3), (1, 12)],
        3: [(0, 1, 2), (3, 1, 2), (8, 0, 7), (5, 8, 6), (4, 2, 0), (9, 1, 0),
            (10, 2, 7), (10, 1, 9), (14, 12, 3), (0, 14, 2), (3, 6, 13)]}


def _rand(shape, rng, dt):
    x = rng.standard_normal(shape)
    if dt.is_complex:
        x = x + 1j * rng.standard_normal(shape)
    return torch.from_numpy(np.asarray(x).astype(NP[dt]))


@pytest.mark.parametrize("per_state", [False, True])
@pytest.mark.parametrize("dt", list(TOL))
@pytest.mark.parametrize("k,n,batch", [(2, 8, 33), (2, 10, 5), (2, 13, 1), (2, 12, 3),
                                       (3, 9, 70), (3, 9, 63), (3, 11, 17), (3, 15, 1)])
def test_low_targets(device, dt, k, n, batch, per_state):
    rng = np.random.default_rng(100 * n + batch)
    size = batch * 2 ** n
    for bits in BITS[k]:
        if max(bits) >= n:
            continue
        qubits = [n - 1 - b for b in bits]
        ops = _rand(((batch,) if per_state else ()) + (2 ** k, 2 ** k), rng, dt)
        st = _rand((batch, 2 ** n), rng, dt)
        wide = {True: np.complex128, False: np.float64}[dt.is_complex]
        ref = U.apply_operator(ops.numpy().astype(wide), qubits, st.numpy().astype(wide))
        opd, x = ops.to(device), st.to(device)
        out = sim.apply_operator(opd, qubits, x)
        err = np.max(np.abs(out.cpu().numpy() - ref)) / np.max(np.abs(ref))
        assert err < TOL[dt], (bits, err)
        buf = torch.empty(2 * size + 4, dtype=dt, device=device)
        off, res = buf[1:1 + size].view(batch, 2 ** n), buf[size + 1:2 * size + 1].view(batch, -1)
        off.copy_(x)

        def call(o, i):
            _lib.check(_lib.load().ua_apply_operator(
                _lib.ptr(o), _lib.ptr(i), _lib.ptr(opd), _lib.DTYPE_CODES[dt], n, k,
                _lib.int_array(qubits), batch, 2 ** n, 4 ** k if per_state else 0,
                _lib.stream_handle(device)), "apply_operator")
        call(res, off)
        assert torch.equal(res, out), bits
        call(x, x)                                  # in place
        assert torch.equal(x, out), bits


@pytest.mark.parametrize("n,batch", [(9, 2), (10, 1), (10, 4096), (10, 4097), (13, 7), (17, 3)])
def test_4_qubit_gates_on_either_side_of_the_matrix_core_rule(device, n, batch):
    """complex64 4-qubit gates: vector kernel under 10 qubits and beyond the
    caches, matrix cores between, any targets and alignment, also in place."""
    rng = np.random.default_rng(n)
    g = torch.Generator(device=device).manual_seed(n)
    pick = sorted({0, batch // 2, batch - 1})
    for bits in [(0, 1, 5, 7), (8, 7, 6, n - 1), (n - 1, 3, 0, n - 3), (2, 4, 5, 7)]:
        if len(set(bits)) < 4:
            continue
        qubits = [n - 1 - b for b in bits]
        op = _rand((16, 16), rng, torch.complex64)
        flat = torch.randn(batch * 2 ** n + 1, generator=g, device=device, dtype=torch.complex64)
        for off in (0, 1):
            x = flat[off:off + batch * 2 ** n].view(batch, 2 ** n)
            ref = U.apply_operator(op.numpy().astype(np.complex128), qubits,
                                   x[pick].cpu().numpy().astype(np.complex128))
            out = sim.apply_operator(op.to(device), qubits, x)
            err = np.max(np.abs(out[pick].cpu().numpy() - ref)) / np.max(np.abs(ref))
            assert err < 8e-6, (bits, off, err)     # 32 products: as above, twice the terms
            y, opd = x.clone(), op.to(device)
            _lib.check(_lib.load().ua_apply_operator(
                _lib.ptr(y), _lib.ptr(y), _lib.ptr(opd), _lib.UA_COMPLEX64, n, 4,
                _lib.int_array(qubits), batch, 2 ** n, 0, _lib.stream_handle(device)), "in place")
            assert torch.equal(y, out)


@pytest.mark.parametrize("dt", list(TOL))
@pytest.mark.parametrize("n,batch,per_state", [(12, 64, True), (12, 300, True), (12, 2048, True),
                                               (10, 1024, True), (10, 4097, True),
                                               (18, 1, False), (19, 1, False), (20, 1, False),
                                               (13, 300, False), (24, 1, False)])
def test_low_targets_on_either_side_of_the_sizes(device, dt, n, batch, per_state):
    """From states that wait for accesses to states beyond the caches: whichever
    kernel the size calls for, the bits are those of the general one (the same
    call on a state one element off the alignment)."""
    g = torch.Generator(device=device).manual_seed(n + batch)
    size = batch * 2 ** n
    buf = torch.empty(2 * size + 4, dtype=dt, device=device)
    off, res = buf[1:1 + size].view(batch, 2 ** n), buf[size + 1:2 * size + 1].view(batch, -1)
    x = torch.randn(batch, 2 ** n, generator=g, device=device, dtype=dt)
    off.copy_(x)
    for k in (2, 3):
        ops = torch.randn(((batch,) if per_state else ()) + (2 ** k, 2 ** k), generator=g,
                          device=device, dtype=dt)
        for bits in BITS[k] + [(0, 3), (3, 5), (n - 1, 0)][:3 * (3 - k)] + \
                [(n - 1, 1, 3), (n - 1, 0, 2), (6, 7, 8)][:3 * (k - 2)]:
            if max(bits) >= n:
                continue
            qubits = _lib.int_array([n - 1 - b for b in bits])
            for o, i in ((res, off), (x, x.clone())):
                _lib.check(_lib.load().ua_apply_operator(
                    _lib.ptr(o), _lib.ptr(i), _lib.ptr(ops), _lib.DTYPE_CODES[dt], n, k, qubits,
                    batch, 2 ** n, 4 ** k if per_state else 0, _lib.stream_handle(device)),
                    "apply_operator")
            assert torch.equal(res, x), bits
            x.copy_(off)


@pytest.mark.parametrize("batch", [256, 257, 512])
def test_4_qubit_gates_on_the_lowest_bit(device, batch):
    """complex64 states of 13 qubits around 2^21 and 2^22 amplitudes in all, where gates
    with and without a target on the lowest bit change kernels."""
    n = 13
    g = torch.Generator(device=device).manual_seed(batch)
    x = torch.randn(batch, 2 ** n, generator=g, device=device, dtype=torch.complex64)
    op = torch.randn(16, 16, generator=g, device=device, dtype=torch.complex64)
    pick = [0, batch // 2, batch - 1]
    for bits in [(0, 5, 9, 12), (7, 0, 6, 8), (1, 5, 9, 12)]:
        qubits = [n - 1 - b for b in bits]
        out = sim.apply_operator(op, qubits, x)
        ref = U.apply_operator(op.cpu().numpy().astype(np.complex128), qubits,
                               x[pick].cpu().numpy().astype(np.complex128))
        assert np.max(np.abs(out[pick].cpu().numpy() - ref)) / np.max(np.abs(ref)) < 8e-6, bits
