"""6- to 10-qubit complex gates on the matrix cores (wide_mfma.hip) against the
oracle: the smallest states and two qubits more, targets on the lowest, the
highest and mixed index bits, whole tiles in one workgroup and rows split over
several, one operator and one per batch entry, out of place and in place."""
import numpy as np
import pytest
import torch

from unitair_amd import _lib
from unitair_amd import simulation as sim
from oracle import unitair_np as U

pytestmark = pytest.mark.gpu

# an output sums 2 * 2^k products; rounding errors add up like a random walk:
# sqrt(2 * 1024) * 2^-24 = 2.7e-6 of the typical amplitude at most (the largest
# is several times that, so the bar relative to it has the same margin again)
TOL = {torch.complex64: 1e-5, torch.complex128: 2e-14}
NP = {torch.complex64: np.complex64, torch.complex128: np.complex128}

# smallest n the path takes, for each width
SIZES = [(torch.complex64, 6, 12), (torch.complex64, 7, 12), (torch.complex64, 8, 13),
         (torch.complex64, 9, 14), (torch.complex64, 10, 14), (torch.complex128, 6, 12),
         (torch.complex128, 7, 12), (torch.complex128, 8, 12), (torch.complex128, 9, 13)]


def _rand(shape, rng, dt):
    return (rng.standard_normal(shape) + 1j * rng.standard_normal(shape)).astype(NP[dt])


def _rel(out, ref):
    return float(np.max(np.abs(out - ref)) / np.max(np.abs(ref)))


@pytest.mark.parametrize("where", ["low", "high", "mixed"])
@pytest.mark.parametrize("extra,batch", [(0, 1), (0, 8), (2, 3)])
@pytest.mark.parametrize("dt,k,n0", SIZES)
def test_wide_gates(device, dt, k, n0, extra, batch, where):
    n = n0 + extra
    rng = np.random.default_rng(1000 * k + 10 * n + batch)
    order = [int(q) for q in rng.permutation(n)]
    if where == "low":
        order = [n - 1 - int(b) for b in rng.permutation(k)]
    elif where == "high":
        order = [int(q) for q in rng.permutation(k)]
    qubits = order[:k]
    op = _rand((2 ** k, 2 ** k), rng, dt) / NP[dt](2 ** (k / 2))
    st = _rand((batch, 2 ** n), rng, dt)
    opd, std = torch.from_numpy(op).to(device), torch.from_numpy(st).to(device)
    ref = U.apply_operator(op.astype(np.complex128), qubits, st.astype(np.complex128))
    out = sim.apply_operator(opd, qubits, std)
    assert _rel(out.cpu().numpy(), ref) < TOL[dt]
    # in place, one (equal) operator per entry: the whole tile in one workgroup
    ops = opd.expand(batch, -1, -1).contiguous()
    x = std.clone()
    rc = _lib.load().ua_apply_operator(
        _lib.ptr(x), _lib.ptr(x), _lib.ptr(ops), _lib.DTYPE_CODES[dt], n, k,
        _lib.int_array(qubits), batch, 2 ** n, 4 ** k, _lib.stream_handle(device))
    _lib.check(rc, "in place")
    assert torch.equal(x, out)       # the same sums in the same order


@pytest.mark.parametrize("dt,k,n", [(torch.complex64, 8, 21), (torch.complex128, 7, 20)])
def test_wide_gates_many_tiles(device, dt, k, n):
    """At least 256 tiles, out of place: whole tiles, one per workgroup."""
    rng = np.random.default_rng(k)
    qubits = [int(q) for q in rng.permutation(n)[:k]]
    op = _rand((2 ** k, 2 ** k), rng, dt) / NP[dt](2 ** (k / 2))
    st = _rand((2 ** n,), rng, dt)
    out = sim.apply_operator(torch.from_numpy(op).to(device), qubits,
                             torch.from_numpy(st).to(device))
    ref = U.apply_operator(op.astype(np.complex128), qubits, st.astype(np.complex128))
    assert _rel(out.cpu().numpy(), ref) < TOL[dt]


# 2, 48, 50, 254, 256, 320, 352 and 354 tiles of 2^13 amplitudes
@pytest.mark.parametrize("n,batch", [(14, 1), (14, 24), (14, 25), (14, 127), (14, 128), (15, 80),
                                     (14, 176), (14, 177)])
def test_8_qubit_gates_by_tiles(device, n, batch):
    """complex64: columns split over the wavefronts and rows over 16 or 8
    workgroups of a tile, or a tile in one piece; in place (one operator for each
    entry: in one piece) the sums are the same, in the same order."""
    k = 8
    rng = np.random.default_rng(batch)
    g = torch.Generator(device=device).manual_seed(batch)
    st = torch.randn(batch, 2 ** n, generator=g, device=device, dtype=torch.complex64)
    op = _rand((2 ** k, 2 ** k), rng, torch.complex64) / np.complex64(16)
    opd = torch.from_numpy(op).to(device)
    pick = sorted({0, batch // 2, batch - 1})
    for bits in (list(range(k)), [int(b) for b in rng.permutation(n)[:k]]):
        qubits = [n - 1 - b for b in bits]
        out = sim.apply_operator(opd, qubits, st)
        ref = U.apply_operator(op.astype(np.complex128), qubits,
                               st[pick].cpu().numpy().astype(np.complex128))
        assert _rel(out[pick].cpu().numpy(), ref) < TOL[torch.complex64]
        x, ops = st.clone(), opd.expand(batch, -1, -1).contiguous()
        _lib.check(_lib.load().ua_apply_operator(
            _lib.ptr(x), _lib.ptr(x), _lib.ptr(ops), _lib.UA_COMPLEX64, n, k,
            _lib.int_array(qubits), batch, 2 ** n, 4 ** k, _lib.stream_handle(device)), "in place")
        assert torch.equal(x, out)
