"""Reverse-sweep programs (cqs_adjoint_passes) op by op, against complex128 NumPy: gradient sums of single ops
on thread, lane, register and outer bits, at tile widths on both sides of the decoded interpreter's range."""

import numpy as np
import pytest
import torch

from cirq_amd import engine
from cirq_amd._lib import SEL_BOTH, SEL_PHI, SEL_PSI, check, lib, ptr
from cirq_amd.adjoint import adjoint_waves
from cirq_amd.tape import LOp, PackedProgram, Pass

pytestmark = pytest.mark.gpu


def _bits(idx, targets):
    return sum((((idx >> b) & 1) << m) for m, b in enumerate(targets))


def _apply(psi, op, idx):
    kind = op.kind.removeprefix("grad_")
    if kind == "scale":
        return psi * op.mat
    if kind == "pair":
        return np.where(_bits(idx, op.targets) == 3, psi * op.mat, psi)
    if kind == "diag":
        return psi * op.mat[_bits(idx, op.targets)]
    ok = np.all([((idx >> b) & 1) == v for b, v in op.controls], axis=0) if op.controls else np.ones(len(idx), bool)
    row, rest = _bits(idx, op.targets), idx
    for b in op.targets:
        rest = rest & ~(1 << b)
    new = np.zeros_like(psi)
    for c in range(1 << len(op.targets)):
        src = rest | sum(((c >> m) & 1) << b for m, b in enumerate(op.targets))
        new += op.mat[row, c] * psi[src]
    return np.where(ok, new, psi)


def _reference(psi, phi, ops):
    psi, phi, idx, grads = psi.astype(np.complex128), phi.astype(np.complex128), np.arange(len(psi)), {}
    for op in ops:
        if op.kind.startswith("grad"):
            grads[op.slot] = 2 * np.vdot(phi, _apply(psi, op, idx)).real
            continue
        if op.sel != SEL_PHI:
            psi = _apply(psi, op, idx)
        if op.sel != SEL_PSI:
            phi = _apply(phi, op, idx)
    return psi, phi, np.array([grads[s] for s in sorted(grads)])


def _state(rng, n):
    v = (rng.randn(2**n) + 1j * rng.randn(2**n)).astype(np.complex64)
    return v / np.linalg.norm(v)


def _run(gpu, psi, phi, ops, local, n, specialize):
    L = len(local)
    slots = sum(op.kind.startswith("grad") for op in ops)
    prog = PackedProgram([Pass(L, tuple(local), ops)], n)
    dev = engine.DeviceProgram(prog, gpu, adjoint=True)
    a, b = torch.from_numpy(psi).to(gpu), torch.from_numpy(phi).to(gpu)
    stride = (1 << (n - L)) * adjoint_waves(L)
    partial = torch.full((slots, stride), float("nan"), dtype=torch.float64, device=gpu)
    args = [ptr(a), ptr(b), n, dev.pass_arr.ctypes.data, int(prog.n_passes), ptr(dev.ops), ptr(dev.mats), ptr(dev.aux),
            ptr(partial), stride]
    if specialize:
        from cirq_amd.specialize import specialize as compile_passes

        spec = compile_passes(prog, adjoint=True)
        check(lib().cqs_adjoint_passes_specialized(*args, spec.handles, engine.stream_handle()), "specialised")
    else:
        check(lib().cqs_adjoint_passes(*args, engine.stream_handle()), "cqs_adjoint_passes")
    return a.cpu().numpy(), b.cpu().numpy(), partial.cpu().numpy().sum(axis=1)


X, Y = np.array([[0, 1], [1, 0]]), np.array([[0, -1j], [1j, 0]])


@pytest.mark.parametrize("n,L,specialize", [(3, 3, False), (5, 5, False), (6, 6, False), (9, 7, False), (10, 9, False), (12, 11, False),
                                            (12, 11, True), (13, 12, False), (13, 13, False), (14, 12, True)])
def test_products_are_summed_in_fp64(gpu, n, L, specialize):
    """Gradient ops of one bit and diagonal ones on states that no op touches: the inputs are FP32 values, so the
    sums differ from NumPy's by FP64 rounding only."""
    print(f"gradient sums n={n} L={L} specialize={specialize}", flush=True)
    rng = np.random.RandomState(100 * n + L)
    psi, phi = _state(rng, n), _state(rng, n)
    local = sorted(int(b) for b in rng.permutation(n)[:L])
    f32 = lambda m: m.astype(np.complex64).astype(np.complex128)  # noqa: E731
    ops = []
    for b in local:
        ops += [LOp("grad_dense", (b,), f32(m)) for m in (0.5j * X, 0.5j * Y, rng.randn(2, 2) + 1j * rng.randn(2, 2))]
    for b in range(n):
        c = int(rng.choice([x for x in range(n) if x != b]))
        ops += [LOp("grad_diag", (b,), f32(1j * rng.randn(2))), LOp("grad_diag", (b, c), f32(1j * rng.randn(4))),
                LOp("grad_diag", (c, b), f32(rng.randn(4) + 1j * rng.randn(4)))]
    if n > 2:
        ops.append(LOp("grad_diag", (0, n - 1, 1), f32(1j * rng.randn(8))))
    for s, op in enumerate(ops):
        op.slot = s
    got_psi, got_phi, got = _run(gpu, psi, phi, ops, local, n, specialize)
    assert np.array_equal(got_psi, psi) and np.array_equal(got_phi, phi)
    want = _reference(psi, phi, ops)[2]
    scale = np.array([np.abs(op.mat).sum() for op in ops])
    # at most 2^7 additions in a row of terms that sum to at most |G| in absolute value
    assert np.all(np.abs(got - want) < 2.0**-53 * 2**7 * scale), (np.abs(got - want) / scale).max()
