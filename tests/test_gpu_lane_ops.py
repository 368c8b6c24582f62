"""One-bit ops on lane bits (exchanged between lanes in registers) and gradients by generators, at the tile
widths where the layout changes: tiles smaller than a wave, than a workgroup, one element per thread,
several, 512 threads."""

import numpy as np
import pytest
import sympy
import torch

import cirq_amd as cirq
from cirq_amd import engine
from cirq_amd.adjoint import AdjointGradient
from cirq_amd.tape import LOp, compile_ops
from tests.test_adjoint_host import _oracle_grad

pytestmark = pytest.mark.gpu


def _apply(psi, n, bit, u, ctl):
    v = psi.reshape(2 ** (n - bit - 1), 2, 2**bit)
    new = np.stack([u[0, 0] * v[:, 0] + u[0, 1] * v[:, 1], u[1, 0] * v[:, 0] + u[1, 1] * v[:, 1]], axis=1).reshape(-1)
    idx = np.arange(2**n)
    ok = np.ones(2**n, dtype=bool)
    for b, val in ctl:
        ok &= ((idx >> b) & 1) == val
    return np.where(ok, new, psi)


@pytest.mark.parametrize("n,L,specialize", [(1, 1, False), (4, 4, False), (6, 6, False), (9, 7, False), (9, 8, False), (11, 9, False),
                                            (12, 11, True), (13, 12, False), (15, 13, True)])
def test_one_bit_ops_on_every_tile_bit(gpu, n, L, specialize):
    print(f"lane ops n={n} L={L}", flush=True)
    rng = np.random.RandomState(10 * n + L)
    psi = (rng.randn(2**n) + 1j * rng.randn(2**n)).astype(np.complex64)
    psi /= np.linalg.norm(psi)
    want, ops = psi.astype(np.complex128), []
    for i in range(3 * n):
        b = i % n
        u = np.linalg.qr(rng.randn(2, 2) + 1j * rng.randn(2, 2))[0]
        others = [x for x in range(n) if x != b]
        ctl = tuple((int(c), int(rng.randint(2))) for c in rng.permutation(others)[: i // n])  # 0, 1, 2 controls
        ops.append(LOp("dense", (b,), u, ctl))
        want = _apply(want, n, b, u, ctl)
    prog = engine.DeviceProgram(compile_ops(ops, n, L=L, coalesce=min(4, L), fuse=False, blocks=False), gpu)
    if specialize:
        prog.specialize()
    st = torch.from_numpy(psi).to(gpu)
    prog.run(st)
    # 3 n gates, each rounding an amplitude of at most 1 by about 2^-23
    assert np.abs(st.cpu().numpy() - want).max() < 3 * n * 2.0**-23


@pytest.mark.parametrize("n,specialize", [(1, False), (2, False), (5, False), (7, False), (8, False), (9, True), (11, False), (12, True)])
def test_gradients_on_every_bit(gpu, n, specialize):
    """Rotations about X, Y, Z and diagonal pairs on every qubit, beside fixed CZ and CNOT: the adjoint sweep against
    the two-term shift rule (controlled rotations, which have no such rule, are below)."""
    print(f"gradients n={n}", flush=True)
    rng = np.random.RandomState(n)
    qs = cirq.LineQubit.range(n)
    c, syms = cirq.Circuit(), []

    def sym():
        syms.append(sympy.Symbol(f"p{len(syms):03d}"))
        return syms[-1]

    for _ in range(2):
        for q in qs:
            c.append([cirq.ry(sym()).on(q), cirq.rz(sym()).on(q), cirq.rx(sym()).on(q)])
            c.append(cirq.PhasedXPowGate(phase_exponent=0.3, exponent=sym()).on(q))
        for a, b in zip(qs, qs[1:]):
            c.append([cirq.ZZPowGate(exponent=sym()).on(a, b), cirq.CZ.on(a, b), cirq.CNOT.on(b, a)])
    h = sum((float(rng.randn()) * cirq.X(q) for q in qs[1:]), float(rng.randn()) * cirq.Z(qs[0]))
    for a, b in zip(qs, qs[1:]):
        h = h + float(rng.randn()) * cirq.Y(a) * cirq.Z(b)
    ag = AdjointGradient(c, h)
    if specialize:
        ag.specialize()
    x = rng.uniform(-2, 2, len(syms))
    v, g = ag.value_and_grad(x)
    v2, g2 = ag.parameter_shift(x)
    # complex64 states of about 10 n gates; H's coefficients sum to about 2 n
    assert abs(v - v2) < 1e-5 * n and np.abs(g - g2).max() < 1e-5 * n


@pytest.mark.parametrize("n,L,specialize", [(3, None, False), (5, None, False), (7, 6, False), (9, 8, False), (9, 8, True), (9, 9, False)])
def test_gradients_of_controlled_rotations(gpu, n, L, specialize):
    """Generators with controls folded in (two- and three-bit gradient ops) and diagonal ones, on thread, register and
    outer bits, against central differences of complex128 simulations."""
    print(f"controlled gradients n={n} L={L}", flush=True)
    rng = np.random.RandomState(n)
    qs = cirq.LineQubit.range(n)
    c, syms = cirq.Circuit([cirq.H(q) for q in qs]), []

    def sym():
        syms.append(sympy.Symbol(f"p{len(syms):03d}"))
        return syms[-1]

    for i in range(n):
        a, b, d = (qs[int(x)] for x in rng.permutation(n)[:3])
        c.append([cirq.ControlledGate(cirq.ry(sym())).on(a, b), cirq.CXPowGate(exponent=sym()).on(b, d),
                  cirq.CZPowGate(exponent=sym()).on(a, d), cirq.rx(0.3 + i).on(a),
                  cirq.ControlledGate(cirq.rx(sym()), control_values=[0]).on(d, a),
                  cirq.ControlledGate(cirq.ry(sym()), num_controls=2).on(a, b, d), cirq.rz(0.7 * i).on(b)])
    h = sum((float(rng.randn()) * cirq.X(q) for q in qs[1:]), float(rng.randn()) * cirq.Z(qs[0]))
    for a, b in zip(qs, qs[1:]):
        h = h + float(rng.randn()) * cirq.Y(a) * cirq.Z(b)
    ag = AdjointGradient(c, h, adjoint_tile_bits=L)
    if specialize:
        ag.specialize()
    x = rng.uniform(-2, 2, len(syms))
    names = dict(zip(syms, x))
    value, grad = ag.value_and_grad([names[s] for s in ag.symbols])
    want = _oracle_grad(c, qs, h, ag.symbols, np.array([names[s] for s in ag.symbols]))
    size = sum(abs(complex(t.coefficient)) for t in h)
    print(f"  largest error {np.abs(grad - want).max() / size:.2e} of sum |c|", flush=True)
    # complex64 states of up to 65 ops leave 3e-8 to 1.3e-7 of sum |c|, stated with four times that; the differences
    # (h = 1e-5) are good to 1e-10
    assert np.abs(grad - want).max() < 5e-7 * size
