"""Reverse-sweep programs (cqs_adjoint_passes) op by op, against complex128 NumPy: gradient sums of single ops
on thread, lane, register and outer bits, and random programs of one op, one chunk of decoded records, one more and
several, at tile widths on both sides of the decoded interpreter's range and compiled."""

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


def _reference(psi, phi, ops, outer={}):
    """outer: slot -> (bit, value), the outer control of a gradient op."""
    psi, phi, idx, grads = psi.astype(np.complex128), phi.astype(np.complex128), np.arange(len(psi)), {}
    for op in ops:
        if op.kind.startswith("grad"):
            bit, value = outer.get(op.slot, (0, None))
            on = np.ones(len(idx)) if value is None else ((idx >> bit) & 1) == value
            grads[op.slot] = 2 * np.vdot(phi, on * _apply(psi, op, idx)).real
            continue
        if op.sel != SEL_PHI:
            psi = _apply(psi, op, idx)
        if op.sel != SEL_PSI:
            phi = _apply(phi, op, idx)
    return psi, phi, np.array([grads[s] for s in sorted(grads)])


def _state(rng, n):
    v = (rng.randn(2**n) + 1j * rng.randn(2**n)).astype(np.complex64)
    return v / np.linalg.norm(v)


def _run(gpu, psi, phi, ops, local, n, specialize, outer={}):
    L = len(local)
    slots = sum(op.kind.startswith("grad") for op in ops)
    prog = PackedProgram([Pass(L, tuple(local), ops)], n)
    for slot, (bit, value) in outer.items():  # no circuit's program has these: set in the packed ops
        (i,) = np.nonzero((prog.ops_arr["slot"] == slot) & ((prog.ops_arr["kind"] & 0xFF) >= 6))[0]
        prog.ops_arr["co_mask_lo"][i], prog.ops_arr["co_val_lo"][i] = 1 << bit, value << bit
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


def _random_op(rng, n, local, unit=True):
    """An op of a reverse program; unit=False: diagonal ops of any modulus."""
    def phase(k):
        return np.exp(2j * np.pi * rng.rand(k)) * (1 if unit else rng.uniform(0.8, 1.2, k))

    def unitary(d):
        return np.linalg.qr(rng.randn(d, d) + 1j * rng.randn(d, d))[0]

    anyb, loc = [int(b) for b in rng.permutation(n)], [int(b) for b in rng.permutation(local)]
    kinds = ["dense1", "dense1", "dense1c", "dense2", "dense3", "diag1", "diag2", "diag3", "pair", "pair", "scale",
             "grad_dense1", "grad_dense1", "grad_dense2", "grad_dense3", "grad_diag1", "grad_diag2", "grad_diag3"]
    kind = str(rng.choice([k for k in kinds if int(k[-1] if k[-1].isdigit() else 2) <= len(loc)]))
    sel = int(rng.choice([SEL_BOTH, SEL_BOTH, SEL_BOTH, SEL_PSI, SEL_PHI]))
    if kind.startswith("grad"):
        k = int(kind[-1])
        if "diag" in kind:
            real = rng.rand() < 0.3
            return LOp("grad_diag", tuple(anyb[:k]), 1j * rng.randn(1 << k) + (rng.randn(1 << k) if real else 0))
        g = rng.randn(1 << k, 1 << k) + 1j * rng.randn(1 << k, 1 << k)
        return LOp("grad_dense", tuple(loc[:k]), g - g.conj().T if rng.rand() < 0.5 else g)
    if kind == "scale":
        return LOp("scale", (), phase(1)[0], (), None, sel)
    if kind == "pair":
        return LOp("pair", tuple(anyb[:2]), phase(1)[0])
    if kind.startswith("diag"):
        return LOp("diag", tuple(anyb[: int(kind[4])]), phase(1 << int(kind[4])), (), None, sel)
    if kind == "dense1c":
        ctl = tuple((b, int(rng.randint(2))) for b in anyb if b != loc[0])[: rng.randint(1, 3)]
        return LOp("dense", (loc[0],), unitary(2), ctl, None, sel)
    k = int(kind[5])
    return LOp("dense", tuple(loc[:k]), unitary(1 << k), (), None, sel)


def _check_program(gpu, rng, n, L, ops, local, specialize, unit=True):
    slot, outer = 0, {}
    out = [b for b in range(n) if b not in local]
    for op in ops:
        if op.kind.startswith("grad"):
            op.slot = slot
            if out and rng.rand() < 0.2:
                outer[slot] = (int(rng.choice(out)), int(rng.randint(2)))
            slot += 1
    psi, phi = _state(rng, n), _state(rng, n)
    got_psi, got_phi, got = _run(gpu, psi, phi, ops, local, n, specialize, outer)
    want_psi, want_phi, want = _reference(psi, phi, ops, outer)
    # each op rounds every amplitude by about 2^-23, errors add up at random, four deviations; without unit modulus the
    # norms wander
    size = 1.0 if unit else 2.0 * max(1, np.linalg.norm(want_psi), np.linalg.norm(want_phi)) ** 2
    bound = 4 * np.sqrt(len(ops) + 1) * 2.0**-23 * size
    assert np.linalg.norm(got_psi - want_psi) < bound and np.linalg.norm(got_phi - want_phi) < bound
    norms = np.array([np.abs(op.mat).max() if op.kind == "grad_diag" else np.linalg.norm(op.mat, 2)
                      for op in ops if op.kind.startswith("grad")])
    assert np.all(np.abs(got - want) <= 2 * norms * (2 * bound + 2.0**-22)), np.max(np.abs(got - want) / norms)


PROGRAMS = [(4, 4, 40, False), (7, 5, 63, False), (6, 6, 1, False), (9, 6, 63, False), (9, 7, 64, False), (8, 8, 130, False),
            (10, 9, 64, False), (12, 10, 200, False), (13, 11, 130, False), (14, 12, 64, False), (14, 13, 40, False),
            (9, 7, 15, False), (9, 7, 16, False), (18, 6, 31, False), (18, 6, 32, False), (21, 11, 6, False),  # decoded or not
            (8, 7, 30, True), (12, 10, 60, True), (13, 11, 60, True), (13, 12, 40, True)]


@pytest.mark.parametrize("n,L,count,specialize", PROGRAMS)
def test_random_reverse_programs(gpu, n, L, count, specialize):
    print(f"reverse program n={n} L={L} ops={count} specialize={specialize}", flush=True)
    rng = np.random.RandomState(7000 * n + 10 * L + count)
    local = sorted(int(b) for b in rng.permutation(n)[:L])
    _check_program(gpu, rng, n, L, [_random_op(rng, n, local) for _ in range(count)], local, specialize)


@pytest.mark.parametrize("specialize", [False, True])
@pytest.mark.parametrize("sel", [SEL_PSI, SEL_PHI])
def test_programs_that_touch_one_state(gpu, sel, specialize):
    """Passes of ops on one state, through registers and through LDS: the other state stays as it is."""
    print(f"one state sel={sel} specialize={specialize}", flush=True)
    rng = np.random.RandomState(sel)
    ops = [LOp("dense", t, np.linalg.qr(rng.randn(2 ** len(t), 2 ** len(t)))[0] + 0j, (), None, sel)
           for t in ((9, 10), (0, 7), (3,), (7,))]
    for chosen in ([ops[0]], [ops[1]], ops):
        _check_program(gpu, rng, 12, 11, chosen, list(range(11)), specialize)


@pytest.mark.parametrize("n,L,count,specialize", [(5, 5, 30, False), (9, 7, 64, False), (12, 11, 64, False), (13, 12, 40, False),
                                                  (12, 11, 40, True)])
def test_diagonal_ops_of_any_modulus(gpu, n, L, count, specialize):
    """Gradients on both sides of diagonal ops that change conj(phi) psi (scales, diagonals, pairs on both states)."""
    print(f"any modulus n={n} L={L} ops={count} specialize={specialize}", flush=True)
    rng = np.random.RandomState(31 * n + L)
    local = sorted(int(b) for b in rng.permutation(n)[:L])
    ops = []
    while len(ops) < count:
        op = _random_op(rng, n, local, unit=False)
        if "diag" in op.kind or op.kind in ("pair", "scale"):
            ops.append(op)
    _check_program(gpu, rng, n, L, ops, local, specialize, unit=False)
