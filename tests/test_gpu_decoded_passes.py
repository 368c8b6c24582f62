"""Passes whose program is decoded into LDS (csrc/staged.hpp): every form of op that has a record of its own,
on thread, register and outer bits, beside forms that run through the general path, against complex128
NumPy; programs of one op, of exactly one chunk of records, one more, and several chunks."""

import numpy as np
import pytest
import torch

from cirq_amd import engine
from cirq_amd.tape import LOp, PackedProgram, Pass, compile_ops

pytestmark = pytest.mark.gpu


def _bits(idx, targets):
    return sum((((idx >> b) & 1) << m) for m, b in enumerate(targets))


def _apply(psi, op, idx):
    if op.kind == "scale":
        return psi * op.mat
    if op.kind == "pair":
        return np.where(_bits(idx, op.targets) == 3, psi * op.mat, psi)
    if op.kind == "diag":
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


def _random_op(rng, n, local):
    phase = lambda k: np.exp(2j * np.pi * rng.rand(k))  # noqa: E731
    unitary = lambda d: np.linalg.qr(rng.randn(d, d) + 1j * rng.randn(d, d))[0]  # noqa: E731
    kind = rng.choice(["dense1", "dense1", "dense1c", "dense2", "diag1", "diag2", "diag3", "pair", "pair", "scale"])
    anyb = [int(b) for b in rng.permutation(n)]
    loc = [int(b) for b in rng.permutation(local)]
    if kind == "scale":
        return LOp("scale", (), phase(1)[0])
    if kind == "pair":
        return LOp("pair", tuple(anyb[:2]), phase(1)[0])
    if kind.startswith("diag"):
        k = int(kind[4])
        return LOp("diag", tuple(anyb[:k]), phase(1 << k))
    if kind == "dense2":
        return LOp("dense", tuple(loc[:2]), unitary(4))
    ctl = tuple((b, int(rng.randint(2))) for b in anyb if b != loc[0])[: rng.randint(1, 3)] if kind == "dense1c" else ()
    return LOp("dense", (loc[0],), unitary(2), ctl)


@pytest.mark.parametrize("n,L,count", [(6, 6, 1), (9, 6, 63), (8, 7, 64), (11, 8, 130), (10, 9, 200), (12, 10, 63), (13, 11, 127),
                                       (14, 12, 150), (15, 13, 80), (18, 6, 40)])
def test_random_programs(gpu, n, L, count):
    print(f"decoded pass n={n} L={L} ops={count}", flush=True)
    rng = np.random.RandomState(1000 * n + L)
    local = sorted(int(b) for b in rng.permutation(n)[:L])
    ops = [_random_op(rng, n, local) for _ in range(count)]
    psi = (rng.randn(2**n) + 1j * rng.randn(2**n)).astype(np.complex64)
    psi /= np.linalg.norm(psi)
    want, idx = psi.astype(np.complex128), np.arange(2**n)
    for op in ops:
        want = _apply(want, op, idx)
    st = torch.from_numpy(psi).to(gpu)
    engine.DeviceProgram(PackedProgram([Pass(L, tuple(local), ops)], n), gpu).run(st)
    got = st.cpu().numpy()
    # each op rounds every amplitude by about 2^-23; their errors add up at random, four deviations
    bound = 4 * np.sqrt(count + 1) * 2.0**-23
    assert np.linalg.norm(got - want) < bound
    # and from a basis state, through the planner (PERMUTE ops, several passes)
    b = int(rng.randint(2**n))
    ref = np.zeros(2**n, dtype=np.complex128)
    ref[b] = 1
    for op in ops:
        ref = _apply(ref, op, idx)
    out = torch.full((2**n,), float("nan"), dtype=torch.complex64, device=gpu)
    engine.DeviceProgram(compile_ops(ops, n, L=L, coalesce=min(4, L - 2)), gpu).run(out, basis=b)
    assert np.linalg.norm(out.cpu().numpy() - ref) < bound
