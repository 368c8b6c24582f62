"""cqs_expect_paulis over terms with X masks (k_pauli_terms) against FP64 NumPy sums: states of part
of a chunk, exactly one chunk (2^11), the first sizes with several slices, and more chunks than
slices; one term, a partial group of 8, more terms than one launch takes; states that do not start on
16 bytes; density matrices."""

import numpy as np
import pytest
import torch

from cirq_amd._lib import check, lib, ptr

pytestmark = pytest.mark.gpu


def _terms(rng, n, count):
    top = 1 << n
    xm = np.array([int(rng.randint(0, top)) for _ in range(count)], dtype=np.uint64)
    xm[1::5] = xm[0]  # equal masks share reads
    xm[2::7] &= np.uint64(min(top - 1, 2047))  # masks that stay inside a chunk
    zm = np.array([int(rng.randint(0, top)) for _ in range(count)], dtype=np.uint64)
    return xm, zm, rng.randn(2 * count)


def _signs(idx, z):
    v = idx & z
    for s in (32, 16, 8, 4, 2, 1):
        v = v ^ (v >> np.uint64(s))
    return 1.0 - 2.0 * (v & np.uint64(1)).astype(np.float64)


def _run(st, n, is_dm, xm, zm, cf):
    T = len(xm)
    ws = torch.empty(int(lib().cqs_expect_workspace_bytes(T)), dtype=torch.uint8, device=st.device)
    out = torch.full((2 * T,), np.nan, dtype=torch.float64, device=st.device)
    check(lib().cqs_expect_paulis(ptr(st), n, int(is_dm), T, xm.ctypes.data, zm.ctypes.data, cf.ctypes.data, ptr(out),
                                  ptr(ws), torch.cuda.current_stream().cuda_stream), "cqs_expect_paulis")
    return out.cpu().numpy().view(np.complex128)


@pytest.mark.parametrize("n,count,offset", [(0, 1, 0), (1, 3, 1), (3, 8, 0), (5, 9, 1), (10, 42, 0), (11, 97, 0), (11, 5, 1),
                                            (12, 40, 0), (13, 200, 1), (20, 17, 0)])
def test_state_vector_terms(gpu, n, count, offset):
    rng = np.random.RandomState(100 * n + count)
    psi = (rng.randn(2**n) + 1j * rng.randn(2**n)).astype(np.complex64)
    psi /= np.linalg.norm(psi)
    buf = torch.empty(2**n + offset, dtype=torch.complex64, device=gpu)
    st = buf[offset:]
    st.copy_(torch.from_numpy(psi))
    xm, zm, cf = _terms(rng, n, count)
    got = _run(st, n, False, xm, zm, cf)
    p, idx = psi.astype(np.complex128), np.arange(2**n, dtype=np.uint64)
    for t in range(count):
        w = complex(cf[2 * t], cf[2 * t + 1]) * np.sum(np.conj(p[(idx ^ xm[t]).astype(np.int64)]) * _signs(idx, zm[t]) * p)
        # products of float32 values are exact in FP64; sums of unit norm round by at most n * 2^-53 per tree level
        assert abs(got[t] - w) < 1e-13 * max(1, abs(complex(cf[2 * t], cf[2 * t + 1]))) * max(1, n)


@pytest.mark.parametrize("n,count", [(1, 2), (4, 9), (11, 3), (12, 20)])
def test_density_matrix_terms(gpu, n, count):
    rng = np.random.RandomState(n)
    rho = (rng.randn(2**n, 2**n) + 1j * rng.randn(2**n, 2**n)).astype(np.complex64)
    st = torch.from_numpy(rho.reshape(-1)).to(gpu)
    xm, zm, cf = _terms(rng, n, count)
    got = _run(st, n, True, xm, zm, cf)
    idx = np.arange(2**n, dtype=np.uint64)
    for t in range(count):
        d = rho[idx.astype(np.int64), (idx ^ xm[t]).astype(np.int64)].astype(np.complex128)
        c = complex(cf[2 * t], cf[2 * t + 1])
        # 2^n entries of unit size in FP64
        assert abs(got[t] - c * np.sum(_signs(idx, zm[t]) * d)) < 2.0**-53 * 2**n * 8 * abs(c)


@pytest.mark.parametrize("n", [0, 1, 5, 11, 12, 16])
def test_norm_of_the_scaled_state_without_writing_it(gpu, n):
    """engine.norm2 with a scale gives the bits of engine.scale followed by engine.norm2."""
    from cirq_amd import engine

    rng = np.random.RandomState(n)
    st = torch.from_numpy((rng.randn(2**n) + 1j * rng.randn(2**n)).astype(np.complex64)).to(gpu)
    ws = engine.Workspace(st.device)
    for s in (1.0, 0.7310585, 1.0000001):
        t = st.clone()
        engine.scale(t, n, s)
        assert engine.norm2(st, n, ws, scale=s) == engine.norm2(t, n, ws)


@pytest.mark.parametrize("n,offset", [(21, 0), (22, 1)])
def test_terms_of_states_with_several_chunks_per_slice(gpu, n, offset):
    """Masks whose top bit numbers a slice, a slice's chunks, the state's halves; equal masks with either parity of Y in a
    row; 16 terms (the small argument block) and more."""
    rng = np.random.RandomState(n)
    psi = (rng.randn(2**n) + 1j * rng.randn(2**n)).astype(np.complex64)
    psi /= np.linalg.norm(psi)
    buf = torch.empty(2**n + offset, dtype=torch.complex64, device=gpu)
    st = buf[offset:]
    st.copy_(torch.from_numpy(psi))
    xs = [1 << 12, 1 << 12, (1 << 12) | 3, 1 << 19, (1 << 20) | 1, 1 << (n - 1), (1 << (n - 1)) | (1 << 11), (1 << n) - 1, 5, 5, 5, 5]
    zs = [0, 1 << 12, 1 << 20, (1 << 19) | 1, 1 << 20, 1 << (n - 1), 7, (1 << n) - 1, 0, 1, 4, 5]
    xm, zm = np.array(xs, dtype=np.uint64), np.array(zs, dtype=np.uint64)
    p, idx = psi.astype(np.complex128), np.arange(2**n, dtype=np.uint64)
    want = np.array([np.sum(np.conj(p[(idx ^ x).astype(np.int64)]) * _signs(idx, z) * p) for x, z in zip(xm, zm)])
    for count in (1, 12, 16, 17, 30):
        pick = np.arange(count) % len(xs) if count > 1 else np.array([0])
        got = _run(st, n, False, xm[pick], zm[pick], np.tile([1.0, 0.0], count))
        assert np.abs(got - want[pick]).max() < 1e-13 * n  # as above
