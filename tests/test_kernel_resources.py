"""Registers of compiled kernels, read from the code objects' metadata: the pass kernels keep their tiles in registers
and use no scratch memory (a scratch access per element and op is what they exist to avoid)."""

import re
import struct
import subprocess
from pathlib import Path

import numpy as np
import pytest

from cirq_amd import _build, generators, specialize
from cirq_amd.adjoint import AdjointProgram

READELF = Path("/opt/rocm/llvm/bin/llvm-readelf")
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def _scratch(path: Path, tmp: Path) -> dict:
    """{kernel: bytes of scratch memory per lane} of every gfx950 kernel in a shared object."""
    if not READELF.exists():
        pytest.skip("llvm-readelf is not installed")
    data, out, at = path.read_bytes(), {}, 0
    while (at := data.find(MAGIC, at)) >= 0:
        pos = at + len(MAGIC) + 8
        for _ in range(struct.unpack_from("<Q", data, at + len(MAGIC))[0]):
            offset, size, length = struct.unpack_from("<QQQ", data, pos)
            triple = data[pos + 24 : pos + 24 + length]
            pos += 24 + length
            if b"gfx950" in triple and size:
                obj = tmp / "code.o"
                obj.write_bytes(data[at + offset : at + offset + size])
                notes = subprocess.run([str(READELF), "--notes", str(obj)], capture_output=True, text=True, check=True).stdout
                for kernel in notes.split("- .agpr_count")[1:]:
                    out[re.search(r"\.name:\s+(\S+)", kernel)[1]] = int(
                        re.search(r"\.private_segment_fixed_size:\s+(\d+)", kernel)[1])
        at += len(MAGIC)
    return out


def test_reverse_pass_interpreters_use_no_scratch(tmp_path):
    """Tiles of 2^14 have 1024 threads of 128 registers, which two states of 16 amplitudes do not fit."""
    if not _build.LIB_PATH.exists():
        _build.build()
    found = _scratch(_build.LIB_PATH, tmp_path)
    kernels = {k: v for k, v in found.items() if re.search(r"k_(batch_adjoint|adjoint_pass|adjoint_staged)ILi", k)}
    assert len(kernels) >= 15 + 9 + 6  # every tile width, and the decoded ones
    assert {k: v for k, v in kernels.items() if v and "ILi14E" not in k} == {}


def test_specialised_reverse_passes_use_no_scratch(tmp_path):
    """Runs of diagonal gradients and phases on thread, register and outer bits, with controlled-phase layers."""
    circuit, _, _ = generators.hardware_efficient_ansatz(12, 3, seed=1)
    psum = generators.random_pauli_sum(sorted(circuit.all_qubits()), 4, 3, seed=1)
    prog = AdjointProgram(circuit, psum, adjoint_tile_bits=11)
    assert max(np.sum(prog.rev.ops_arr["kind"] == 7), 0) > 12  # GRAD_DIAG
    found = _scratch(specialize.specialize(prog.rev, cache_dir=tmp_path, adjoint=True).path, tmp_path)
    assert len(found) == int(prog.rev.n_passes) and not any(found.values()), found
