"""The interpreter's program of a group, read back on the CPU
(tests/cpp/encode_harness.cpp links the library's planner and encoder)."""
import os
import shutil
import subprocess

import numpy as np
import pytest

import oracle
from helpers import CRZ, CU1, CZ, RZ, S, T, U1, Z, to_oracle

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
CXX = "/opt/rocm/llvm/bin/clang++"
APART = 0


@pytest.fixture(scope="module")
def harness(hq, tmp_path_factory):
    cxx = CXX if os.path.exists(CXX) else shutil.which("g++")
    if cxx is None or not os.path.exists("/opt/rocm/include/hip/hip_runtime.h"):
        pytest.skip("needs a C++ compiler and the HIP headers")
    exe = tmp_path_factory.mktemp("encode") / "harness"
    lib = os.path.join(ROOT, "hyquas_amd")
    csrc = os.path.join(lib, "csrc")
    subprocess.run([cxx, "-O1", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    "-I" + os.path.join(ROOT, "include"), "-I" + os.path.join(csrc, "host"),
                    "-I" + os.path.join(csrc, "device"), os.path.join(HERE, "cpp", "encode_harness.cpp"),
                    os.path.join(lib, "libhyquas_amd.so"), "-Wl,-rpath," + lib, "-o", str(exe)], check=True)
    return exe


@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("n,mask", [(7, 0x7f), (9, 0x0ff), (10, 0x37b), (14, 0x2fff)])
def test_diagonal_gates_apart(harness, tmp_path, n, mask, prec):
    """Every gate by itself, on register, thread and block bits and across them."""
    rs = np.random.default_rng(n)
    spec = []
    for q in range(n):
        spec += [(RZ, q, -1, (float(rs.uniform(0, 6)),)), (T, q, -1), (Z, q, -1), (S, q, -1),
                 (U1, q, -1, (float(rs.uniform(0, 6)),))]
    for t in range(n):
        for c in range(n):
            if c != t and rs.uniform() < 0.3:
                spec.append([(CZ, t, c), (CU1, t, c, (float(rs.uniform(0, 6)),)),
                             (CRZ, t, c, (float(rs.uniform(0, 6)),))][int(rs.integers(0, 3))])
    g = to_oracle(spec)
    g.tofile(tmp_path / "gates.bin")
    subprocess.run([str(harness), str(n), str(prec), hex(mask), str(APART), str(tmp_path / "gates.bin"),
                    str(tmp_path / "out.bin")], check=True, timeout=60)
    got = np.fromfile(tmp_path / "out.bin", dtype=np.complex128)
    want = oracle.run_plain(g, n, np.full(1 << n, 2.0 ** (-n / 2), dtype=np.complex128)) * 2.0 ** (n / 2)
    # a factor is rounded once per gate
    assert np.abs(got - want).max() <= len(spec) * (1e-7 if prec else 4e-16)
