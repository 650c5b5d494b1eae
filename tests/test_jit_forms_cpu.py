"""Forms the specialised kernel generator gives its ops, read from the source it
emits (no GPU).  What the kernels compute is checked in test_jit_cpu.py."""
import re

import pytest

from helpers import CNOT, CU1, H, RZ, to_oracle

N, MASK = 13, (1 << 13) - 1


def _source(hq, spec, prec=0, variant=0, n=N, mask=MASK):
    return hq.sharemem_source(n, to_oracle(spec), mask, prec, 0, variant)[0]


@pytest.mark.parametrize("variant", [0, 1, 4, 20])
@pytest.mark.parametrize("prec", [0, 1])
def test_x_under_a_thread_bit_control(hq, prec, variant):
    """The 2x2 update with per-lane 0 and 1: by selects, the kernels of 22 to 31
    qubits were up to 4 % slower."""
    spec = [(H, q, -1) for q in range(N)] + [(CNOT, t, c) for t in range(4) for c in range(6, 12)]
    src = _source(hq, spec, prec, variant)
    assert re.search(r"const R m0 = pc \? \(R\)0 : \(R\)1", src)
    assert not re.search(r"= pc \? hi\.x : lo\.x", src)


@pytest.mark.parametrize("variant", [0, 1, 4, 20])
@pytest.mark.parametrize("prec", [0, 1])
def test_factors_of_diagonal_gates_are_loaded_outside_conditions(hq, prec, variant):
    """A coefficient loaded where a lane's condition selects it is a branch, with
    copies of every amplitude at its join."""
    spec = [(H, q, -1) for q in range(N)]
    spec += [(CU1, t, c, (0.1 + t + c,)) for t in range(N) for c in range(t)] + [(RZ, q, -1, (0.3,)) for q in range(N)]
    src = _source(hq, spec, prec, variant)
    assert "? kr : (R)1" in src
    assert not re.search(r"\? *cf\[", src)


@pytest.mark.parametrize("variant", [0, 1, 4, 20])
@pytest.mark.parametrize("prec", [0, 1])
def test_diagonal_gates_across_block_bits_do_not_branch(hq, prec, variant):
    """A gate on a register bit and a block bit touches half a thread's
    amplitudes: its factor is selected by the block, without a branch around them."""
    n = 18
    spec = [(H, q, -1) for q in range(N)]
    spec += [(CU1, t, c, (0.1 + t + c,)) for t in range(N) for c in range(N, n)]
    spec += [(CU1, c, t, (0.2 + t + c,)) for t in range(N) for c in range(N, n)] + [(H, q, -1) for q in range(N)]
    src = _source(hq, spec, prec, variant, n)
    assert re.search(r"pc = \(b & 0x[0-9a-f]+ull\) == 0x[0-9a-f]+ull;", src)
    assert "if ((b & " not in src


@pytest.mark.parametrize("gates", [1, 2, 255, 256, 257, 258])
def test_products_of_many_factors_keep_two_floats(hq, gates):
    """A table entry of a complex64 program that is a product of several gates'
    factors is held as two floats, however many they are."""
    # between two H the target is a register bit, and the gates stay in one table
    spec = [(H, 0, -1)] + [(RZ, 0, -1, (0.01 * (i + 1),)) for i in range(gates)] + [(H, 0, -1)]
    src = _source(hq, spec, 1)
    assert bool(re.search(r"const R ex\d+ = cf\[", src)) == (gates > 1)
