"""Forms the specialised kernel generator gives its ops, read from the source it
emits (no GPU).  What the kernels compute is checked in test_jit_cpu.py."""
import re

import pytest

from helpers import CNOT, H, to_oracle

N, MASK = 13, (1 << 13) - 1


def _source(hq, spec, prec=0, variant=0, n=N, mask=MASK):
    return hq.sharemem_source(n, to_oracle(spec), mask, prec, 0, variant)[0]


@pytest.mark.parametrize("variant", [0, 1, 4, 20])
@pytest.mark.parametrize("prec", [0, 1])
def test_x_under_a_thread_bit_control(hq, prec, variant):
    """Selects in complex64, in complex128 the 2x2 update with per-lane 0 and 1:
    both take eight operations a pair there, and the kernels of 22 to 25 qubits
    were 2 to 4 % slower by selects."""
    spec = [(H, q, -1) for q in range(N)] + [(CNOT, t, c) for t in range(4) for c in range(6, 12)]
    src = _source(hq, spec, prec, variant)
    selects = re.findall(r"= pc \? hi\.x : lo\.x", src)
    updates = re.findall(r"const R m0 = pc \? \(R\)0 : \(R\)1", src)
    assert "const bool pc" in src
    assert (len(selects) > 0) == (prec == 1)
    assert (len(updates) > 0) == (prec == 0)
