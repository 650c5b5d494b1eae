"""Runs of gates that share one pass on the plain path: lane, register and other
targets, controls and diagonal gates anywhere, runs longer than a launch holds,
the smallest states that take them and the ones below, against the oracle."""
import numpy as np
import pytest

import oracle
from helpers import CU1, CZ, H, random_mixed, rel_err, to_oracle

pytestmark = pytest.mark.gpu


def _gates(n, m, seed, targets):
    """m random gates of every type, targets among the given ones."""
    out = [g for g in random_mixed(n, m * (n if targets else 1), seed) if targets is None or g[1] in targets]
    return to_oracle(out[:m])


@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("n,m,targets", [
    (3, 30, None), (9, 60, None), (10, 120, None), (11, 300, None), (13, 300, None),
    (13, 100, range(6)), (13, 100, range(6, 10)), (13, 100, [0, 5, 6, 12]), (18, 200, None), (22, 40, None)])
def test_runs_match_oracle(gpu, n, m, targets, prec):
    g = _gates(n, m, 1000 * n + m, targets)
    rs = np.random.default_rng(n)
    psi = rs.standard_normal((1 << n, 2))
    psi = (psi[:, 0] + 1j * psi[:, 1]) / np.linalg.norm(psi)
    psi = psi.astype(np.complex64 if prec else np.complex128)
    s = gpu.State(n, gpu.HQ_C64 if prec else gpu.HQ_C128)
    s.upload(psi)
    s.apply_plain(g)
    # a few roundings of 1.1e-16 (6e-8) per gate, adding in squares
    assert rel_err(s.download(), oracle.run_plain(g, n, psi.astype(np.complex128))) <= \
        4 * np.sqrt(m) * (6e-8 if prec else 1.2e-16)
    s.close()


def test_gates_that_do_not_fill_a_pass(gpu):
    """24 qubits: phases under controls that together touch less than one pass
    stay single, the same gates beside others join a run; same state."""
    n = 24
    few = to_oracle([(CU1, 3, 20, (0.3,)), (CZ, 22, 7)])
    s = gpu.State(n)
    s.apply_plain(to_oracle([(H, q, -1) for q in range(n)]))
    s.apply_plain(few)
    a = s.download()
    s.reset()
    s.apply_plain(to_oracle([(H, q, -1) for q in range(n)] + [(CU1, 3, 20, (0.3,)), (CZ, 22, 7)]))
    b = s.download()
    s.close()
    i = np.arange(1 << n)
    want = np.exp(0.3j * ((i >> 3) & (i >> 20) & 1)) * (1 - 2 * ((i >> 22) & (i >> 7) & 1)) / 4096
    for got in (a, b):
        assert np.abs(got - want).max() <= 30 * 1.2e-16 / 4096
