"""Gates that share a pass of the plain path leave the amplitudes they do not select untouched, as
one gate a pass does: also an infinite one, which a product with 1 + 0i would
make NaN."""
import numpy as np
import pytest

import oracle
from helpers import CCX, CNOT, CRX, CRZ, CU1, CY, CZ, S, T, U1, Y, Z, random_mixed, rel_err, to_oracle

pytestmark = pytest.mark.gpu


# 12 qubits take 8 amplitudes a thread, 19 take 16
@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("n", [12, 19])
def test_unselected_amplitude_stays_infinite(gpu, n, prec):
    rs = np.random.default_rng([n, prec])
    spec = []
    for _ in range(60):
        a, b, c = (int(x) for x in rs.choice(n, 3, replace=False))
        t = float(rs.uniform(0.1, 6))
        # none of these touches the amplitude of |0...0>
        spec.append([(T, a, -1), (S, a, -1), (Z, a, -1), (U1, a, -1, (t,)), (CZ, a, b), (CU1, a, b, (t,)),
                     (CRZ, a, b, (t,)), (CNOT, a, b), (CY, a, b), (CRX, a, b, (t,)), (CCX, a, b, (), c)]
                    [int(rs.integers(0, 11))])
    # in pairs, Y moves it and brings it back
    for q in range(n):
        spec += [(Y, q, -1), (Y, q, -1)]
    g = to_oracle(spec)
    psi = rs.standard_normal((1 << n, 2)) / np.sqrt(2.0 * (1 << n))
    psi = (psi[:, 0] + 1j * psi[:, 1]).astype(np.complex64 if prec else np.complex128)
    psi[0] = 0
    want = oracle.run_plain(g, n, psi.astype(np.complex128))
    psi[0] = complex(np.inf, 0)
    s = gpu.State(n, gpu.HQ_C64 if prec else gpu.HQ_C128)
    s.upload(psi)
    s.apply_plain(g)
    got = s.download()
    s.close()
    assert got[0].real == np.inf and got[0].imag == 0
    assert np.isfinite(got[1:]).all()
    got[0] = 0
    assert rel_err(got, want) <= 4 * np.sqrt(len(spec)) * (6e-8 if prec else 1.2e-16)


# 19 qubits: 16 amplitudes a thread.  Lane targets alone fill runs of 32 gates;
# four high targets are the register bits, the fourth among them, with controls
# on them and elsewhere; any targets take every form
@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("m,targets", [(300, range(6)), (200, range(15, 19)), (200, [6, 9, 12, 18]), (300, None)])
def test_sixteen_amplitude_runs(gpu, m, targets, prec):
    n = 19
    spec = [g for g in random_mixed(n, 12 * m, 77 + m) if targets is None or g[1] in targets][:m]
    assert len(spec) == m
    g = to_oracle(spec)
    rs = np.random.default_rng(m)
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
