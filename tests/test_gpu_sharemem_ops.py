"""Interpreter programs at the edges of their slots: several windows of ops,
tables and lane factors of merged diagonal gates, and groups whose factored
scalars would leave float's range."""
import numpy as np
import pytest

import oracle
from helpers import CCX, CNOT, CRZ, CU1, CZ, H, RX, RY, RZ, S, T, X, Y, Z, U3, rel_err, to_oracle

pytestmark = pytest.mark.gpu


def _diagonal_heavy(n, tile, m, seed):
    """Random gates, two thirds diagonal, non-diagonal targets inside the tile; controls anywhere."""
    rs = np.random.default_rng(seed)
    out = []
    for _ in range(m):
        q = [int(x) for x in rs.choice(n, 3, replace=False)]
        t = int(rs.choice(tile))
        c = [x for x in q if x != t]
        a = (float(rs.uniform(0, 2 * np.pi)),)
        k = int(rs.integers(0, 18))
        if k < 4: out.append((RZ, q[0], -1, a))
        elif k < 6: out.append((T, q[0], -1))
        elif k < 8: out.append((CZ, q[0], q[1]))
        elif k < 9: out.append((CU1, q[0], q[1], a))
        elif k < 10: out.append((CRZ, q[0], q[1], a))
        elif k < 11: out.append((Z if k % 2 else S, q[0], -1))
        elif k < 12: out.append((X, t, -1))
        elif k < 13: out.append((Y, t, -1))
        elif k < 14: out.append((CNOT, t, c[0]))
        elif k < 15: out.append((CCX, t, c[0], (), c[1]))
        elif k < 16: out.append((H, t, -1))
        elif k < 17: out.append((RX if rs.random() < .5 else RY, t, -1, a))
        else: out.append((U3, t, -1, (a[0], 0.3, 0.7)))
    return to_oracle(out)


# 96 (complex128) and 160 (complex64) slots a window; tiles with one and with
# several register bits, and block bits beside them
@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("n,k,m", [(7, 7, 40), (9, 8, 200), (12, 12, 700), (14, 10, 150), (15, 12, 500),
                                   (14, 13, 300)])
def test_merged_diagonals_match_oracle(gpu, n, k, m, prec):
    tile = list(range(2)) + sorted(int(x) for x in np.random.default_rng(n).choice(np.arange(2, n), k - 2,
                                                                                  replace=False))
    g = _diagonal_heavy(n, tile, m, 100 * n + k)
    rs = np.random.default_rng(5)
    psi = rs.standard_normal((1 << n, 2))
    psi = (psi[:, 0] + 1j * psi[:, 1]) / np.linalg.norm(psi)
    psi = psi.astype(np.complex128 if prec == 0 else np.complex64)
    want = oracle.run_plain(g, n, psi.astype(np.complex128))
    s = gpu.State(n, gpu.HQ_C128 if prec == 0 else gpu.HQ_C64)
    # one rounding of 1.1e-16 (6e-8) per gate and a few per merged factor, adding in squares
    tol = 4 * np.sqrt(m) * (1.2e-16 if prec == 0 else 6e-8)
    for specialised in (False, True) if m <= 200 else (False,):
        s.upload(psi)
        p = s.program_sharemem(g, sum(1 << q for q in tile))
        if specialised:
            p.specialize()
        s.launch(p)
        assert rel_err(s.download(), want) <= tol, specialised
    s.close()


@pytest.mark.parametrize("family", ["random", "ansatz"])
def test_deep_whole_state_group_stays_in_range(gpu, family):
    """13 qubits, 150 layers in one complex64 group: the amplitudes grow by
    the factored scalars' inverse, far beyond 2^127 if it were applied once."""
    c = gpu.Circuit(13)
    (c.add_random_layers if family == "random" else c.add_hea_layers)(150, 7)
    e = gpu.Engine(gpu.HQ_C64, 1 << 28)
    d = gpu.Engine(gpu.HQ_C128, 1 << 28)
    r, x = [], []
    for eng, out in ((e, r), (d, x)):
        j = eng.submit(c, gpu.HQ_OUT_EXPECT)
        eng.drain()
        out.append(eng.result(j))
        eng.close()
    # 1950 to 3900 gates of 6e-8 each, adding in squares for the state and at
    # worst linearly for its norm
    assert abs(r[0]["norm"] - 1) <= 3900 * 6e-8
    assert abs(r[0]["z"] - x[0]["z"]) <= 13 * 3900 * 6e-8
