"""Readouts of a device state at the edges of their kernels' tiles, against
numpy in float64 on the same amplitudes."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _state(gpu, n, prec, seed):
    """A state with uploaded random amplitudes; (state, |a|^2 in float64)."""
    rs = np.random.default_rng([seed, n, prec])
    psi = rs.standard_normal((1 << n, 2)) / np.sqrt(2.0 * (1 << n))
    psi = (psi[:, 0] + 1j * psi[:, 1]).astype(np.complex128 if prec == 0 else np.complex64)
    s = gpu.State(n, gpu.HQ_C128 if prec == 0 else gpu.HQ_C64)
    s.upload(psi)
    a = psi.astype(np.complex128)
    return s, a.real ** 2 + a.imag ** 2


# below, at and above one 13-bit chunk; 8 chunk bits fill the grid at 21
# qubits, the loop over chunks starts at 22
@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("n", [1, 2, 6, 7, 9, 10, 12, 13, 14, 17, 21, 22, 24])
def test_expect_z_tiles(gpu, n, prec):
    s, p = _state(gpu, n, prec, 11)
    z, zz = s.expect_z()
    # sums of at most 2^24 terms that total about 1, in trees: far below 1e-13
    for q in range(n):
        m = p.reshape(-1, 2, 1 << q).sum((0, 2))
        assert abs(z[q] - (m[0] - m[1])) <= 1e-13, (n, q)
        if q + 1 < n:
            m = p.reshape(-1, 2, 2, 1 << q).sum((0, 3))
            assert abs(zz[q] - (m[0, 0] + m[1, 1] - m[0, 1] - m[1, 0])) <= 1e-13, (n, q)
    s.close()


def test_expect_z_largest_loop(gpu):
    """32 qubits: more than 10 loop bits.  A product state: RY(theta) on every
    third qubit, X on every seventh, |0> elsewhere."""
    n = 32
    s = gpu.State(n, gpu.HQ_C64)
    gates, want = [], np.ones(n)
    for q in range(n):
        if q % 7 == 3:
            gates.append(gpu.Gate.X(q))
            want[q] *= -1
        if q % 3 == 1:
            gates.append(gpu.Gate.RY(q, 0.3 + 0.05 * q))
            want[q] *= np.cos(0.3 + 0.05 * q)
    s.apply_plain(gates)
    z, zz = s.expect_z()
    s.close()
    # single-precision gates: one rounding of 6e-8 per coefficient and product, 15 gates
    assert np.max(np.abs(z - want)) <= 5e-6
    assert np.max(np.abs(zz - want[:-1] * want[1:])) <= 5e-6


def _draws(p, shots, seed):
    """The documented draw: the smallest index whose cumulative probability exceeds u * total."""
    from helpers import Rng
    cdf = np.cumsum(p)
    r = Rng(seed)
    u = np.array([r.uniform() for _ in range(shots)])
    return np.searchsorted(cdf, u * cdf[-1], side="right")


# one part, one chunk, several chunks, more than one and two steps of the 64-way prefix search
@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("n", [1, 5, 6, 11, 12, 13, 18, 19, 22])
def test_sample_searches(gpu, n, prec):
    s, p = _state(gpu, n, prec, 3)
    assert np.array_equal(s.sample(5000, 21).astype(np.int64), _draws(p, 5000, 21))
    s.close()


def test_sample_sparse_and_batches(gpu):
    """A state with 9 nonzero amplitudes (first and last of parts and chunks)
    and more shots than one launch takes."""
    n = 15
    idx = np.array([0, 63, 64, 4095, 4096, 9000, 20479, 20480, (1 << n) - 1])
    psi = np.zeros(1 << n, np.complex128)
    psi[idx] = np.sqrt(np.arange(1, 10) / 45.0)
    s = gpu.State(n)
    s.upload(psi)
    shots = (1 << 18) + 7
    got = s.sample(shots, 5).astype(np.int64)
    assert np.array_equal(got, _draws(np.abs(psi) ** 2, shots, 5))
    assert set(got.tolist()) <= set(idx.tolist())
    s.close()


def test_sample_without_part_sums(gpu):
    """30 qubits: a wave sums the parts of its chunk itself.  H on three qubits
    of |0...0>: eight outcomes of probability 1/8 (to float rounding)."""
    n = 30
    s = gpu.State(n, gpu.HQ_C64)
    s.apply_plain([gpu.Gate.H(q) for q in (0, 13, 29)])
    got = s.sample(4000, 9).astype(np.int64)
    s.close()
    out = np.array([a | b << 13 | c << 29 for c in (0, 1) for b in (0, 1) for a in (0, 1)])
    assert np.array_equal(got, out[_draws(np.full(8, 0.125), 4000, 9)])


# one block, several, and (2^23 amplitudes) chunks longer than 4096
@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("n", [1, 3, 4, 9, 12, 13, 17, 23])
def test_topk_lists(gpu, n, prec):
    s, p = _state(gpu, n, prec, 4)
    k = min(16, 1 << n)
    idx, prob = s.topk(k)
    order = np.lexsort((np.arange(1 << n), -p))[:k]
    assert list(idx) == order.tolist()
    np.testing.assert_allclose(prob, p[order], rtol=1e-14)
    # few nonzero amplitudes: the rest of the list are the smallest indices of probability 0
    if n >= 9:
        psi = np.zeros(1 << n, np.complex128 if prec == 0 else np.complex64)
        psi[[5, (1 << n) - 1, 300]] = [0.5, 0.5, 0.25]
        s.upload(psi)
        idx, prob = s.topk(16)
        assert list(idx) == [5, (1 << n) - 1, 300, 0, 1, 2, 3, 4, 6, 7, 8, 9, 10, 11, 12, 13]
        assert prob[3:] == [0.0] * 13
    s.close()


@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("n", [1, 2, 9, 10, 13, 20, 21])
def test_norm_and_measure_elements(gpu, n, prec):
    s, p = _state(gpu, n, prec, 8)
    assert abs(s.norm2() - p.sum()) <= 1e-13
    for q in sorted({0, min(1, n - 1), n // 2, n - 1}):
        assert abs(s.measure_zero(q) - p.reshape(-1, 2, 1 << q)[:, 0].sum()) <= 1e-13, (n, q)
    s.close()


def test_threads_share_a_state(gpu):
    """Samples and top lists of one state drawn from several threads at a time
    are those drawn one after another (both use the state's workspace)."""
    from concurrent.futures import ThreadPoolExecutor
    s, _ = _state(gpu, 16, 0, 6)
    jobs = [(k, seed) for seed in range(6) for k in (3, 16)]
    run = lambda j: (s.topk(j[0]), s.sample(500 + 4000 * (j[1] % 3), j[1]).tolist())
    want = [run(j) for j in jobs]
    s.sync()
    with ThreadPoolExecutor(4) as ex:
        assert list(ex.map(run, jobs * 2)) == want * 2
    s.close()


@pytest.mark.parametrize("prec", [0, 1])
def test_threads_read_a_fresh_state(gpu, prec):
    """Every kind of readout of one state from several threads at a time, the
    first of them growing its buffers, gives what one thread gets."""
    from concurrent.futures import ThreadPoolExecutor
    n = 15
    kinds = [lambda s: s.norm2(), lambda s: s.get_amp(12345), lambda s: [x.tolist() for x in map(np.asarray, s.expect_z())],
             lambda s: s.measure_zero(3), lambda s: s.inner(s), lambda s: s.measure_zero(n - 1),
             lambda s: s.get_amp(7), lambda s: [np.asarray(x).tolist() for x in s.topk(16)],
             lambda s: s.sample(300, 2).tolist()]
    ref, _ = _state(gpu, n, prec, 12)
    want = [k(ref) for k in kinds]
    ref.close()
    for first in range(len(kinds)):
        s, _ = _state(gpu, n, prec, 12)
        order = [(first + i) % len(kinds) for i in range(len(kinds))] * 4
        with ThreadPoolExecutor(4) as ex:
            got = list(ex.map(lambda k: kinds[k](s), order))
        s.close()
        for k, g in zip(order, got):
            assert g == want[k], (first, k)
