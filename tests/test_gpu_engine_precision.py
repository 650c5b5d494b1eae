"""Complex64 engines against complex128 at a size where merged diagonal factors,
rounded once for a whole circuit, meet expectation values far below 1."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _sums(gpu, prec, jit, n, layers, seeds, family):
    e = gpu.Engine(prec, 8 << 30)
    e.set_option("jit", jit)
    e.set_option("compile_threads", 8)
    jobs = []
    for s in seeds:
        c = gpu.Circuit(n)
        (c.add_hea_layers if family == "ansatz" else c.add_random_layers)(layers, s)
        jobs.append(e.submit(c))
    e.drain()
    e.poll()
    out = np.array([[r["norm"], r["z"], r["zz"]] for r in (e.result(j) for j in jobs)])
    e.close()
    return out


@pytest.mark.parametrize("family,jit", [("ansatz", 0), ("ansatz", 1), ("random", 0)])
def test_large_circuits(gpu, family, jit):
    n, layers, seeds = 24, 24, range(3)
    want = _sums(gpu, gpu.HQ_C128, 0, n, layers, seeds, family)
    got = _sums(gpu, gpu.HQ_C64, jit, n, layers, seeds, family)
    # one rounding of 6e-8 for each of the n * layers * 2 rotations, adding in
    # squares, twice in a probability
    assert np.abs(got - want).max() <= 2 * 6e-8 * np.sqrt(2 * n * layers)
