"""TransMM in complex64 at K = 64, whose tiles are 32 columns wide: the smallest
states of the MFMA form, the state below them, and tile counts around the
number of blocks a launch keeps resident."""
import numpy as np
import pytest

from helpers import rel_err
from test_gpu_kernels import _rand_state, _rand_unitary, dense_at_reference

pytestmark = pytest.mark.gpu

# 64 products of rounded inputs summed in FP32: 6e-8 * (3 + sqrt(64)) at most in the 2-norm
TOL = 7e-7


@pytest.mark.parametrize("n", [10, 11, 12, 13, 21])
def test_lowest_qubits(gpu, n):
    U, psi0 = _rand_unitary(64, n), _rand_state(n, 40 + n)
    colmajor = U.T.reshape(-1)
    s = gpu.State(n, gpu.HQ_C64, with_buffer=True)
    s.upload(psi0.astype(np.complex64))
    s.apply_dense(colmajor, 6)
    assert rel_err(s.download(), dense_at_reference(psi0, n, list(range(6)), U)) <= TOL
    s.close()


@pytest.mark.parametrize("n,positions", [(12, [11, 0, 5, 7, 2, 9]), (12, [6, 7, 8, 9, 10, 11]),
                                         (13, [1, 12, 3, 10, 5, 8]), (21, [20, 1, 18, 4, 11, 0])])
def test_any_qubits(gpu, n, positions):
    U, psi0 = _rand_unitary(64, 7 * n), _rand_state(n, 80 + n)
    s = gpu.State(n, gpu.HQ_C64)
    s.upload(psi0.astype(np.complex64))
    p = s.program_dense(positions, U.T.reshape(-1))
    s.launch(p)
    s.sync()
    assert rel_err(s.download(), dense_at_reference(psi0, n, positions, U)) <= TOL
    p.close()
    s.close()


def test_one_tile_below_is_refused(gpu):
    s = gpu.State(11, gpu.HQ_C64)
    with pytest.raises(RuntimeError):
        s.program_dense([0, 1, 2, 3, 4, 5], np.eye(64).reshape(-1))
    s.close()
