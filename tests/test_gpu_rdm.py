"""Reduced density matrices with traced sites before, between and after kept ones.

rho = M M^H of a state vector; the sweep makes 2 n FP32 contractions of at most k = 14
terms a sum, each off by less than (2 k + 16) 2^-23 of its absolute sum; random
tensors keep the absolute sums within sqrt(terms) ~ 4 of the sums themselves."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d,bonds,kept", [(2, [3, 5, 4, 6, 2], [2]), (2, [3, 5, 4, 6, 2], [1, 3]),
                                          (2, [1, 1, 2, 7, 3], [0, 2, 5]), (3, [3, 4, 5], [1, 2]),
                                          (3, [2, 4, 3, 2], [0, 3]), (2, [2, 3], [0, 1, 2])])
def test_reduced_density_matrix_of_uneven_chains(d, bonds, kept):
    import torch
    from mpsim_amd import MPS
    rng = np.random.RandomState(sum(bonds))
    n, b = len(bonds) + 1, [1] + bonds + [1]
    ts = [(rng.randn(b[i], d, b[i + 1]) + 1j * rng.randn(b[i], d, b[i + 1])).astype(np.complex64) for i in range(n)]
    mps = MPS(n, d)
    mps.tensors[:] = [torch.from_numpy(t).cuda() for t in ts]
    psi = ts[0].astype(np.complex128).reshape(d, -1)
    for t in ts[1:]:
        psi = (psi @ t.reshape(t.shape[0], -1).astype(np.complex128)).reshape(-1, t.shape[2])
    rest = [i for i in range(n) if i not in kept]
    m = psi.reshape([d] * n).transpose(kept + rest).reshape(d ** len(kept), -1)
    want = m @ m.conj().T
    got = mps.reduced_density_matrix(kept)
    assert np.linalg.norm(got - want) <= 2 * n * 4 * (2 * 14 + 16) * 2.0 ** -23 * np.linalg.norm(want)
