"""Equal singular values of rows that nothing couples keep the rows' order ("ties in
input order", include/mpsx.h), whichever kernel takes the problem: the factors of a
diagonal matrix are then known exactly. Sizes around the limits of the kernels
(64 rows one workgroup, 64-row leaves of the direct solver, 1024 rows) and
truncated, so that the order decides which values are kept; and where the serial
deflation runs beside such rows.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _split(mats, k):
    import torch
    from mpsim_amd.engine import Engine, SplitItem
    res = Engine.get().two_site([SplitItem(torch.from_numpy(m.astype(np.complex64)).cuda(), kk, want_s=True)
                                 for m, kk in zip(mats, k)])
    torch.cuda.synchronize()
    return res


@pytest.mark.parametrize("n", [8, 63, 64, 65, 96, 128, 129, 200, 256, 513, 1024, 1040])
def test_tied_rows_keep_their_order(n):
    i = np.arange(n)
    diags = [np.ones(n), np.where(i % 3 == 1, 2.0, 1.0), np.where(i < n // 3, 0.0, 1.0 + i % 2)]
    ks = [n, max(1, n // 2), max(1, n // 2)]
    print("rows", n, flush=True)
    for v, k, r in zip(diags, ks, _split([np.diag(v) for v in diags], ks)):
        order = np.argsort(-v, kind="stable")[:k]
        assert np.array_equal(r.s.cpu().numpy(), v[order].astype(np.float32)), n
        # absorb right: column j of a_out is the unit vector of row order[j]
        assert np.array_equal(np.abs(r.a_out.cpu().numpy().reshape(n, k)), np.eye(n)[:, order]), n


@pytest.mark.parametrize("n", [100, 300, 640])
def test_tied_rows_beside_coupled_ones(n):
    """A dense block of repeated values (whose merges rotate poles together) between
    two stretches of tied rows that it does not touch."""
    rng = np.random.RandomState(n)
    h = n // 3
    q = np.linalg.qr(rng.randn(h, h) + 1j * rng.randn(h, h))[0]
    q2 = np.linalg.qr(rng.randn(h, h) + 1j * rng.randn(h, h))[0]
    m = np.zeros((n, n), complex)
    m[:h, :h] = 3.0 * np.eye(h)
    m[h:2 * h, h:2 * h] = (q * np.repeat([1.0, 0.5, 0.25, 0.125], -(-h // 4))[:h]) @ q2
    m[2 * h:, 2 * h:] = 3.0 * np.eye(n - 2 * h)
    print("rows", n, flush=True)
    r = _split([m], [n])[0]
    a = r.a_out.cpu().numpy().reshape(n, n)
    b = r.b_out.cpu().numpy().reshape(n, n)
    assert np.linalg.norm(a.astype(complex) @ b - m) <= 1e-6 * np.linalg.norm(m)
    order = np.r_[np.arange(h), np.arange(2 * h, n)]
    # (to the rounding that the block's rows leave in the reflectors' products)
    assert np.max(np.abs(np.abs(a[:, :len(order)]) - np.eye(n)[:, order])) <= 1e-6
