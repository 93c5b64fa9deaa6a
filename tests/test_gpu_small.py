"""The one-workgroup kernel of small problems (csrc/small.hip, up to 64 rows of
at most 512 columns) against numpy's FP64 SVD: every way through it (nothing
to rotate; Jacobi up to 8 rows; the direct route from 9 on; further passes for
graded and rank-deficient spectra), partial 16-row tiles, one row, tall and
wide shapes, both orientations, and the first size beyond it in either
direction (65 rows, 513 columns).

Bounds, F = ||theta||_F: complex64 factors, so ||a b - theta|| <= 1e-6 F and an
isometry to 1e-5; the values of the one-sided test (every pair of rows
orthogonal within 1e-7 of their norms), so 1e-4 sigma_i on every value above
the null threshold (1e-9 F), as for the one-sided rounds.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _haar(n, rng):
    return np.linalg.qr(rng.randn(n, n) + 1j * rng.randn(n, n))[0]


def _matrix(M, N, kind, rng):
    m = min(M, N)
    if kind == "random":
        return (rng.randn(M, N) + 1j * rng.randn(M, N)) / np.sqrt(N)
    if kind == "diagonal":  # orthogonal rows, out of order
        return np.eye(M, N) * (1.0 + np.arange(M) % 3)[:, None]
    if kind == "zero":
        return np.zeros((M, N))
    s = {"graded": 10.0 ** (-6.0 * np.arange(m) / max(m - 1, 1)),
         "rank 2": np.r_[[1.0, 0.5], np.zeros(max(m - 2, 0))][:m],
         "repeated": np.repeat([1.0, 0.5, 1e-3], -(-m // 3))[:m]}[kind]
    return (_haar(M, rng)[:, :m] * s) @ _haar(N, rng)[:m]


def _check(A, k, left, r, tag):
    M, N = A.shape
    a = r.a_out.cpu().numpy().reshape(M, k).astype(np.complex128)
    b = r.b_out.cpu().numpy().reshape(k, N).astype(np.complex128)
    fro = max(np.linalg.norm(A), 1e-30)
    u, s, vh = np.linalg.svd(A, full_matrices=False)
    best = (u[:, :k] * s[:k]) @ vh[:k]
    if k == len(s) or s[k - 1] - s[k] > 1e-2 * s[0]:  # a cut inside a cluster has no unique best
        assert np.linalg.norm(a @ b - best) <= 1e-6 * fro, tag
    iso = b @ b.conj().T if left else a.conj().T @ a
    assert np.linalg.norm(iso - np.eye(k)) <= 1e-5, tag
    got = r.s.cpu().numpy().astype(np.float64)
    big = s[:k] > 1e-6 * fro  # values well above the complex64 rounding of A itself
    assert np.all(np.abs(got - s[:k])[big] <= 1e-4 * s[:k][big]), tag
    assert np.all(np.abs(got - s[:k]) <= 1e-6 * fro), tag
    assert abs(float(r.discarded.cpu()) - np.sum(s[k:] ** 2)) <= 1e-6 * fro ** 2, tag


@pytest.mark.parametrize("n", [1, 2, 3, 4, 7, 8, 9, 15, 16, 17, 31, 33, 48, 63, 64, 65])
def test_small_sizes_and_spectra(n):
    import torch
    from mpsim_amd.engine import Engine, SplitItem
    eng = Engine.get()
    rng = np.random.RandomState(n)
    cases = [(n, n, kind, n, False) for kind in ("random", "graded", "rank 2", "repeated", "diagonal", "zero")]
    cases += [(n, n + 29, "random", n, False), (n + 29, n, "random", n, True), (n, 512, "random", n, False),
              (n, 513, "graded", n, False), (n, max(1, n // 3), "random", max(1, n // 3), False),
              (n, 2 * n, "random", max(1, n // 2), False), (2 * n, n, "graded", max(1, n // 2), True)]
    mats = [_matrix(M, N, kind, rng).astype(np.complex64) for M, N, kind, _, _ in cases]
    items = [SplitItem(torch.from_numpy(A).cuda(), k, absorb_left=left, want_s=True)
             for A, (_, _, _, k, left) in zip(mats, cases)]
    print(f"n={n}: one grouped call", flush=True)
    res = eng.two_site(items)
    torch.cuda.synchronize()
    for A, c, r in zip(mats, cases, res):
        print("case", c, flush=True)
        _check(A.astype(np.complex128), c[3], c[4], r, c)
        print("alone", flush=True)
        one = eng.two_site([SplitItem(torch.from_numpy(A).cuda(), c[3], absorb_left=c[4], want_s=True)])[0]
        torch.cuda.synchronize()
        assert torch.equal(one.a_out, r.a_out) and torch.equal(one.b_out, r.b_out) and torch.equal(one.s, r.s), c


@pytest.mark.parametrize("d,cl,cm,cr,k,left", [(2, 1, 1, 1, 2, False), (2, 5, 7, 3, 4, True), (3, 21, 10, 9, 20, False),
                                               (4, 16, 5, 4, 16, False), (5, 3, 4, 12, 15, True), (16, 4, 3, 2, 30, False)])
def test_small_two_site_updates(d, cl, cm, cr, k, left):
    """Gates on site tensors of every qudit dimension's theta kernel."""
    import torch
    from mpsim_amd import gates
    from mpsim_amd.engine import Engine, TwoSiteItem
    eng = Engine.get()
    rng = np.random.RandomState(d)
    A = ((rng.randn(cl, d, cm) + 1j * rng.randn(cl, d, cm)) / np.sqrt(2 * d * cm)).astype(np.complex64)
    B = ((rng.randn(cm, d, cr) + 1j * rng.randn(cm, d, cr)) / np.sqrt(2)).astype(np.complex64)
    G = gates.haar_unitary(d * d, rng).astype(np.complex64)
    t = np.einsum("abpq,lpqr->labr", G.reshape(d, d, d, d).astype(np.complex128),
                  np.tensordot(A.astype(np.complex128), B.astype(np.complex128), axes=([2], [0])))
    theta = t.reshape(d * cl, d * cr)
    print("update", (d, cl, cm, cr, k, left), flush=True)
    r = eng.two_site([TwoSiteItem(torch.from_numpy(A).cuda(), torch.from_numpy(B).cuda(), eng.gate(G), k,
                                  absorb_left=left, want_s=True)])[0]
    torch.cuda.synchronize()
    _check(theta, k, left, r, (d, cl, cm, cr, k, left))
