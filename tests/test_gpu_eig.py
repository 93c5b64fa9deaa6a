"""The direct eigensolver of the Gram method (csrc/eig.hip) against numpy's
FP64 SVD, at the sizes where its code changes: one workgroup per problem up
to 128 rows, groups of up to 4, 16 and 64 workgroups up to 256, 512 and 1024,
64-row leaves and their merges.

Spectra: random; graded (six decades); rank 3, repeated values, the identity
and zero (every merge deflates, reflectors of zero columns); two blocks and
zero rows (T splits).

Bounds, with F = ||theta||_F: the factors are complex64 (6e-8 relative per
entry, two factors), so ||a b - theta|| <= 1e-6 F and the unscaled factor is
an isometry to 1e-5; the values come from H = X X^H in FP64, known to about
n eps F^2, so within 2e-6 F.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SIZES = [65, 127, 128, 129, 192, 256, 257, 511, 512, 513, 1000, 1024]


def _haar(n, rng):
    return np.linalg.qr(rng.randn(n, n) + 1j * rng.randn(n, n))[0]


def _matrix(M, N, kind, rng):
    m = min(M, N)
    if kind == "random":
        return (rng.randn(M, N) + 1j * rng.randn(M, N)) / np.sqrt(N)
    if kind == "identity":
        return np.eye(M, N)
    if kind == "zero":
        return np.zeros((M, N))
    if kind == "blocks":
        a, h = np.zeros((M, N), complex), m // 3
        a[:h, :h] = _haar(h, rng)
        a[h + 5:2 * h, h:2 * h] = rng.randn(h - 5, h)
        return a
    s = {"graded": 10.0 ** (-6.0 * np.arange(m) / (m - 1)),
         "rank 3": np.r_[[1.0, 0.5, 0.5], np.zeros(m - 3)],
         "repeated": np.repeat([1.0, 0.5, 0.25, 1e-3], -(-m // 4))[:m]}[kind]
    return (_haar(M, rng)[:, :m] * s) @ _haar(N, rng)[:m]


def _check(A, left, r, tag):
    M, N = A.shape
    k = min(M, N)
    a = r.a_out.cpu().numpy().reshape(M, k).astype(np.complex128)
    b = r.b_out.cpu().numpy().reshape(k, N).astype(np.complex128)
    fro = max(np.linalg.norm(A), 1e-30)
    assert np.linalg.norm(a @ b - A) <= 1e-6 * fro, tag
    u = b @ b.conj().T if left else a.conj().T @ a
    assert np.linalg.norm(u - np.eye(k)) <= 1e-5, tag
    s = np.linalg.svd(A, compute_uv=False)
    assert np.max(np.abs(r.s.cpu().numpy() - s)) <= 2e-6 * fro, tag


@pytest.mark.parametrize("n", SIZES)
def test_direct_solver_sizes_and_spectra(n):
    import torch
    from mpsim_amd.engine import Engine, SplitItem
    eng = Engine.get()
    rng = np.random.RandomState(n)
    kinds = ["random", "graded", "rank 3", "repeated", "identity", "zero", "blocks"]
    if n > 513:
        kinds = ["random", "rank 3", "blocks"]
    cases = [(n, n, kind, False) for kind in kinds]
    cases += [(n, n + 37, "random", False), (n + 20, n, "random", True), (n, 3 * n // 4, "graded", False),
              (n, n // 4, "random", False)]
    mats = [_matrix(M, N, kind, rng).astype(np.complex64) for M, N, kind, _ in cases]
    items = [SplitItem(torch.from_numpy(A).cuda(), min(A.shape), absorb_left=left, want_s=True)
             for A, (_, _, _, left) in zip(mats, cases)]
    print(f"n={n}: one grouped call", flush=True)
    res = eng.two_site(items)
    torch.cuda.synchronize()
    for A, c, r in zip(mats, cases, res):
        print("case", c, flush=True)
        _check(A.astype(np.complex128), c[3], r, c)


def test_direct_solver_is_the_same_alone_and_in_a_batch():
    """Bitwise: a problem's workgroups exchange only their own values."""
    import torch
    from mpsim_amd.engine import Engine, SplitItem
    eng = Engine.get()
    rng = np.random.RandomState(3)
    mats = [torch.from_numpy(_matrix(n, n, "random", rng).astype(np.complex64)).cuda()
            for n in (300, 100, 512, 130, 600, 256)]
    res = eng.two_site([SplitItem(m, m.shape[0], want_s=True) for m in mats])
    torch.cuda.synchronize()
    for m, r in zip(mats, res):
        print("alone", tuple(m.shape), flush=True)
        one = eng.two_site([SplitItem(m, m.shape[0], want_s=True)])[0]
        torch.cuda.synchronize()
        for x, y in ((one.a_out, r.a_out), (one.b_out, r.b_out), (one.s, r.s)):
            assert torch.equal(x, y), tuple(m.shape)
