"""The grouped product at the edges of its tiles, in every operand form, against FP64.

Bound per entry: a real sum of n FP32 products is off by at most
(n + 1) 2^-24 sum |a||b| to first order; an entry has two such sums of k terms in each
part, their difference and the product with alpha: (2 k + 16) 2^-23 (|A| |B|) |alpha|."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# (m, n, k, products): thin, mid and wide tiles and their remainders
SHAPES = [(1, 1, 1, 1), (1, 1, 4097, 3), (15, 17, 33, 1), (16, 16, 64, 1), (65, 129, 40, 1), (256, 300, 48, 1),
          (449, 417, 35, 1), (33, 31, 47, 200), (64, 65, 36, 96), (900, 1030, 50, 1), (2049, 400, 33, 1),
          (130, 5, 0, 1)]


@pytest.mark.parametrize("flags", range(8))
@pytest.mark.parametrize("m,n,k,count", SHAPES)
def test_grouped_products_against_fp64(m, n, k, count, flags):
    import torch
    from mpsim_amd.engine import Engine
    rng = np.random.RandomState(m + 3 * n + 7 * k + flags)
    dev = torch.device("cuda")

    def operand(rows, cols, odd):
        # odd: an odd row stride and start, so that rows are 8-byte aligned only
        ld = cols + 1 + (cols + odd + 1) % 2 if odd else cols + cols % 2
        off = 3 if odd else 0
        buf = (rng.randn(off + rows * ld) + 1j * rng.randn(off + rows * ld)).astype(np.complex64)
        mat = buf[off:].reshape(rows, ld)[:, :cols].astype(np.complex128)
        return torch.from_numpy(buf).to(dev), off, ld, mat

    ops, want, outs = [], [], []
    alpha = 0.75 - 0.5j
    for i in range(count):
        odd = i % 2 if count > 1 else flags & 1
        ra, ca = (k, m) if flags & 1 else (m, k)
        rb, cb = (n, k) if flags & 2 else (k, n)
        a, ao, lda, am = operand(max(ra, 1), max(ca, 1), odd)
        b, bo, ldb, bm = operand(max(rb, 1), max(cb, 1), odd)
        c, co, ldc, cm = operand(m, n, odd)
        am, bm = am[:ra, :ca], bm[:rb, :cb]
        am = am.conj().T if flags & 1 else am
        bm = bm.conj().T if flags & 2 else bm
        w = alpha * (am @ bm) + (cm if flags & 4 else 0)
        bound = (2 * k + 16) * 2.0 ** -23 * (abs(alpha) * (abs(am) @ abs(bm)) + (abs(cm) if flags & 4 else 0))
        ops.append(dict(A=(a, ao), B=(b, bo), C=(c, co), m=m, n=n, k=k, lda=lda, ldb=ldb, ldc=ldc, flags=flags,
                        alpha=alpha))
        want.append((w, bound, ldc, co))
        outs.append((c, c.clone()))
    Engine.get().gemm(ops)
    for (w, bound, ldc, co), (c, before) in zip(want, outs):
        got = c.cpu().numpy()[co:].reshape(m, ldc)
        assert (abs(got[:, :n] - w) <= bound).all()
        # nothing beside the matrix is written
        old = before.cpu().numpy()
        assert np.array_equal(got[:, n:], old[co:].reshape(m, ldc)[:, n:]) and np.array_equal(
            c.cpu().numpy()[:co], old[:co])


def test_infinities_stay_in_their_row_and_column():
    import torch
    from mpsim_amd.engine import Engine
    m, n, k = 35, 37, 50
    rng = np.random.RandomState(5)
    a = rng.randn(m, k).astype(np.complex64)
    b = rng.randn(k, n).astype(np.complex64)
    a[34, 49], b[0, 36] = np.inf, np.nan
    c = torch.empty((m, n), dtype=torch.complex64, device="cuda")
    Engine.get().gemm([dict(A=torch.from_numpy(a).cuda(), B=torch.from_numpy(b).cuda(), C=c, m=m, n=n, k=k,
                            lda=k, ldb=n, ldc=n)])
    got = c.cpu().numpy()
    assert np.isfinite(got[:34, :36]).all()
    assert not np.isfinite(got[34]).any() and not np.isfinite(got[:, 36]).any()
