"""The grouped product where its matrices fill little of the tile that the device could
be filled with, so that a smaller one is taken (16, 24, 40, 65 and 80 of 64 columns;
batches of small squares), and where such matrices share a launch with others (which
keeps the larger tile). Against FP64, with the bound of test_gpu_gemm."""
import numpy as np
import pytest

from test_gpu_gemm import test_grouped_products_against_fp64 as against_fp64

pytestmark = pytest.mark.gpu

# (m, n, k, products)
SHAPES = [(20000, 3, 33, 1), (17, 14000, 41, 1), (13000, 24, 40, 1), (13000, 40, 36, 1), (7000, 80, 35, 1),
          (8, 8, 40, 300), (17, 17, 50, 250), (65, 65, 40, 60)]


@pytest.mark.parametrize("flags", [0, 3, 6])
@pytest.mark.parametrize("m,n,k,count", SHAPES)
def test_narrow_products_against_fp64(m, n, k, count, flags):
    against_fp64(m, n, k, count, flags)


def test_narrow_products_beside_others():
    import torch
    from mpsim_amd.engine import Engine
    rng = np.random.RandomState(11)
    k, ops, want = 40, [], []
    for m, n in [(7000, 2), (3, 7000), (200, 210), (1, 1)] * 12:
        a = (rng.randn(m, k) + 1j * rng.randn(m, k)).astype(np.complex64)
        b = (rng.randn(k, n) + 1j * rng.randn(k, n)).astype(np.complex64)
        c = torch.empty((m, n), dtype=torch.complex64, device="cuda")
        ops.append(dict(A=torch.from_numpy(a).cuda(), B=torch.from_numpy(b).cuda(), C=c, m=m, n=n, k=k, lda=k, ldb=n,
                        ldc=n))
        a, b = a.astype(np.complex128), b.astype(np.complex128)
        want.append((a @ b, (2 * k + 16) * 2.0 ** -23 * (abs(a) @ abs(b))))
    Engine.get().gemm(ops)
    for o, (w, bound) in zip(ops, want):
        assert (abs(o["C"].cpu().numpy() - w) <= bound).all(), (o["m"], o["n"])
