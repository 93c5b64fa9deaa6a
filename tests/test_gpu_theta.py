"""theta at the edges of the matrix-core kernel's tiles, through an untruncated update.

The factors are rounded to complex64 from FP64 ones: with a unitary, |da| <= 2^-24 |a| and
|db| <= 2^-24 |b| entry by entry, so ||a b - theta||_F <= 2^-24 (sqrt(k) + 1) ||theta||_F,
and nothing else is of that size (theta itself is exact to FP64 rounding)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d", [2, 3])
@pytest.mark.parametrize("cl,cm,cr", [(1, 1, 1), (2, 1, 3), (5, 15, 4), (16, 16, 16), (17, 17, 15), (15, 33, 18),
                                      (31, 32, 33), (33, 48, 32), (3, 130, 65), (70, 7, 2), (64, 37, 31)])
@pytest.mark.parametrize("left", [False, True])
def test_untruncated_update_against_fp64(d, cl, cm, cr, left):
    import torch
    from mpsim_amd.engine import Engine, TwoSiteItem
    rng = np.random.RandomState(97 * d + 31 * cl + 7 * cm + cr)

    def rand(*s):
        return (rng.randn(*s) + 1j * rng.randn(*s)).astype(np.complex64)

    a, b, g = rand(cl, d, cm), rand(cm, d, cr), rand(d * d, d * d)
    # an odd element offset: 8-byte aligned only
    buf = torch.zeros(a.size + 1, dtype=torch.complex64, device="cuda")
    buf[1:] = torch.from_numpy(a.reshape(-1)).cuda()
    k = d * min(cl, cr)
    r = Engine.get().two_site([TwoSiteItem(buf[1:].view(cl, d, cm), torch.from_numpy(b).cuda(),
                                           torch.from_numpy(g).cuda(), k, absorb_left=left)])[0]
    t = np.tensordot(a.astype(np.complex128), b.astype(np.complex128), axes=([2], [0]))
    theta = np.einsum("abpq,lpqr->labr", g.astype(np.complex128).reshape(d, d, d, d), t).reshape(cl * d, d * cr)
    x = r.a_out.cpu().numpy().astype(np.complex128).reshape(cl * d, k)
    y = r.b_out.cpu().numpy().astype(np.complex128).reshape(k, d * cr)
    err = np.linalg.norm(x @ y - theta) / np.linalg.norm(theta)
    assert err <= 1.01 * 2.0 ** -24 * (np.sqrt(k) + 1)
