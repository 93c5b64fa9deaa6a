"""Routes of the two-site update that a whole MI355X seldom takes
(mpsx_two_site_forced): the Jacobi rounds of the Gram method, alone and behind the
Householder QR, for the sizes the direct solver otherwise takes; and the
one-workgroup tridiagonalisation of problems whose group was given up. Then
inputs that are not finite.

Bounds: the rounds meet the direct solver's where both are backward stable in
FP64 (singular values within 2e-6 relative + 1e-7 ||theta||_F, as between the
methods elsewhere), and numpy's as test_gpu_qr._check states them. The given-up
groups have the same bits (every sum is formed in the same order).
"""
import ctypes

import numpy as np
import pytest

from test_gpu_eig import _matrix
from test_gpu_qr import SHAPES, _check, _theta

pytestmark = pytest.mark.gpu


def _forced(items, cfg, force):
    """(results, return code) of one call through mpsx_two_site_forced, waited for.
    With FORCE_LOST every problem's control block says so afterwards."""
    import torch
    from mpsim_amd import _native as nat
    from mpsim_amd.engine import Engine
    eng = Engine.get()
    c = cfg.to_c()
    outs, tab, dtab, ws = eng._prepare_two_site(items, c)
    sweeps = ctypes.c_int(0)
    rc = nat.load().mpsx_two_site_forced(eng.stream, tab.ctypes.data, dtab.data_ptr(), len(tab), ctypes.byref(c),
                                         ws.data_ptr(), ws.numel(), ctypes.byref(sweeps), force)
    torch.cuda.synchronize()
    if force == nat.FORCE_LOST:
        at = torch.from_numpy(tab["ws_off"].astype(np.int64) // 4 + 7).cuda()  # ProblemCtl.group
        assert bool((ws[:ws.numel() // 4 * 4].view(torch.int32)[at] >= 1 << 30).all())
    return outs, rc


def _same(x, y, tag):
    import torch
    for a, b in ((x.a_out, y.a_out), (x.b_out, y.b_out), (x.s, y.s)):
        assert torch.equal(a, b), tag


@pytest.mark.parametrize("pre", [0, 2])
def test_jacobi_rounds_vs_lapack_and_the_direct_solver(pre):
    """The shapes of the preconditioned method's tests, through the kernels their
    names state: rounds from H = X X^H (0) or from the QR's R (2)."""
    import torch
    from mpsim_amd import _native as nat
    from mpsim_amd import gates
    from mpsim_amd.engine import Engine, SvdConfig, TwoSiteItem
    eng = Engine.get()
    rng = np.random.RandomState(78)
    cases, items = [], []
    for (cl, cm, cr, d, k, left) in SHAPES:
        A = ((rng.randn(cl, d, cm) + 1j * rng.randn(cl, d, cm)) / np.sqrt(2 * d * cm)).astype(np.complex64)
        B = ((rng.randn(cm, d, cr) + 1j * rng.randn(cm, d, cr)) / np.sqrt(2)).astype(np.complex64)
        G = gates.haar_unitary(d * d, rng)
        cases.append((cl, cm, cr, d, k, left, A, B, G))
        items.append(TwoSiteItem(torch.from_numpy(A).cuda(), torch.from_numpy(B).cuda(), eng.gate(G), k,
                                 absorb_left=left, want_s=True))
    cfg = SvdConfig(block_switch=eng.svd.block_switch, inner_sweeps=eng.svd.inner_sweeps, precondition=pre)
    direct = eng.two_site(items, cfg)
    torch.cuda.synchronize()
    nat.profile_read(reset=True)
    nat.profile_enable(True)
    print("rounds, precondition", pre, flush=True)
    res, rc = _forced(items, cfg, nat.FORCE_ROUNDS)
    nat.profile_enable(False)
    ran = nat.profile_read(reset=True)
    assert rc == nat.MPSX_OK and "k_hround" in ran and "k_tridiag" not in ran
    assert ("k_qr_step" in ran) == (pre == 2)
    for (cl, cm, cr, d, k, left, A, B, G), r, r0 in zip(cases, res, direct):
        tag = (cl, cm, cr, d, k, left)
        print("case", tag, flush=True)
        theta = _theta(d, A, B, G)
        s = _check(theta, k, left, r, tag)
        s0 = r0.s.cpu().numpy().astype(np.float64)
        assert np.all(np.abs(s - s0) <= 2e-6 * s0 + 1e-7 * np.linalg.norm(theta)), tag


@pytest.mark.parametrize("M,N", [(96, 96), (97, 130), (150, 90), (513, 513), (600, 200), (1024, 100)])
def test_jacobi_rounds_of_tall_and_padded_problems(M, N):
    """Six blocks, odd blocks and padded rows, and tall problems whose rounds run on
    the R of the QR only (precondition 2)."""
    import torch
    from mpsim_amd import _native as nat
    from mpsim_amd.engine import Engine, SplitItem, SvdConfig
    eng = Engine.get()
    rng = np.random.RandomState(M + N)
    mats = [_matrix(M, N, kind, rng).astype(np.complex64) for kind in ("random", "rank 3")]
    items = [SplitItem(torch.from_numpy(A).cuda(), min(A.shape), want_s=True) for A in mats]
    for pre in (0, 2):
        cfg = SvdConfig(block_switch=eng.svd.block_switch, inner_sweeps=eng.svd.inner_sweeps, precondition=pre)
        print("rounds", M, N, "precondition", pre, flush=True)
        res, rc = _forced(items, cfg, nat.FORCE_ROUNDS)
        assert rc == nat.MPSX_OK
        for A, r in zip(mats, res):
            _check(A.astype(np.complex128), min(A.shape), False, r, (M, N, pre))


@pytest.mark.parametrize("n", [129, 200, 256, 257, 512, 513, 1000, 1024])
def test_given_up_groups_have_the_same_bits(n):
    """Sizes where a group's class and last member change, beside a problem of one
    workgroup (which has no group to give up); a rank-deficient matrix, on which
    the iteration stops early, and a tall one."""
    import torch
    from mpsim_amd import _native as nat
    from mpsim_amd.engine import Engine, SplitItem
    eng = Engine.get()
    rng = np.random.RandomState(n)
    mats = [_matrix(n, n, "random", rng), _matrix(n, n, "rank 3", rng), _matrix(n, n // 2, "random", rng),
            _matrix(100, 100, "random", rng)]
    items = [SplitItem(torch.from_numpy(A.astype(np.complex64)).cuda(), min(A.shape), want_s=True) for A in mats]
    ref, rc0 = _forced(items, eng.svd, 0)
    print("given up", n, flush=True)
    res, rc = _forced(items, eng.svd, nat.FORCE_LOST)
    assert rc0 == rc == nat.MPSX_OK
    for i, (x, y) in enumerate(zip(ref, res)):
        _same(x, y, (n, i))


@pytest.mark.parametrize("bad", [np.nan, np.inf, -np.inf])
def test_not_finite_inputs_stay_with_their_problem(bad):
    """A matrix with one entry that is not finite, in every kind of kernel, ends and
    leaves the other problems of its call as they are without it (bitwise)."""
    import torch
    from mpsim_amd import _native as nat
    from mpsim_amd.engine import Engine, SplitItem
    eng = Engine.get()
    rng = np.random.RandomState(9)
    sizes = (5, 40, 64, 100, 200, 300, 600)
    mats = [(rng.randn(n, n + 3) + 1j * rng.randn(n, n + 3)).astype(np.complex64) for n in sizes]
    good = [SplitItem(torch.from_numpy(A).cuda(), A.shape[0], want_s=True) for A in mats]
    mixed = []
    for A, it in zip(mats, good):
        B = A.copy()
        B[A.shape[0] // 2, 1] = bad
        mixed += [it, SplitItem(torch.from_numpy(B).cuda(), A.shape[0], want_s=True)]
    ref, rc0 = _forced(good, eng.svd, 0)
    print("not finite:", bad, flush=True)
    res, rc = _forced(mixed, eng.svd, 0)
    assert rc0 == rc == nat.MPSX_OK
    for i, (x, y) in enumerate(zip(ref, res[::2])):
        _same(x, y, sizes[i])
    for i, r in enumerate(res[1::2]):
        # the values of a matrix that is not finite are not either
        assert not bool(torch.isfinite(r.s).all()), sizes[i]


def test_launches_wait_for_their_groups_for_different_times():
    """Four calls one after the other, each in its own workspace, have four different
    limits (TwoSiteHeader.spread) wherever their workspaces lie."""
    import torch
    from mpsim_amd import _native as nat
    from mpsim_amd.engine import Engine, SplitItem
    eng = Engine.get()
    m = torch.randn(200, 200, dtype=torch.complex64, device="cuda")
    c = eng.svd.to_c()
    seen = set()
    for _ in range(4):
        outs, tab, dtab, ws = eng._prepare_two_site([SplitItem(m, 200)], c)
        ws = torch.empty(32 << 20, dtype=torch.uint8, device="cuda")
        nat.check(eng.lib.mpsx_two_site(eng.stream, tab.ctypes.data, dtab.data_ptr(), 1, ctypes.byref(c), ws.data_ptr(),
                                        ws.numel(), None))
        seen.add(int(ws[:512].view(torch.int32)[65].item()))
    assert seen == {0, 1, 2, 3}
