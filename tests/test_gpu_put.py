"""mpsx_put (descriptor tables in launch arguments) and GemmChain (many dependent
products behind one table)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nbytes", [4, 96, 3836, 3840, 3844, 7680, 16384])
def test_put_copies_the_bytes_and_nothing_else(nbytes):
    import torch
    from mpsim_amd import _native as nat
    rng = np.random.RandomState(nbytes)
    src = rng.randint(0, 256, nbytes).astype(np.uint8)
    dst = torch.full((nbytes + 8,), 7, dtype=torch.uint8, device="cuda")
    stream = nat.stream_handle(dst.device)
    nat.check(nat.load().mpsx_put(stream, dst.data_ptr(), src.ctypes.data, nbytes))
    want = src.copy()
    src[:] = 0  # the bytes left with the launch
    got = dst.cpu().numpy()
    assert np.array_equal(got[:nbytes], want) and (got[nbytes:] == 7).all()


def test_put_refuses():
    import torch
    from mpsim_amd import _native as nat
    lib, src = nat.load(), np.zeros(16388, dtype=np.uint8)
    dst = torch.zeros(16388, dtype=torch.uint8, device="cuda")
    s = torch.cuda.Stream()
    h, d, p = int(s.cuda_stream), dst.data_ptr(), src.ctypes.data
    for args in ((h, d, p, 16388), (h, d, p, 6), (h, d + 2, p, 4), (h, None, p, 4), (h, d, None, 4)):
        assert lib.mpsx_put(*args) == nat.MPSX_EINVAL
    import ctypes
    g = ctypes.c_void_p(0)
    nat.check(lib.mpsx_graph_begin(h))
    code = lib.mpsx_put(h, d, p, 16)
    nat.check(lib.mpsx_graph_end(h, ctypes.byref(g)))
    nat.check(lib.mpsx_graph_destroy(g))
    assert code == nat.MPSX_EINVAL


@pytest.mark.parametrize("links,size", [(1, 3), (39, 8), (41, 33), (120, 5)])
def test_chain_of_products(links, size):
    """psi <- psi U_i over orthogonal U_i (shorter and longer than a table):
    norms stay, so each link adds at most size * eps of the FP32 products."""
    import torch
    from mpsim_amd.engine import Engine, GemmChain
    eng = Engine.get()
    rng = np.random.RandomState(links)
    us = [np.linalg.qr(rng.randn(size, size) + 1j * rng.randn(size, size))[0].astype(np.complex64)
          for _ in range(links)]
    x = np.eye(size, dtype=np.complex64)
    want = x.astype(np.complex128)
    cur = torch.from_numpy(x).cuda()
    chain = GemmChain(eng)
    for u in us:
        want = want @ u.astype(np.complex128)
        out = torch.empty_like(cur)
        chain.gemm([dict(A=cur, B=torch.from_numpy(u).cuda(), C=out, m=size, n=size, k=size,
                         lda=size, ldb=size, ldc=size)])
        cur = out
    chain.flush()
    err = np.linalg.norm(cur.cpu().numpy() - want)
    assert err <= links * size * 2.0 ** -23 * np.sqrt(size)


@pytest.mark.parametrize("count", [1, 15, 16, 17])
@pytest.mark.parametrize("d", [1, 2, 3, 4, 5])
def test_one_site_gates_with_and_without_a_device_table(count, d):
    """The same bits from mpsx_apply_one_site_now (up to 16 gates) and from a device table."""
    import torch
    from mpsim_amd import _native as nat
    from mpsim_amd.engine import Engine
    eng = Engine.get()
    gen = torch.Generator(device="cuda")
    gen.manual_seed(count + 100 * d)
    lib, stream = nat.load(), eng.stream
    g = torch.randn(d, d, dtype=torch.complex64, device="cuda", generator=gen)
    ts = [torch.randn(3 + i, d, 5, dtype=torch.complex64, device="cuda", generator=gen) for i in range(count)]
    one = [torch.empty_like(t) for t in ts]
    two = [torch.empty_like(t) for t in ts]
    eng.one_site([(t, o, g) for t, o in zip(ts, one)])
    tab = np.array([(nat.ptr(t), nat.ptr(o), nat.ptr(g), t.shape[0], t.shape[2], d, 0) for t, o in zip(ts, two)],
                   dtype=nat.SITE_OP)
    dtab = nat.to_device_table(tab, eng.dev)
    nat.check(lib.mpsx_apply_one_site(stream, tab.ctypes.data, dtab.data_ptr(), count))
    assert all(torch.equal(torch.view_as_real(x), torch.view_as_real(y)) for x, y in zip(one, two))
    code = lib.mpsx_apply_one_site_now(stream, tab.ctypes.data, count)
    assert (code == nat.MPSX_OK) == (count <= nat.SITE_NOW)
