"""Two-site updates of one engine from several torch streams and threads, without
waits on the host: they share its workspaces, so each must see the results it has
when it runs alone (bitwise). Problems of every kind of kernel behind the call:
one workgroup (up to 64 rows), the direct solver, both orientations; sizes that
grow, so that a workspace is replaced while the other stream works on it.
"""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SIZES = (24, 200, 64, 300, 130, 48, 420, 90)


def _items(seed):
    import torch
    from mpsim_amd.engine import SplitItem
    rng = np.random.RandomState(seed)
    out = []
    for i, n in enumerate(SIZES):
        m = (rng.randn(n, n + 16) + 1j * rng.randn(n, n + 16)) / np.sqrt(n)
        out.append(SplitItem(torch.from_numpy(m.astype(np.complex64)).cuda(), n, absorb_left=bool(i % 2),
                             want_s=True))
    return out


def _same(x, y, tag):
    import torch
    for a, b in ((x.a_out, y.a_out), (x.b_out, y.b_out), (x.s, y.s)):
        assert torch.equal(a, b), tag


def _alone(items):
    import torch
    from mpsim_amd.engine import Engine
    eng, ref = Engine.get(), []
    for it in items:
        ref.append(eng.two_site([it])[0])
        torch.cuda.synchronize()
    return ref


def test_alternating_streams_share_an_engine():
    import torch
    from mpsim_amd.engine import Engine
    items = _items(1)
    ref = _alone(items)
    eng = Engine(Engine.get().dev)  # its workspace starts empty and grows
    streams = [torch.cuda.current_stream(), torch.cuda.Stream(), torch.cuda.Stream()]
    got = []
    for r in range(3):
        for i, it in enumerate(items):
            print("pass", r, "rows", SIZES[i], flush=True)
            with torch.cuda.stream(streams[(i + r) % 3]):
                got.append(eng.two_site([it])[0])
    torch.cuda.synchronize()
    for i, g in enumerate(got):
        _same(g, ref[i % len(items)], i)


def test_threads_share_an_engine():
    import torch
    from mpsim_amd.engine import Engine
    items = _items(2)
    ref = _alone(items)
    eng = Engine(Engine.get().dev)
    got, dev = {}, eng.dev

    def work(t):
        torch.cuda.set_device(dev)
        s = torch.cuda.Stream()
        with torch.cuda.stream(s):
            for i, it in enumerate(items):
                got[t, i] = eng.two_site([it])[0]
            s.synchronize()

    print("three threads", flush=True)
    ts = [threading.Thread(target=work, args=(t,)) for t in range(3)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    torch.cuda.synchronize()
    assert len(got) == 3 * len(items)
    for (t, i), g in got.items():
        _same(g, ref[i], (t, SIZES[i]))
