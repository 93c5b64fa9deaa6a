"""Groups of workgroups of the direct solver are not given up because launches (or the
last groups of one launch) block each other: calls that fill the device several times
over, in one launch, split over four streams, and from four engines at once. The
control blocks of all problems say afterwards that no group was given up, and the
results are those of the problem alone (bitwise).
"""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _engine(ways):
    """An engine that keeps (table, workspace) of each library call."""
    from mpsim_amd.engine import Engine
    eng = Engine(Engine.get().dev)
    eng.split_ways, eng.split_min, eng.split_rows = ways, 1, 512
    seen, run = [], eng._run_two_site

    def keep(tab, dtab, ws, cfg, stream):
        out = run(tab, dtab, ws, cfg, stream)
        seen.append((tab, ws))
        return out

    eng._run_two_site = keep
    return eng, seen


def _given_up(seen):
    import torch
    n = 0
    for tab, ws in seen:
        at = torch.from_numpy(tab["ws_off"].astype(np.int64) // 4 + 7).cuda()  # ProblemCtl.group
        n += int((ws[:ws.numel() // 4 * 4].view(torch.int32)[at] >= 1 << 30).sum())
    return n


def _items(rows, count, seed):
    import torch
    from mpsim_amd.engine import SplitItem
    g = torch.Generator(device="cuda").manual_seed(seed)
    return [SplitItem(torch.randn(rows, rows, dtype=torch.complex64, device="cuda", generator=g), rows // 2,
                      want_s=True) for _ in range(count)]


@pytest.mark.parametrize("rows,count,ways", [(900, 11, 1), (400, 31, 1), (1024, 27, 4), (600, 16, 4)])
def test_one_call_gives_up_no_group(rows, count, ways):
    import torch
    eng, seen = _engine(ways)
    items = _items(rows, count, rows)
    alone = eng.two_site(items[:1])[0]
    torch.cuda.synchronize()
    for r in range(12):
        print(rows, "rows", count, "problems", ways, "ways, pass", r, flush=True)
        seen.clear()
        res = eng.two_site(items)
        torch.cuda.synchronize()
        assert _given_up(seen) == 0
        assert torch.equal(res[0].s, alone.s) and torch.equal(res[0].a_out, alone.a_out)


def test_four_engines_give_up_no_group():
    import torch
    lanes = [(_engine(1), _items(1024, 6, i)) for i in range(4)]
    torch.cuda.synchronize()
    out, dev = {}, lanes[0][0][0].dev

    def work(i):
        torch.cuda.set_device(dev)
        (eng, seen), items = lanes[i]
        s = torch.cuda.Stream()
        with torch.cuda.stream(s):
            for r in range(3):
                seen.clear()
                res = eng.two_site(items)
                s.synchronize()
                out[i, r] = (_given_up(seen), res[0].s.clone())
            s.synchronize()

    print("four engines", flush=True)
    ts = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    torch.cuda.synchronize()
    assert len(out) == 12 and all(n == 0 for n, _ in out.values())
    for i in range(4):
        assert all(torch.equal(out[i, 0][1], out[i, r][1]) for r in (1, 2))
