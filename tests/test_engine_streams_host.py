"""The order of calls that share an engine's workspaces (mpsim_amd.engine), with
recording streams and events in place of the device's: a call on another stream
than the last one's waits for that one's end, a replaced workspace stays with the
stream that worked on it, and one thread enqueues at a time."""
import threading
import types
import warnings

import pytest


class _Stream:
    def __init__(self, handle, log):
        self.cuda_stream, self.log = handle, log

    def wait_event(self, ev):
        self.log.append(("wait", self.cuda_stream, ev.at))


class _Buffer:
    def __init__(self, n, log):
        self.n, self.log = n, log

    def numel(self):
        return self.n

    def data_ptr(self):
        return 0

    def record_stream(self, s):
        self.log.append(("kept by", s.cuda_stream, self.n))


def _engine(log, need):
    """An engine without a device: the library call logs its stream."""
    from mpsim_amd.engine import Engine, SvdConfig

    class _Event:
        at = None

        def record(self, s):
            self.at = (s.cuda_stream, sum(1 for e in log if e[0] == "run"))
            log.append(("record", s.cuda_stream))

    eng = Engine.__new__(Engine)
    cuda = types.SimpleNamespace(current_stream=lambda dev: eng.now, Event=_Event)
    eng.torch = types.SimpleNamespace(cuda=cuda, uint8=None,
                                      empty=lambda n, dtype, device: _Buffer(n, log))
    eng.dev, eng.svd = None, SvdConfig()
    eng._ws, eng._wss, eng._keep, eng._helpers = None, [], [], []
    eng.split_ways, eng.split_min, eng.split_rows = 1, 1, 1
    eng._split_stored = eng._split_rounds = (1, 1)
    eng._cus = 256
    eng._enqueue, eng._used, eng._used_end = threading.RLock(), None, None
    eng._used_handle, eng._late = -1, types.SimpleNamespace(value=0)

    def prepare(items, cfg, slot=0, workspace=True, stream=None):
        return list(items), [0], None, eng.workspace(need[0], slot)

    def run(tab, dtab, ws, cfg, stream):
        log.append(("run", stream))
        return 0

    eng._prepare_two_site, eng._run_two_site = prepare, run
    return eng


def _item():
    import numpy as np
    from mpsim_amd.engine import SplitItem
    return SplitItem(np.zeros((2, 2)), 2)


@pytest.mark.parametrize("first,second", [(0, 7), (7, 0), (7, 9)])
def test_call_on_another_stream_waits_for_the_last(first, second):
    log = []
    eng = _engine(log, [2048])
    s = {h: _Stream(h, log) for h in (first, second)}
    for h in (first, first, second, first):
        eng.now = s[h]
        eng.two_site([_item()])
    ops = [e for e in log if e[0] != "record"]
    # each wait is for an event behind all the work of the stream before it
    assert ops == [("run", first), ("run", first), ("wait", second, (first, 2)), ("run", second),
                   ("wait", first, (second, 3)), ("run", first)]


def test_late_report_warns_once():
    from mpsim_amd._native import NotConvergedWarning
    eng = _engine([], [2048])
    eng.now = _Stream(0, [])
    eng._late.value = 1  # a kernel of an earlier call
    with pytest.warns(NotConvergedWarning):
        eng.two_site([_item()])
    with warnings.catch_warnings():
        warnings.simplefilter("error")
        eng.two_site([_item()])
        eng.report()


def test_one_default_stream_records_nothing():
    log = []
    eng = _engine(log, [2048])
    eng.now = _Stream(0, log)
    for _ in range(3):
        eng.two_site([_item()])
    assert log == [("run", 0)] * 3


def test_replaced_workspace_stays_with_its_stream():
    log, need = [], [2048]
    eng = _engine(log, need)
    eng.now = _Stream(7, log)
    eng.two_site([_item()])
    need[0] = 4096
    eng.now = _Stream(9, log)
    eng.two_site([_item()])
    assert [e for e in log if e[0] in ("wait", "kept by")] == [("wait", 9, (7, 1)), ("kept by", 9, 2048)]


def test_threads_enqueue_one_at_a_time():
    log, inside, most = [], [0], [0]
    eng = _engine(log, [2048])
    eng.now = _Stream(0, log)
    gate = threading.Event()

    def run(tab, dtab, ws, cfg, stream):
        inside[0] += 1
        most[0] = max(most[0], inside[0])
        gate.wait(0.05)
        inside[0] -= 1
        return 0

    eng._run_two_site = run
    ts = [threading.Thread(target=eng.two_site, args=([_item()],)) for _ in range(4)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert most[0] == 1
