"""What is said when an SVD that the host does not poll (one workgroup up to 64 rows,
the direct solver up to 1024) does not converge: mpsx_two_site returns
MPSX_ENOTCONV, opts.unconverged counts the problems, and the engine, whose calls
return earlier, warns at the next call or host read.

The one-workgroup kernel is kept from converging by a tolerance below FP64 rounding
(rows orthogonal to 1e-17 of their norms), a group of the direct solver by a limit on
its waits that the host sets (MPSX_FORCE_TIMEOUT); every kernel ends normally.
"""
import ctypes
import dataclasses
import warnings

import numpy as np
import pytest

from test_gpu_routes import _forced, _same

pytestmark = pytest.mark.gpu

TOL = 1e-17


def _items(sizes, seed=4):
    import torch
    from mpsim_amd.engine import SplitItem
    rng = np.random.RandomState(seed)
    return [SplitItem(torch.from_numpy((rng.randn(n, n + 5) + 1j * rng.randn(n, n + 5)).astype(np.complex64)).cuda(),
                      n, want_s=True) for n in sizes]


def _quiet(f, *a):
    with warnings.catch_warnings():
        warnings.simplefilter("error")
        return f(*a)


def test_engine_warns_after_the_call():
    import torch
    from mpsim_amd._native import NotConvergedWarning
    from mpsim_amd.engine import Engine
    eng, items = Engine.get(), _items((32,))
    hard = dataclasses.replace(eng.svd, tol=TOL)
    torch.cuda.synchronize()
    _quiet(eng.report)
    print("report()", flush=True)
    eng.two_site(items, hard)
    torch.cuda.synchronize()
    with pytest.warns(NotConvergedWarning):
        eng.report()
    print("the next call", flush=True)
    eng.two_site(items, hard)
    torch.cuda.synchronize()
    with pytest.warns(NotConvergedWarning):
        res = eng.two_site(items)
    print("a host read", flush=True)
    eng.two_site(items, hard)
    with pytest.warns(NotConvergedWarning):
        eng.host(res[0].s)
    _quiet(eng.two_site, items)
    _quiet(eng.host, res[0].s)


def test_mps_readout_warns():
    from mpsim_amd import MPS
    from mpsim_amd._native import NotConvergedWarning
    from mpsim_amd.engine import Engine
    from mpsim_amd.gates import haar_unitary
    eng, old = Engine.get(), Engine.get().svd
    rng = np.random.RandomState(6)

    def circuit():
        mps = MPS(12)
        for layer in range(8):
            for i in range(layer % 2, 11, 2):
                mps.apply_two_qudit_gate(haar_unitary(4, rng).reshape(2, 2, 2, 2), i, i + 1)
        return mps

    _quiet(lambda: circuit().wavefunction())
    eng.svd = dataclasses.replace(old, tol=TOL)
    try:
        with pytest.warns(NotConvergedWarning):
            circuit().wavefunction()
    finally:
        eng.svd = old


@pytest.mark.parametrize("entry", ["mpsx_two_site", "mpsx_two_site_static"])
def test_small_problems_are_counted_and_returned(entry):
    import torch
    from mpsim_amd import _native as nat
    from mpsim_amd.engine import Engine
    eng = Engine.get()
    items = _items((32, 1, 48))  # one row has nothing to rotate
    for tol, bad in ((TOL, 2), (0.0, 0)):
        n = torch.zeros(1, dtype=torch.int32, device="cuda")
        c = dataclasses.replace(eng.svd, tol=tol, unconverged=n.data_ptr()).to_c()
        outs, tab, dtab, ws = eng._prepare_two_site(items, c)
        sweeps = ctypes.c_int(0)
        print(entry, "tol", tol, flush=True)
        args = [eng.stream, tab.ctypes.data, dtab.data_ptr(), len(tab), ctypes.byref(c)]
        if entry == "mpsx_two_site":
            args += [ws.data_ptr(), ws.numel()]
        rc = getattr(eng.lib, entry)(*args, ctypes.byref(sweeps))
        assert int(n.item()) == bad
        if entry == "mpsx_two_site":
            assert rc == (nat.MPSX_ENOTCONV if bad else nat.MPSX_OK)
        else:  # never reads device memory back
            assert rc == nat.MPSX_OK


@pytest.mark.parametrize("n", [200, 400, 1024])
def test_expired_wait_is_returned(n):
    """The problem whose group gave up a wait is counted and returned; the others of
    the call (one workgroup each) have their bits."""
    import torch
    from mpsim_amd import _native as nat
    from mpsim_amd.engine import Engine
    eng = Engine.get()
    items = _items((100, n, 40))
    ref, rc0 = _forced(items, eng.svd, 0)
    count = torch.zeros(1, dtype=torch.int32, device="cuda")
    print("rows", n, flush=True)
    res, rc = _forced(items, dataclasses.replace(eng.svd, unconverged=count.data_ptr()), nat.FORCE_TIMEOUT)
    assert rc0 == nat.MPSX_OK and rc == nat.MPSX_ENOTCONV and int(count.item()) == 1
    for i in (0, 2):
        _same(ref[i], res[i], i)


@pytest.mark.parametrize("graph", [False, True])
def test_program_warns(graph):
    from mpsim_amd._native import NotConvergedWarning
    from mpsim_amd.circuits import brickwork_haar
    from mpsim_amd.engine import Engine
    from mpsim_amd.program import CircuitProgram
    circ = brickwork_haar(10, 6, 2, maxsvals=16, seed=3)
    prog = CircuitProgram([circ], svd=dataclasses.replace(Engine.get().svd, tol=TOL), graph=graph)
    for r in range(2):
        print("run", r, flush=True)
        with pytest.warns(NotConvergedWarning):
            prog.run()
        assert prog.last_unconverged > 0
    good = CircuitProgram([circ], graph=graph)
    for r in range(2):
        _quiet(good.run)
        assert good.last_unconverged == 0
