"""mpsx_two_site_forced checks its calls as mpsx_two_site does, and its own bits."""
import ctypes

import pytest

from test_abi_host import _plan, _table


@pytest.mark.parametrize("force,ok", [(0, True), (1, True), (2, True), (1 << 20, False), (-1, False)])
def test_forced_call_checks_its_bits_and_table(force, ok):
    from mpsim_amd import _native as nat
    lib = nat.load()
    tab = _table([(64, 64, 64, 2, 64, 0)])
    rc, _, err = _plan(tab)
    assert rc == 0, err
    o = nat.SvdOpts(0, 0, 1, 0, 0.0)
    sweeps = ctypes.c_int(0)
    rc = lib.mpsx_two_site_forced(None, tab.ctypes.data, tab.ctypes.data, 1, ctypes.byref(o), ctypes.c_void_p(0x1000),
                                  1024, ctypes.byref(sweeps), force)
    # a table that passes every check stops at the workspace's size, before any launch
    assert rc == (nat.MPSX_EWORKSPACE if ok else nat.MPSX_EINVAL), lib.mpsx_last_error().decode()
