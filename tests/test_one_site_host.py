"""Engine.one_site_rows with a recording library: a gate whose descriptors go with the
launch is not applied a second time from a table when the launch reports an error (a
gate in place would act twice); only a refusal, before any launch, takes the table."""
import types

import pytest


@pytest.mark.parametrize("code,calls", [(0, ["now"]), (1, ["now", "put", "table"]), (2, ["now"])])
def test_one_site_launch_and_table(monkeypatch, code, calls):
    from mpsim_amd import _native as nat
    from mpsim_amd.engine import Engine
    log = []
    lib = types.SimpleNamespace(
        mpsx_apply_one_site_now=lambda s, h, n: log.append("now") or code,
        mpsx_apply_one_site=lambda s, h, d, n: log.append("table") or 0)
    monkeypatch.setattr(nat, "put_table", lambda t, dev, s: log.append("put") or types.SimpleNamespace(
        data_ptr=lambda: 0))
    monkeypatch.setattr(Engine, "stream", property(lambda self: 0))
    eng = Engine.__new__(Engine)
    eng.lib, eng.dev = lib, None
    rows = [(0x1000, 0x1000, 0x2000, 4, 4, 2, 0)]
    if code == nat.MPSX_EHIP:
        with pytest.raises(nat.MpsxError):
            eng.one_site_rows(rows)
    else:
        eng.one_site_rows(rows)
    assert log == calls
