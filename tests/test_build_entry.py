"""__graft_entry__.build() ends only where both compiled modules load: the HIP library and the host module, which the hot
calls go through."""
import pytest

import __graft_entry__ as entry
import _native


def test_build_loads_both_modules(monkeypatch):
    monkeypatch.setattr(entry.subprocess, "run", lambda *a, **k: None)  # nothing is compiled here
    entry.build()
    monkeypatch.setattr(_native, "_host", None)
    monkeypatch.setattr(_native, "HOST_PATH", _native.HOST_PATH + ".missing")
    with pytest.raises(_native.NativeError, match="missing is not built"):
        entry.build()
