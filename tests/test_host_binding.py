"""CPU tests of the checks before a compiled binding is used."""
import sys
import types

import pytest


@pytest.mark.parametrize("calls", [("single_chunk",), ("single_chunk", "chunks", "rope", "seq_all_to_all")])
def test_a_node_without_every_entry_point_is_not_used(monkeypatch, calls):
    """A _ltr_node.so left from an earlier build has the same ABI version and fewer entry points: the Python side serves."""
    import lightron_amd
    from lightron_amd import _lib, attention
    old = types.ModuleType("lightron_amd._ltr_node")
    old.abi_version = lambda: _lib.LTR_ABI_VERSION
    for name in calls:
        setattr(old, name, lambda *a: None)
    monkeypatch.delenv("LTR_ATTN_LIB", raising=False)
    monkeypatch.setitem(sys.modules, "lightron_amd._ltr_node", old)
    monkeypatch.setattr(lightron_amd, "_ltr_node", old, raising=False)
    monkeypatch.setattr(attention, "_node", None)
    assert not attention._cpp_node()
    for name in attention._NODE_CALLS:
        setattr(old, name, lambda *a: None)
    monkeypatch.setattr(attention, "_node", None)
    assert attention._cpp_node() is old


def test_a_library_without_every_entry_point_is_named(monkeypatch):
    import ctypes
    from lightron_amd import _lib
    monkeypatch.setattr(_lib, "_lib", None)
    monkeypatch.setattr(_lib, "EXPORTS", _lib.EXPORTS + ("ltr_of_a_later_build",))
    with pytest.raises(RuntimeError, match="ltr_of_a_later_build"):
        _lib.load()
    assert ctypes.CDLL(_lib.LIB_PATH).ltr_abi_version() == _lib.LTR_ABI_VERSION
