"""CPU tests: blocksparse_forward takes its block list from the selector's select, wherever that is set."""
import types

import pytest
import qwen_blocksparse as qb

CLASSES = [qb.SelectMax, qb.SelectLastTok, qb.SelectMaxQMax, qb.SelectTwoStage]


@pytest.mark.parametrize("cls", CLASSES)
@pytest.mark.parametrize("where", ["class", "instance", "bound", "subclass"])
def test_a_replaced_select_is_called(cls, where, monkeypatch):
    want = object()
    monkeypatch.setattr(cls, "_select32", lambda self, q, k: pytest.fail("select was passed by"))
    sel = cls.__new__(cls)
    if where == "class":
        monkeypatch.setattr(cls, "select", lambda self, q, k: want)
    elif where == "instance":
        sel.select = lambda q, k: want
    elif where == "bound":
        sel.select = types.MethodType(lambda self, q, k: want, sel)
    else:
        sub = type("Sub", (cls,), {"select": lambda self, q, k: want})
        sel = sub.__new__(sub)
    assert qb._block_list(sel, None, None) is want


@pytest.mark.parametrize("cls", CLASSES)
def test_a_wrapped_select_reaches_the_original(cls, monkeypatch):
    seen = []
    first = cls.select
    monkeypatch.setattr(cls, "_select32", lambda self, q, k: types.SimpleNamespace(long=lambda: "int64 list"))
    monkeypatch.setattr(cls, "select", lambda self, q, k: seen.append(self) or first(self, q, k))
    sel = cls.__new__(cls)
    assert qb._block_list(sel, None, None) == "int64 list" and seen == [sel]


@pytest.mark.parametrize("cls", CLASSES)
def test_the_own_select_is_read_as_int32(cls, monkeypatch):
    want = object()
    monkeypatch.setattr(cls, "_select32", lambda self, q, k: want)
    assert qb._block_list(cls.__new__(cls), None, None) is want
