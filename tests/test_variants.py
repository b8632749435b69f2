"""Kernel sets built on first need are planned and compiled once, loaded once per device, and unloaded with their last owner."""
import gc

from openequivariance_amd import runtime as rt


class Handle:
    def __init__(self, code, plan):
        self.code, self.plan = code, plan


def test_shared_while_held(monkeypatch):
    built, loaded = [], []
    monkeypatch.setattr(rt, "compile_source", lambda source: source.encode())

    def get(key, device=0, source="s"):
        return rt.variant(("test", key), device, lambda: (built.append(key) or source, ["plan"]),
                          lambda code, plan: loaded.append((key, device)) or Handle(code, plan))
    a, plan = get(1)
    assert a.code == b"s" and plan == ["plan"] and get(1)[0] is a and built == [1] and loaded == [(1, 0)]
    b, _ = get(1, device=1)
    assert b is not a and built == [1] and loaded == [(1, 0), (1, 1)]
    del a
    gc.collect()
    a, _ = get(1)                                     # unloaded with its last owner: loaded again, not built again
    assert built == [1] and loaded == [(1, 0), (1, 1), (1, 0)]
    assert get(2, source=None) == (None, ["plan"]) and get(2, source=None)[0] is None and built == [1, 2]
    held = [get(k)[0] for k in range(3, 3 + rt._VARIANTS_MAX)]
    assert len(rt._VARIANTS) == rt._VARIANTS_MAX and get(1)[0] is a and built.count(1) == 2 and len(held) == rt._VARIANTS_MAX
    for key in [k for k in rt._VARIANTS if k[0] == "test"]:
        del rt._VARIANTS[key]
