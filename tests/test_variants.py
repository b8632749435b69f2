"""Kernel sets beside an operator's main one are planned and compiled once, loaded once per device and unloaded with their
last owner; an operator has them when it is constructed."""
import gc

import numpy as np
import pytest
import torch

import common
import openequivariance_amd as oeq
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


def test_no_thread_waits_for_another_problems_compilation(monkeypatch):
    import threading
    entered, release, got = threading.Event(), threading.Event(), []

    def compile_source(source):
        if source == "slow":
            entered.set()
            assert release.wait(30)
        return source.encode()
    monkeypatch.setattr(rt, "compile_source", compile_source)
    monkeypatch.setattr(rt, "_VARIANTS", type(rt._VARIANTS)())
    get = lambda source: got.append(rt.variant((source,), 0, lambda: (source, None), Handle)[0])
    slow = threading.Thread(target=get, args=("slow",))
    slow.start()
    assert entered.wait(30)
    quick = threading.Thread(target=get, args=("quick",))
    quick.start()
    quick.join(10)
    waited = quick.is_alive()
    release.set()
    slow.join(30)
    quick.join(30)
    assert not waited and [h.code for h in got] == [b"quick", b"slow"]


class Impl:
    def __init__(self, code, *steps):
        self.code = code

    def set_forward_workspace(self, *model):
        pass


@pytest.mark.parametrize("case", ["uvu", "uvu_raw", "uvw", "conv", "conv_sorted"])
def test_no_call_waits_for_the_compiler(case, monkeypatch):
    """The kernel sets of second derivatives and of batches of few rows are compiled and loaded with the operator."""
    monkeypatch.setattr(torch.cuda, "current_device", lambda: 0)
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
    monkeypatch.setattr(rt, "compile_source", lambda source, *a, **k: source.encode())
    monkeypatch.setattr(rt, "TPImpl", Impl)
    monkeypatch.setattr(rt, "ConvImpl", Impl)
    monkeypatch.setattr(rt, "_VARIANTS", type(rt._VARIANTS)())
    monkeypatch.setattr(rt, "_LOADED", type(rt._LOADED)())
    if case == "uvw":
        op = oeq.TensorProduct(common.fully_connected(common.DENSE, shared=True)[0], torch_op=False)
    elif case.startswith("uvu"):
        op = oeq.TensorProduct(common.channelwise(common.NEQUIP)[0], torch_op=case == "uvu")
    else:
        op = oeq.TensorProductConv(common.channelwise(common.NEQUIP)[0], torch_op=True, deterministic=case == "conv_sorted")
    kinds = [key[0] for key in rt._VARIANTS]
    assert kinds == {"uvu": ["tp double"], "uvu_raw": [], "uvw": ["uvw few rows"]}.get(case, ["conv double"])

    def refuse(*a):
        raise AssertionError("compiled inside a call")
    monkeypatch.setattr(rt, "compile_source", refuse)
    if case == "uvw":
        limits = op._few_rows_limits
        # (64 channels: no forward is theirs, and none is built with them)
        assert limits == (0, 2048) and b"void forward(" not in op._few_rows.code
        assert [op._pick_rows(n, back) is not None for back in (False, True) for n in (0, 1, limits[back], limits[back] + 1)] \
            == [False] * 5 + [True, True, False]
    elif case == "uvu":
        assert op._double[True].code
    elif case.startswith("conv"):
        before = op._ws_bytes(5000, 300)
        assert op._double_usable() and op._double_impl().code and op._double_impl() is op._double
        assert op._double_ws_bytes(5000, 300) > 0 and op._ws_bytes(5000, 300) == before


def test_workspace_sizes_asked_for_by_several_threads(monkeypatch):
    """Another thread's question in the middle of one does not change its answer."""
    class Conv(oeq.TensorProductConv):
        """Every read of the last answer comes after another thread has asked for a small graph."""
        def __init__(self):
            self._ws_fns, self._double_built = [lambda nnz, nodes: 8 * nnz], (None, lambda nnz, nodes: 16 * nnz)

        def _double_impl(self):
            pass
    for name, factor in (("_ws_last", 8), ("_double_ws_last", 16)):
        def get(self, name=name, factor=factor):
            return ((1, 1) if name == "_double_ws_last" else (1, 1, 1)), factor
        setattr(Conv, name, property(get, lambda self, v: None))
    conv = Conv()
    for nnz in (1000, 1000, 7):
        assert conv._ws_bytes(nnz, 5) == 8 * nnz
        assert conv._double_ws_bytes(nnz, 5) == 16 * nnz


@pytest.mark.parametrize("deterministic", [False, True])
def test_layers_of_one_problem_write_their_convolution_once(deterministic, monkeypatch):
    """The kernels of a second operator, and the backward variant that its first pass builds, are there already; an operator
    with other choices gets its own."""
    from openequivariance_amd import conv as conv_mod, tunables
    from openequivariance_amd.codegen.uvu_det import UVUDetGenerator
    from openequivariance_amd.codegen.uvu_sorted import UVUSortedGenerator
    monkeypatch.setattr(torch.cuda, "current_device", lambda: 0)
    monkeypatch.setattr(rt, "compile_source", lambda source, *a, **k: source.encode())
    monkeypatch.setattr(rt, "ConvImpl", Impl)
    monkeypatch.setattr(rt, "_VARIANTS", type(rt._VARIANTS)())
    monkeypatch.setattr(rt, "_LOADED", type(rt._LOADED)())
    monkeypatch.setattr(conv_mod, "_GENERATED", type(conv_mod._GENERATED)())
    written = []
    for cls in (UVUDetGenerator, UVUSortedGenerator):
        monkeypatch.setattr(cls, "render", lambda self, *a, f=cls.render, **k: written.append(type(self)) or f(self, *a, **k))

    def layer(**kwargs):
        op = oeq.TensorProductConv(common.channelwise(common.NEQUIP)[0], deterministic=deterministic, **kwargs)
        sets = [op._pick(8)] if deterministic else [op._backward_variant(v)[0] for v in ("atomic", "grouped")] + [op._pick(8)]
        return op, sets
    (first, a), n = layer(), len(written)
    (second, b) = layer()
    assert n == len(written) == (2 if deterministic else 3)
    assert first.jit_kernel == second.jit_kernel == first.internal.code.decode() and first.internal is not second.internal
    assert sum(x is y for x, y in zip(a, b)) == len(a) - (not deterministic)        # (all but the operator's own set)
    assert first._ws_bytes(5000, 300) == second._ws_bytes(5000, 300)
    with monkeypatch.context() as m:
        m.setattr(tunables.current, "long_node", 0)
        assert layer()[0].jit_kernel != first.jit_kernel
    with monkeypatch.context() as m:
        m.setattr(UVUDetGenerator, "TEAMS", ())
        assert "forward_few" not in layer()[0].jit_kernel and "forward_few" in first.jit_kernel
    assert layer(idx_dtype=np.int32)[0].jit_kernel != first.jit_kernel
    assert layer()[0].jit_kernel == first.jit_kernel
