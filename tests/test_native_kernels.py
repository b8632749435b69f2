"""The operators' C++ GPU kernels (csrc/oeq_torch.cpp) against their general implementations in Python: every form of call that
either takes, the errors, and the workspace sizes, which both sides work out."""
import numpy as np
import pytest
import torch

import common
import openequivariance_amd as oeq
from openequivariance_amd import autograd_glue
from openequivariance_amd.codegen.uvu_conv_double import conv_double_generator
from openequivariance_amd.codegen.uvu_det import UVUDetGenerator
from openequivariance_amd.codegen.uvu_recv import UVURecvGenerator
from openequivariance_amd.codegen.uvu_sorted import UVUSortedGenerator
from oracle import tp as otp


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_workspace_bytes_are_the_same_on_both_sides(dtype):
    gens = []
    for irreps in (common.NEQUIP, common.MACE, ("5x0e+3x1o+70x2e", "1x0e+1x1o+1x2e", "5x0e+3x1o+70x2e+7x3o")):
        prob = common.channelwise(irreps, dtype=dtype)[0]
        gens += [UVUDetGenerator(prob), UVUDetGenerator(prob, long_node=0), UVURecvGenerator(prob), conv_double_generator(prob, True),
                 conv_double_generator(prob, False), UVUSortedGenerator(prob, grouped_backward=False),
                 *(UVUSortedGenerator(prob, grouped_backward=True, recv_backward=r) for r in (False, True))]
    autograd_glue._operators()
    ops = torch.ops.openequivariance_amd
    for g in gens:
        ws = g.plan()[2]
        id = ops.native_operator([0] * 16, list(g.workspace_terms()), [])
        for nodes in (1, 7, 64, 1000, 54321):
            for nnz in (1, 31, 32, 256, 257, 3 * nodes + 5, 65 * nodes, 10 ** 6):
                assert ops.native_workspace_bytes(id, False, nnz, nodes) == ws(nnz, nodes), (g.describe(), nnz, nodes)


def forms(t, seed):
    """A tensor as callers may hold it: as it is, strided, transposed, off 16-byte alignment, with the sign bit pending."""
    yield "plain", t
    yield "strided", torch.stack([t, t], -1)[..., 0]
    if t.dim() == 2:
        yield "transposed", t.t().contiguous().t()
    yield "misaligned", torch.cat([t.reshape(-1)[:1], t.reshape(-1)])[1:].view(t.shape)
    if t.is_floating_point():
        yield "negative", torch.complex(t, -t).conj().imag


@pytest.mark.gpu
@pytest.mark.parametrize("case", ["uvu", "uvu_shared", "uvw", "uvw_few", "uvw_rows", "conv", "conv_sorted", "conv_sorted_fp64"])
def test_every_form_of_call(cuda, case, monkeypatch):
    dtype = np.float64 if case.endswith("64") else np.float32
    conv = case.startswith("conv")
    sorted_ = case.startswith("conv_sorted")
    if conv:
        prob = common.channelwise(common.NEQUIP, dtype=dtype)[0]
        op = oeq.TensorProductConv(prob, torch_op=True, deterministic=sorted_)
    elif case.startswith("uvw"):
        prob = common.fully_connected(("10x1o+10x1e+48x0e+48x0o", "1x0e+1x1o+1x2e", "10x1o+10x1e+48x0e+48x0o") if case == "uvw_rows"
                                      else common.DENSE, shared=case != "uvw_rows")[0]
        op = oeq.TensorProduct(prob, torch_op=True)
    else:
        prob = common.channelwise(common.NEQUIP)[0]
        if case == "uvu_shared":
            paths = [(i.i_in1, i.i_in2, i.i_out, "uvu", True) for i in prob.instructions]
            prob = oeq.TPProblem(prob.irreps_in1, prob.irreps_in2, prob.irreps_out, paths, shared_weights=True, internal_weights=False)
        op = oeq.TensorProduct(prob, torch_op=True)
    assert op._native is not None
    calls = []
    for name in ("forward_raw", "backward_raw", "double_backward_raw", "exec_conv_rawptrs", "backward_rawptrs", "double_backward_rawptrs"):
        if hasattr(op, name):
            monkeypatch.setattr(op, name, lambda *a, f=getattr(op, name), n=name, **k: calls.append(n) or f(*a, **k))
    n, nodes = (300 if case == "uvw_few" else 5000) if not conv else 900, 70
    if conv:
        host = common.conv_inputs(prob, nodes, n, 3, dtype), common.conv_inputs(prob, nodes, n, 4, dtype)
        rows, cols, tperm, _ = otp.coord_graph(*common.random_graph(nodes, n, 5))
        index = [torch.tensor(a, device=cuda) for a in ((rows, cols, tperm) if sorted_ else (rows, cols))]
    else:
        host, index = (common.tp_inputs(prob, n, 3, dtype), common.tp_inputs(prob, n, 4, dtype)), []
    x, y, w, g, a, b, v = (torch.tensor(t, device=cuda) for t in (*host[0], *host[1][:3]))
    names = [op.forward.name(), op.backward_helper.name()]
    args = [[x, y, w, *index], [x, y, w, g, *index]]
    double = names[1].replace("grad_helper", "double_backward") if not conv else names[1].replace("conv_backward", "conv_double_backward")
    if hasattr(torch.ops.openequivariance_amd, double.split("::")[1]):
        names.append(double)
        args.append([x, y, w, g, a, b, v, *index])

    def run(name, args, general=False):
        out = getattr(torch.ops.openequivariance_amd, name.split("::")[1] + ("_general" if general else "")).default(*args)
        return [out] if torch.is_tensor(out) else out

    def same(got, want, kernels=True):
        """The same bits where the same kernels ran; those for misaligned tensors are others, and the sums of an unsorted edge
        list take the order in which integer atomics land: a few roundings of a few hundred terms."""
        assert len(got) == len(want)
        for p, q in zip(got, want):
            assert p.shape == q.shape and p.dtype == q.dtype and p.is_contiguous() and not p.requires_grad
            if kernels and case != "conv":
                assert torch.equal(p, q)
            else:
                assert not q.numel() or float((p - q).abs().max()) <= (1e-5 if dtype == np.float32 else 1e-13) * float(q.abs().max())
    for name, args_ in zip(names, args):
        print(case, name, flush=True)
        want = run(name, args_, general=True)                          # (takes the workspace, and times the backwards)
        calls.clear()
        same(run(name, args_), want)
        assert not calls, "an ordinary call went through Python"
        for i in range(len(args_)):
            for form, t in forms(args_[i], i):
                if not args_[i].is_floating_point() and form == "misaligned":
                    continue                                           # (8-byte values off 16 bytes are ordinary)
                print(case, name, i, form, flush=True)
                same(run(name, [*args_[:i], t, *args_[i + 1:]]), want, form != "misaligned")
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            for _ in range(2):                                         # a stream without a workspace, and with one
                got = run(name, args_)
        torch.cuda.current_stream().wait_stream(side)
        same(got, want)
        for i, t in enumerate(args_):
            for bad, error in ((t.cpu(), (ValueError, RuntimeError)), (t[:-1], (ValueError, TypeError)),
                               (t.to(torch.float16 if t.is_floating_point() else torch.int16), TypeError)):
                if conv and i == 0 and bad.shape != t.shape and name == names[0]:
                    continue                                           # (a graph of fewer nodes)
                with pytest.raises(error):
                    run(name, [*args_[:i], bad, *args_[i + 1:]])
        empty = [t[:0] if t.dim() == 2 or not t.is_floating_point() else t for t in args_]
        same(run(name, empty), run(name, empty, general=True))
        same(run(name, args_), want)
    # a capture, and the replays of it beside eager calls
    graph, held = torch.cuda.CUDAGraph(), [t.clone() for t in args[1]]
    want = run(names[1], held)
    with torch.cuda.graph(graph):
        got = run(names[1], held)
    for k in range(3):
        for t in got:
            t.fill_(float("nan"))
        same(run(names[1], args[1]), want)
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        same(got, want)


@pytest.mark.gpu
def test_switches_of_the_convolution_reach_the_kernels(cuda):
    """``graph_cache`` and ``autotune`` set on an operator in use: the next calls are the general implementation's."""
    prob = common.channelwise(common.NEQUIP)[0]
    conv = oeq.TensorProductConv(prob, torch_op=True)
    nodes, nnz = 60, 900
    rows, cols = common.random_graph(nodes, nnz, 5)
    r, c = torch.tensor(rows, device=cuda), torch.tensor(cols, device=cuda)
    x, y, w, g = (torch.tensor(t, device=cuda) for t in common.conv_inputs(prob, nodes, nnz, 3))
    want = conv.forward(x, y, w, r, c), *conv.backward_helper(x, y, w, g, r, c)
    rec = conv._workspace_record(nnz, nodes)

    def check():
        for p, q in zip((conv.forward(x, y, w, r, c), *conv.backward_helper(x, y, w, g, r, c)), want):
            assert common.rel_err(p.cpu().numpy(), q.cpu().numpy()) < 1e-5
    check()
    assert rec.fwd_key is None and rec.zero_fwd == (nnz, nodes, "")
    conv.graph_cache = True
    check()
    assert rec.fwd_key is not None
    conv.graph_cache = False
    assert rec.fwd_key is None
    check()
    conv.autotune = False
    check()
    assert rec.zero_bwd == (nnz, nodes, "")
    x2 = x.repeat(50, 1)                                              # a larger graph on the same stream: the scratch grows
    conv.forward(x2, y, w, r, c)
    assert rec.zero_fwd == (nnz, 50 * nodes, "")
    check()


@pytest.mark.gpu
def test_autotune_reaches_the_kernels_both_ways(cuda, monkeypatch):
    """An operator built without ``autotune``, and with either kernel set as its own: no call goes through Python; set later, the
    next backward is measured and the calls after it are C++ again, also after off and on."""
    from openequivariance_amd import tunables
    prob, oprob = common.channelwise(common.NEQUIP)
    nodes, nnz = 60, 900
    rows, cols = common.random_graph(nodes, nnz, 5)
    r, c = torch.tensor(rows, device=cuda), torch.tensor(cols, device=cuda)
    host = common.conv_inputs(prob, nodes, nnz, 3)
    x, y, w, g = (torch.tensor(t, device=cuda) for t in host)
    want = common.conv_reference_on_valid_edges(otp, oprob, *host, rows, cols, np.ones(nnz, bool))[1:]
    for default in ("atomic", "grouped"):
        monkeypatch.setattr(tunables.current, "conv_backward", default)
        conv = oeq.TensorProductConv(prob, torch_op=True)
        monkeypatch.undo()
        assert not conv.autotune and conv.backward_overwrites == (default == "grouped")
        python = []
        monkeypatch.setattr(conv, "backward_rawptrs", lambda *a, f=conv.backward_rawptrs, **k: python.append(1) or f(*a, **k))

        def calls():
            before = len(python)
            for got, ref in zip(conv.backward_helper(x, y, w, g, r, c), want):
                assert common.rel_err(got.cpu().numpy(), ref) < 1e-5
            return len(python) - before
        assert calls() == 1 and calls() == 0                       # (the first takes the workspace)
        conv.autotune = True
        assert calls() > 1 and len(conv._choices) == 1 and calls() == 0
        conv.autotune = False
        assert calls() == 0
        conv.autotune = True
        assert calls() == 1 and calls() == 0                       # the choice is known, and lent again


@pytest.mark.gpu
@pytest.mark.parametrize("problem", ["nequip", "mace"])
def test_both_backwards_of_unsorted_edges(cuda, problem, monkeypatch):
    """Each variant as the choice, whatever a stopwatch would say: from C++ (float atomics into zeros, groups by sender and - mace -
    in receiver order), the kinds of their counters kept apart, sizes changing between calls."""
    prob, oprob = common.channelwise(dict(nequip=common.NEQUIP, mace=common.MACE)[problem])
    conv = oeq.TensorProductConv(prob, torch_op=True)
    graphs = []
    for nodes, nnz, seed in ((60, 900, 5), (61, 1001, 6)):
        rows, cols = common.random_graph(nodes, nnz, seed)
        host = common.conv_inputs(prob, nodes, nnz, seed)
        want = common.conv_reference_on_valid_edges(otp, oprob, *host, rows, cols, np.ones(nnz, bool))
        graphs.append(([torch.tensor(t, device=cuda) for t in (*host, rows, cols)], want))
    assert conv._backward_variant("grouped")[0] is not conv._backward_variant("atomic")[0]
    (x, y, w, g, r, c), _ = graphs[1]
    conv.backward_helper(x, y, w, g, r, c)                                  # (the larger one's workspace; times the variants)
    sizes = (int(r.numel()).bit_length(), int(x.shape[0]).bit_length())
    python = []
    for name in ("exec_conv_rawptrs", "backward_rawptrs"):
        monkeypatch.setattr(conv, name, lambda *a, f=getattr(conv, name), n=name, **k: python.append(n) or f(*a, **k))
    for choice in ("atomic", "grouped", "atomic"):
        conv._bwd_choice = {sizes: choice}
        conv._lend_variant(sizes)
        for k in (0, 1, 1, 0, 0):
            (x, y, w, g, r, c), want = graphs[k]
            got = conv.forward(x, y, w, r, c), *conv.backward_helper(x, y, w, g, r, c)
            for a, b in zip(got, want):
                assert common.rel_err(a.cpu().numpy(), b) < 2e-5, (choice, k)
            assert conv._workspace_record(int(r.numel()), int(x.shape[0])).zero_bwd == (int(r.numel()), int(x.shape[0]), choice)
    assert not python, "a call went through Python"
