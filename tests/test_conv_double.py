"""Double backward of the fused convolution in two passes: the generated source on the host (tests/host_emu) and the
operator on the GPU against the second derivatives of the fp64 oracle, at the edges of the schedule: one and two row
groups per wavefront, LDS-staged and register loops, ragged multiplicities over two chunks, output blocks in several
launches, nodes long enough to be walked in pieces, nodes without edges, edges naming no node, blocks no path touches."""
import os
import tempfile

import numpy as np
import pytest

import common
import openequivariance_amd as oeq
from common import rel_err
from host_emu import emu
from openequivariance_amd import tunables
from openequivariance_amd.codegen.uvu_conv_double import UVUDetDoubleGenerator, conv_double_generator
from oracle import tp as otp
from oracle import torch_cpu

CASES = {   # irreps, nodes, edges, hub?, staged loops (None: by the rule)
    "two_row_groups_staged": (common.NEQUIP, 7, 40, False, True),
    "two_row_groups_registers": (common.NEQUIP, 7, 40, False, False),
    "hubs": (("16x0e+16x1o", "1x0e+1x1o", "16x0e+16x1o"), 12, 400, True, None),
    "hubs_chunks_groups": (("70x0e+70x1o+70x2e", "1x0e+1x1o+1x2e+1x3o", "70x0e+70x1o+70x2e+70x3o"), 12, 300, True, None),
    "ragged_two_chunks": (("5x0e+3x1o+70x2e", "1x0e+1x1o+1x2e", "5x0e+3x1o+70x2e+7x3o"), 5, 23, False, None),
    "blocks_no_path_touches": (("1x0e+1x1o+16x3o", "1x0e+1x1o", "16x0e+16x0o+16x1e+16x1o"), 6, 17, False, None),
}
MAIN = r"""
int main(int argc, char** argv) {
    const std::string d = argv[1];
    FILE* job = fopen((d + "/job.txt").c_str(), "r");
    unsigned long long nnz, nodes, d1, d2, d3, wn, wsb;
    if (fscanf(job, "%llu %llu %llu %llu %llu %llu %llu", &nnz, &nodes, &d1, &d2, &d3, &wn, &wsb) != 7) return 3;
    auto in = [&](const char* name, unsigned long long w) { return emu_read(d + "/" + name + ".bin", w * sizeof(T)); };
    auto X = in("X", nodes * d1), Y = in("Y", nnz * d2), W = in("W", nnz * wn), G = in("G", nodes * d3);
    auto A = in("A", nodes * d1), B = in("B", nnz * d2), V = in("V", nnz * wn);
    auto rows = emu_read(d + "/rows.bin", nnz * 8), cols = emu_read(d + "/cols.bin", nnz * 8), tperm = emu_read(d + "/tperm.bin", nnz * 8);
    auto out = [&](unsigned long long w) { return std::vector<char>(w * sizeof(T), (char)0x7f); };
    auto Xg = out(nodes * d1), Yg = out(nnz * d2), Wg = out(nnz * wn), Gg = out(nodes * d3);
    std::vector<char> ws(wsb, (char)0x7f);
    char name[64]; unsigned threads, gx, gy;
#define CALL(fn) if (k == #fn) { emu_run(gx, gy, threads, [&] { fn((const T*)X.data(), (const T*)Y.data(), (const T*)W.data(), (const T*)G.data(), \
        (const T*)A.data(), (const T*)B.data(), (const T*)V.data(), (T*)Xg.data(), (T*)Yg.data(), (T*)Wg.data(), (T*)Gg.data(), \
        (const i64*)rows.data(), (const i64*)cols.data(), nnz, nodes, ws.data(), (const i64*)tperm.data()); }); continue; }
    while (fscanf(job, "%63s %u %u %u", name, &threads, &gx, &gy) == 4) {
        const std::string k = name;
@CALLS@
        fprintf(stderr, "unknown kernel %s\n", name); return 3;
    }
    emu_write(d + "/Xg.bin", Xg); emu_write(d + "/Yg.bin", Yg); emu_write(d + "/Wg.bin", Wg); emu_write(d + "/Gg.bin", Gg);
    return 0;
}
"""


def _graph(case, deterministic, seed):
    _, nodes, nnz, hub, _ = CASES[case]
    rows, cols = (common.hub_graph(nodes - 1, nnz, seed, hub_in=3, hub_out=5, in_edges=150, out_edges=130) if hub
                  else common.random_graph(nodes - 1, nnz, seed))          # the last node has no edges
    return otp.coord_graph(rows, cols)[:3] if deterministic else (rows, cols, np.full(nnz, 12345))


def _inputs(prob, nodes, nnz, seed, dtype):
    X, Y, W, G = common.conv_inputs(prob, nodes, nnz, seed, dtype)
    A, B, V, _ = common.conv_inputs(prob, nodes, nnz, seed + 1, dtype)
    return X, Y, W, G, A, B, V


def _reference(oprob, rows, cols, X, Y, W, G, A, B, V):
    """fp64 second derivatives; edges that name no node contribute nothing and have zero gradients."""
    import torch
    n = X.shape[0]
    ok = (rows >= 0) & (rows < n) & (cols >= 0) & (cols < n)
    r, c = torch.tensor(rows[ok]), torch.tensor(cols[ok])
    x, y, w, g = (torch.tensor(a.astype(np.float64), requires_grad=True) for a in (X, Y, W, G))
    z = torch.zeros_like(g).index_add(0, r, torch_cpu.TorchTP(oprob, dtype=torch.float64).forward(x[c], y[ok], w[ok]))
    first = torch.autograd.grad(z, (x, y, w), g, create_graph=True)
    second = torch.autograd.grad(first, (x, y, w, g), [torch.tensor(a.astype(np.float64)) for a in (A, B, V)])
    return [t.numpy() for t in second]


def _run_emulated(g, rows, cols, tperm, X, Y, W, G, A, B, V):
    nnz, nodes = rows.shape[0], X.shape[0]
    steps = g.steps()
    exe = emu.build(g.render(prelude=emu.emu_prelude(g.T)),
                    MAIN.replace("@CALLS@", "\n".join(f"        CALL({k})" for k in dict.fromkeys(s["kernel"] for s in steps))))
    dt = X.dtype
    with tempfile.TemporaryDirectory() as d:
        for k, a in dict(X=X, Y=Y, W=W, G=G, A=A, B=B, V=V, rows=rows, cols=cols, tperm=tperm).items():
            np.ascontiguousarray(a, dtype=np.int64 if k in ("rows", "cols", "tperm") else dt).tofile(os.path.join(d, k + ".bin"))
        with open(os.path.join(d, "job.txt"), "w") as f:
            f.write(f"{nnz} {nodes} {X.shape[1]} {Y.shape[1]} {G.shape[1]} {W.shape[1]} {g.plan()[2](nnz, nodes)}\n")
            for s in steps:
                f.write(f"{s['kernel']} {s['num_threads']} {emu.grid_of(s, nnz, nodes)} {s.get('grid_y', 1)}\n")
        emu._run(exe, d)
        return [np.fromfile(os.path.join(d, k + ".bin"), dtype=dt).reshape(a.shape) for k, a in
                (("Xg", X), ("Yg", Y), ("Wg", W), ("Gg", G))]


@pytest.mark.parametrize("deterministic", [False, True])
@pytest.mark.parametrize("case", sorted(CASES))
def test_generated_source(case, deterministic, monkeypatch):
    irreps, nodes, nnz, hub, staged = CASES[case]
    prob, oprob = common.channelwise(irreps)
    if case == "hubs_chunks_groups":
        monkeypatch.setattr(tunables.current, "det_split", 60)
    g = conv_double_generator(prob, deterministic)
    if staged is not None:
        if not deterministic:
            pytest.skip("the unsorted kernels take the rule's loops")
        g = UVUDetDoubleGenerator(prob, lds=staged)
        assert g.lds_backward == staged
    d = g if deterministic else g.bwd
    if case == "hubs_chunks_groups":
        assert d.NCH == 2 and d.H > 1
    rows, cols, tperm = _graph(case, deterministic, 31)
    args = _inputs(prob, nodes, nnz, 32, np.float32)
    for a, b in zip(_run_emulated(g, rows, cols, tperm, *args), _reference(oprob, rows, cols, *args)):
        assert rel_err(a, b) < 4e-6       # twice the terms of a first derivative, fp32 against fp64


@pytest.mark.parametrize("deterministic", [False, True])
def test_generated_source_edges_naming_no_node(deterministic):
    prob, oprob = common.channelwise(("8x0e+8x1o", "1x0e+1x1o+1x2e", "8x0e+8x1o+8x2e"), np.float64)
    nodes, nnz = 9, 300
    rows, cols, valid = common.with_invalid_edges(*common.random_graph(nodes, nnz, 5, self_loops=True), nodes, 6)
    tperm = np.full(nnz, 12345)
    if deterministic:
        order = np.lexsort((cols, rows))
        rows, cols, valid = rows[order], cols[order], valid[order]
        tperm = np.lexsort((np.arange(nnz), rows, cols)).astype(np.int64)
    args = _inputs(prob, nodes, nnz, 33, np.float64)
    got = _run_emulated(conv_double_generator(prob, deterministic), rows, cols, tperm, *args)
    for a, b in zip(got, _reference(oprob, rows, cols, *args)):
        assert rel_err(a, b) < 1e-13
    assert not got[1][~valid].any() and not got[2][~valid].any()


def _device(cuda, arrays):
    import torch
    return [torch.tensor(a, device=cuda) for a in arrays]


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("deterministic", [False, True])
@pytest.mark.parametrize("case", sorted(CASES))
def test_operator(cuda, case, deterministic, dtype, monkeypatch):
    import torch
    if case == "hubs_chunks_groups":
        monkeypatch.setattr(tunables.current, "det_split", 60)
    irreps, nodes, nnz, _, _ = CASES[case]
    prob, oprob = common.channelwise(irreps, dtype)
    tol = 2e-5 if dtype == np.float32 else 2e-12       # two chained kernels' worth of the first-order tolerances
    conv = oeq.TensorProductConv(prob, torch_op=True, deterministic=deterministic)
    rows, cols, tperm = _graph(case, deterministic, 34)
    args = _inputs(prob, nodes, nnz, 35, dtype)
    index = _device(cuda, (rows, cols, tperm) if deterministic else (rows, cols))
    x, y, w, g = (t.requires_grad_() for t in _device(cuda, args[:4]))
    cots = _device(cuda, args[4:])
    first = torch.autograd.grad(conv(x, y, w, *index), (x, y, w), g, create_graph=True)
    second = torch.autograd.grad(first, (x, y, w, g), cots, retain_graph=True)
    assert conv._double is not None, "the second derivatives did not come from the fused kernels"
    for a, b in zip(second, _reference(oprob, rows, cols, *args)):
        assert rel_err(a.cpu().numpy(), b) <= tol
    # forward and backward calls in between find their own preparation again; a repeat gives the same numbers
    again = torch.autograd.grad(torch.autograd.grad(conv(x, y, w, *index), (x, y, w), g, create_graph=True), (x, y, w, g), cots)
    for a, b in zip(again, second):
        assert torch.equal(a, b) if deterministic else rel_err(a.cpu().numpy(), b.cpu().numpy()) <= tol
    # a graph of the second derivatives is built from first-order calls: the same numbers, differentiable again
    composed = torch.autograd.grad(first, (x, y, w, g), cots, create_graph=True)
    for a, b in zip(composed, second):
        assert rel_err(a.detach().cpu().numpy(), b.cpu().numpy()) <= tol
    assert all(bool(torch.isfinite(t).all()) for t in torch.autograd.grad(composed[0].square().sum(), (y, w)))


@pytest.mark.gpu
@pytest.mark.parametrize("deterministic", [False, True])
def test_graph_cache_keeps_the_preparations_of_all_three_directions(cuda, deterministic, monkeypatch):
    """With ``graph_cache`` a training step on forces over an unchanged edge list prepares nothing anew; a change of the
    edge list, seen by the version counter, rebuilds."""
    import torch
    from openequivariance_amd import runtime as rt
    irreps, nodes, nnz, _, _ = CASES["hubs"]
    prob, oprob = common.channelwise(irreps)
    conv = oeq.TensorProductConv(prob, torch_op=True, deterministic=deterministic, graph_cache=True)
    calls, plain = [], rt.ConvImpl.double_backward
    monkeypatch.setattr(rt.ConvImpl, "double_backward", lambda self, *a: calls.append(a[-2:]) or plain(self, *a))
    args = _inputs(prob, nodes, nnz, 41, np.float32)
    x, y, w, g = (t.requires_grad_() for t in _device(cuda, args[:4]))
    cots = _device(cuda, args[4:])
    graphs = [_graph("hubs", deterministic, seed)[:3 if deterministic else 2] for seed in (42, 43)]
    index = _device(cuda, graphs[0])
    for k, graph in enumerate((graphs[0], graphs[0], graphs[0], graphs[1], graphs[1])):
        if k == 3:
            for dst, src in zip(index, _device(cuda, graphs[1])):
                dst.copy_(src)
        first = torch.autograd.grad(conv(x, y, w, *index), (x, y, w), g, create_graph=True)
        rec = conv._workspace_record(nnz, nodes)
        keys = rec.fwd_key, rec.bwd_key
        assert k == 0 or None not in keys     # (the first backward of the unsorted operator lets the workspace grow)
        second = torch.autograd.grad(first, (x, y, w, g), cots)
        assert conv._workspace_record(nnz, nodes) is rec and (rec.fwd_key, rec.bwd_key) == keys
        for a, b in zip(second, _reference(oprob, graph[0], graph[1], *args)):
            assert rel_err(a.cpu().numpy(), b) <= 2e-5
    assert [prepared for prepared, _ in calls] == [False, True, True, False, True]


@pytest.mark.gpu
@pytest.mark.parametrize("deterministic", [False, True])
def test_empty_edge_list_and_other_graph_sizes(cuda, deterministic):
    """No edges: node gradients are zeros.  A larger graph afterwards grows the workspace, a smaller one reuses it."""
    import torch
    prob, oprob = common.channelwise(common.NEQUIP)
    conv = oeq.TensorProductConv(prob, torch_op=True, deterministic=deterministic)
    for nodes, nnz in ((5, 0), (200, 3000), (20, 90)):
        rows, cols = common.random_graph(nodes, nnz, 36)
        tperm = np.zeros(0, dtype=np.int64)
        if deterministic and nnz:
            rows, cols, tperm, _ = otp.coord_graph(rows, cols)
        args = _inputs(prob, nodes, nnz, 37, np.float32)
        index = _device(cuda, (rows, cols, tperm) if deterministic else (rows, cols))
        x, y, w, g = (t.requires_grad_() for t in _device(cuda, args[:4]))
        first = torch.autograd.grad(conv(x, y, w, *index), (x, y, w), g, create_graph=True)
        second = torch.autograd.grad(first, (x, y, w, g), _device(cuda, args[4:]))
        if nnz == 0:
            assert not second[0].any() and not second[3].any()
            continue
        for a, b in zip(second, _reference(oprob, rows, cols, *args)):
            assert rel_err(a.cpu().numpy(), b) <= 2e-5


@pytest.mark.gpu
def test_capture_before_first_use_composes(cuda):
    """The first use takes its workspace, which a stream capture does not: the second derivatives recorded before it come
    from the first-order ones, recorded afterwards from the fused ones; every replay gives the eager numbers."""
    import torch
    prob, _ = common.channelwise(common.NEQUIP)
    conv = oeq.TensorProductConv(prob, torch_op=True, deterministic=True)
    rows, cols, tperm, _ = otp.coord_graph(*common.random_graph(30, 400, 38))
    index = _device(cuda, (rows, cols, tperm))
    args = _inputs(prob, 30, 400, 39, np.float32)
    x, y, w, g = (t.requires_grad_() for t in _device(cuda, args[:4]))
    cots = _device(cuda, args[4:])

    def step():
        first = torch.autograd.grad(conv(x, y, w, *index), (x, y, w), g, create_graph=True)
        return torch.autograd.grad(first, (x, y, w, g), cots)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    graphs = []
    for _ in range(2):
        with torch.cuda.stream(side):
            torch.autograd.grad(conv(x, y, w, *index), (x, y, w), g)       # workspace of this stream, first order only
        side.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=side):
            out = step()
        graphs.append((graph, out, conv._double is not None))
        eager = step()
        torch.cuda.synchronize()
        assert conv._double is not None
        with torch.cuda.stream(side):
            step()                                                       # grows this stream's workspace before the next capture
        side.synchronize()
    assert [f for _, _, f in graphs] == [False, True]
    for graph, out, _ in graphs:
        for _ in range(3):
            graph.replay()
            torch.cuda.synchronize()
            for a, b in zip(out, eager):
                assert rel_err(a.cpu().numpy(), b.cpu().numpy()) <= 2e-5
            step()
            torch.cuda.synchronize()
