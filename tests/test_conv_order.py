"""The launch order of the backward's nodes, made beside the position list of an unsorted edge list: more nodes than a pass of
the ordering workgroup holds in registers, nodes without edges, hubs beyond the last bin, edges naming no node."""
import numpy as np
import pytest

import common
from host_emu import emu
from openequivariance_amd.codegen.uvu_sorted import UVUSortedGenerator
from oracle import tp as otp

IRREPS = ("4x0e+4x1o", "1x0e+1x1o", "4x0e+4x1o")
# one rounding a product and a sum, at most a hundred terms a value beside a hub's 400 edges
TOL = {np.float32: 1e3 * 6.0e-8, np.float64: 1e3 * 1.2e-16}


def graph(nodes, nnz, hub):
    if nnz == 0:
        return np.zeros(0, np.int64), np.zeros(0, np.int64), np.zeros(0, bool)
    rows, cols = common.random_graph(nodes - 1, nnz, 5, self_loops=True)
    cols[:hub] = 3
    rows, cols, _ = common.with_invalid_edges(rows, cols, nodes, 6)
    valid = (rows >= 0) & (rows < nodes) & (cols >= 0) & (cols < nodes)
    return rows, cols, valid


@pytest.mark.parametrize("nodes,nnz,hub", [(6, 0, 0), (1, 3, 0), (30, 300, 150)])
def test_emulated(nodes, nnz, hub):
    prob, oprob = common.channelwise(IRREPS, dtype=np.float32)
    g = UVUSortedGenerator(prob, grouped_backward=True).add_few_nodes()
    _, bwd, ws = g.plan_few()
    names = [s["kernel"] for s in bwd if "few_nodes" not in s]
    assert names == ["group_clear_backward", "group_count_backward", "group_fill_backward", "backward"]
    assert "order_backward" not in g.render() and "order_backward" in UVUSortedGenerator(prob, grouped_backward=True).render()
    steps = [s for s in bwd if "few_nodes" not in s]
    assert [s.get("grid_y", 1) for s in steps[:3]] == [1, 1, 2]
    rows, cols, valid = (np.zeros(nnz, np.int64), np.zeros(nnz, np.int64), np.ones(nnz, bool)) if nodes == 1 else graph(nodes, nnz, hub)
    X, Y, W, G = common.conv_inputs(prob, nodes, nnz, 8)
    # (the tests' host build knows order_backward by name: a kernel that nothing launches)
    render = g.render
    g.render = lambda prelude=None: render(prelude) + "\nstatic void order_backward(BWD_ARGS) {}\n"
    out = emu.run_conv(g, steps, X, Y, W, rows, cols, G=G, tperm=np.arange(nnz), ws_bytes=ws(nnz, nodes))
    if nnz == 0:
        assert not out["Xg"].any()
        return
    for got, want in zip((out["Xg"], out["Yg"], out["Wg"]), common.conv_reference_on_valid_edges(otp, oprob, X, Y, W, G, rows, cols, valid)[1:]):
        assert np.abs(got - want).max() <= TOL[np.float32] * np.abs(want).max()


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_on_the_gpu(cuda, dtype):
    import torch
    import openequivariance_amd as oeq
    prob, oprob = common.channelwise(IRREPS, dtype=dtype)
    conv = oeq.TensorProductConv(prob, torch_op=True, deterministic=False)
    conv._bwd_choice = type("Grouped", (dict,), dict(__contains__=lambda s, k: True, __getitem__=lambda s, k: "grouped"))()
    for nodes, nnz, hub in ((5000, 9000, 400), (9000, 20000, 300), (30, 500, 300)):
        print(nodes, nnz, flush=True)
        rows, cols, valid = graph(nodes, nnz, hub)
        X, Y, W, G = common.conv_inputs(prob, nodes, nnz, 8, dtype)
        want = common.conv_reference_on_valid_edges(otp, oprob, X, Y, W, G, rows, cols, valid)
        index = [torch.tensor(a, device=cuda) for a in (rows, cols)]
        for _ in range(2):
            x, y, w, g = (torch.tensor(a, device=cuda).requires_grad_() for a in (X, Y, W, G))
            z = conv(x, y, w, *index)
            for got, ref in zip((z, *torch.autograd.grad(z, (x, y, w), g.detach())), want):
                assert np.abs(got.detach().cpu().numpy() - ref).max() <= TOL[dtype] * np.abs(ref).max()
